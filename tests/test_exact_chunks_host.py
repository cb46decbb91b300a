"""What the chunk-parallel exact kernels of the decay rule ask of the host (T2FW_FLAG_EXACT_CHUNKS): the workspace and the
choice of the kernels.  No device needed."""
import pytest
import torch


@pytest.mark.parametrize("rows,T,D,K", [(96, 1024, 64, 64), (1024, 4096, 8, 8), (13, 385, 33, 17), (1, 1, 1, 1), (7, 65, 16, 49)])
def test_workspace_follows_the_widths(rows, T, D, K):
    """Per chunk of 64 steps one state and the gate products in fp32, widths in whole tiles of 16, and flags: 1024 x 4096
    steps of an 8 x 8 state need 75 MB (1.1 GB when every chunk had room for a 64 x 64 state)."""
    from t2fw_amd import _lib
    lib = _lib.load()
    items, Dp, Kp = rows * -(-T // 64), -(-D // 16) * 16, -(-K // 16) * 16
    up = lambda n: -(-n // 256) * 256
    want = items * (Dp * Kp + Dp + Kp) * 4 + up(4 * items) + up(16 * rows)
    a = (rows, T, D, K, 64, _lib.F32, _lib.FLAG_EXACT_CHUNKS)
    assert lib.t2fw_lfw_forward_workspace_bytes(*a) == want
    assert lib.t2fw_lfw_workspace_bytes(*a) == want


def test_the_choice_is_made_once_per_shape():
    from t2fw_amd import _lib, functional_lfw as F
    F._forward_plan.cache_clear()
    for dtype, D, want in ((torch.float32, 64, _lib.FLAG_EXACT_CHUNKS), (torch.float16, 64, 0), (torch.float16, 33, _lib.FLAG_EXACT_CHUNKS)):
        a = F._forward_plan(12, 333, D, D, 64, dtype, 0)
        assert a is F._forward_plan(12, 333, D, D, 64, dtype, 0)
        assert a[0] == want and a[1:] == F._sizes(12, 333, D, D, 64, _lib.DTYPE_CODE[dtype], want)
    assert F._forward_plan.cache_info().misses == 3 and F._forward_plan.cache_info().hits == 3


def test_tensors_in_host_memory_switch_no_device():
    from t2fw_amd.functional_lfw import _on_device
    with _on_device(torch.zeros(1).device):
        pass
