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
        a = F._forward_plan(12, 333, D, D, 64, dtype, 0, True)
        assert a is F._forward_plan(12, 333, D, D, 64, dtype, 0, True)
        assert a[0] == want and a[1:] == F._sizes(12, 333, D, D, 64, _lib.DTYPE_CODE[dtype], want)
    assert F._forward_plan.cache_info().misses == 3 and F._forward_plan.cache_info().hits == 3


def test_tensors_in_host_memory_switch_no_device():
    from t2fw_amd.functional_lfw import _on_device
    with _on_device(torch.zeros(1).device):
        pass


F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


@pytest.mark.parametrize("rows,T,D,K,need_grad,taken", [
    (96, 223, 64, 64, True, False), (96, 224, 64, 64, True, True), (96, 224, 64, 64, False, True),      # steps
    (256, 224, 64, 64, True, True), (257, 224, 64, 64, True, False),                                     # 64 x 64
    (1024, 224, 8, 8, True, True), (1025, 224, 8, 8, True, False), (256, 224, 8, 64, True, True),        # a width up to 8
    (1024, 224, 16, 16, True, False), (1024, 1024, 16, 16, True, False),      # measured 0.74 and 0.81 times as fast
    (384, 447, 16, 9, True, True), (385, 447, 16, 9, True, False), (640, 448, 9, 16, True, True), (641, 448, 16, 16, True, False),
    (384, 224, 17, 32, True, True), (385, 224, 32, 32, True, False), (256, 224, 33, 17, True, True), (257, 224, 33, 17, True, False),
    (160, 447, 63, 63, True, True), (161, 447, 63, 63, True, False), (256, 448, 63, 33, True, True), (257, 448, 33, 63, True, False),
    (1024, 224, 16, 8, False, True), (128, 224, 64, 8, False, True), (129, 224, 64, 8, False, False),    # forward alone
    (256, 224, 16, 64, False, True), (257, 224, 16, 64, False, False), (64, 224, 63, 63, False, True), (65, 224, 63, 63, False, False),
    (384, 1023, 16, 16, False, False), (384, 1024, 16, 16, False, True), (512, 1024, 16, 16, False, False),
    (513, 448, 16, 16, False, True), (768, 448, 16, 16, False, True), (769, 448, 16, 16, False, False), (640, 447, 16, 16, False, False),
])
def test_choice_of_the_kernels(rows, T, D, K, need_grad, taken):
    """Edges of the rule; what was measured on both sides stands beside it."""
    from t2fw_amd import _lib
    from t2fw_amd.functional_lfw import _exact_chunk_flags as choose
    want = _lib.FLAG_EXACT_CHUNKS if taken else 0
    assert choose(rows, T, D, K, 64, F32, 0, need_grad) == want
    if (D, K) != (64, 64):
        assert choose(rows, T, D, K, 64, F16, 0, need_grad) == choose(rows, T, D, K, 64, BF16, 0, need_grad) == want


def test_calls_that_keep_their_kernels():
    from t2fw_amd import _lib
    from t2fw_amd.functional_lfw import _exact_chunk_flags as choose
    for need_grad in (False, True):
        assert choose(96, 1024, 64, 64, 64, F16, 0, need_grad) == choose(96, 1024, 64, 64, 64, BF16, 0, need_grad) == 0
        assert choose(4, 1024, 64, 64, 64, torch.float64, 0, need_grad) == choose(4, 1024, 33, 17, 64, torch.float64, 0, need_grad) == 0
        for C in (32, 63, 65, 128):
            assert choose(4, 1024, 64, 64, C, F32, 0, need_grad) == 0
        for D, K in ((65, 64), (64, 65), (128, 128)):
            assert choose(4, 1024, D, K, 64, F32, 0, need_grad) == 0
        for caller in (_lib.FLAG_FORCE_SCAN, _lib.FLAG_NO_FIXUP, _lib.FLAG_BLOCKWISE, _lib.FLAG_EXACT_CHUNKS):
            assert choose(4, 64, 64, 64, 64, F32, caller, need_grad) == caller
