"""The delta rule's backward with the key side's chunks of 64 tokens side by side: lengths around the edges of its blocks of 16,
stages of 32 and chunks of 64, for the types and operand modes that run it.  Against the oracle in float64 at the tolerance
of the per-step kernels (single bf16 operands: 1e-2 of the largest element, as in tests/test_dfw_chunk_gpu.py); the edges lie in the
results' memory (t2fw_dfw_backward) or in a workspace (t2fw_dfw_backward_sums), which gives the same bits."""
import pytest
import torch

from oracle.dfw_ref import dfw_reference_grads
from tests.test_dfw_chunk_gpu import run_abi
from tests.test_dfw_gpu import NAMES, TOL_DFW, make_inputs
from tests.test_lfw_gpu import assert_close

GUARD = 4096


def run_sums(q, k, s, go, gs, delta, fin, flags):
    from t2fw_amd import _lib
    lib = _lib.load()
    B, T, D = delta.shape
    code = _lib.DTYPE_CODE[delta.dtype]
    n = lib.t2fw_dfw_backward_sums_workspace_bytes(B, T, D, 64, code, flags)
    assert n > 0
    ws = torch.full((n + GUARD,), 7, dtype=torch.uint8, device="cuda")
    grads = [torch.full_like(t, float("nan")) for t in (q, k, delta, s)]
    P = _lib.ptr
    call = lambda size: lib.t2fw_dfw_backward_sums(P(go), P(gs), P(q), P(k), P(delta), P(fin), *[P(t) for t in grads], B, T, D, 64, code,
                                                     flags, P(ws), size, _lib.current_stream_handle(delta.device))
    assert call(n - 1) != 0
    _lib.check(call(n))
    torch.cuda.synchronize()
    assert (ws[n:] == 7).all()
    return grads


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,flags", [(torch.float32, 0), (torch.float32, 16), (torch.float16, 16), (torch.bfloat16, 16)])
@pytest.mark.parametrize("B,T", [(1, 1), (3, 15), (2, 16), (2, 17), (2, 32), (3, 33), (1, 63), (2, 64), (2, 65), (3, 96), (2, 97), (9, 128), (2, 129),
                                 (2, 200), (1, 449)])
def test_lengths_around_the_edges(dtype, flags, B, T):
    ts = make_inputs(B, T, 64, 64, dtype, seed=900 + T)
    _, _, refs = dfw_reference_grads(*ts)
    q, k, v, s, go, gs = [t.cuda() for t in ts]
    _, fin, delta, grads = run_abi(q, k, v, s, go, gs, flags)
    tol = TOL_DFW[dtype] if not flags else (1e-2, 1e-2)
    for n, g, r in zip(NAMES, grads, refs):
        assert_close(g, r, dtype, n, tol=tol)
    for a, b in zip(run_sums(q, k, s, go, gs, delta, fin, flags), grads):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("which", [0, 2, 4])
@pytest.mark.parametrize("T,at", [(150, 100), (150, 131), (128, 64)])
def test_values_that_are_not_finite(which, T, at):
    """a NaN among queries, values or the outputs' gradients: what the per-step kernels keep free of it stays so here, but for
    the 16 tokens around it"""
    ts = [t.cuda() for t in make_inputs(1, T, 64, 64, torch.float32, seed=8)]
    ts[which][0, at, 5] = float("nan")
    exact, got = run_abi(*ts, 1)[3], run_abi(*ts, 0)[3]
    block = torch.arange(T, device="cuda") // 16 == at // 16
    for n, a, b in zip(NAMES, got, exact):
        if a.shape[1] == T and n != "d_state":
            a, b = a[:, ~block], b[:, ~block]
        assert torch.equal(a.isnan(), b.isnan()), n


def test_where_the_sums_are_not_taken():
    from t2fw_amd import _lib
    lib = _lib.load()
    size = lib.t2fw_dfw_backward_sums_workspace_bytes
    assert size(96, 1024, 64, 64, _lib.F32, 0) == 2 * 96 * 1024 * 64 * 4
    assert size(48, 777, 128, 64, _lib.BF16, 16) == 2 * 48 * 777 * 128 * 2
    for call in ((2, 10, 64, 64, _lib.F64, 0), (2, 10, 64, 64, _lib.F32, 1), (2, 10, 96, 64, _lib.F32, 0), (2, 10, 64, 32, _lib.F32, 0), (0, 10, 64, 64, _lib.F32, 0),
                 (2, 0, 64, 64, _lib.F32, 0), (2, 10, 128, 64, _lib.F16, 0), (2, 10, 128, 64, _lib.BF16, 0), (2, 1 << 25, 64, 64, _lib.F32, 0),
                 (2, 10, 64, 64, 99, 0), (-1, 10, 64, 64, _lib.F32, 0)):
        assert size(*call) == 0, call
