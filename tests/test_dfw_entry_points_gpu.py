"""The delta rule's backward through the C ABI where DFWFunction does not go: the shares of several value blocks
(t2fw_dfw_backward_blocks) for every type and operand mode, and their sums (t2fw_dfw_backward_sums), with guards around the workspace
and the results."""
import pytest
import torch

from oracle.dfw_ref import dfw_reference_grads
from tests.test_dfw_gpu import NAMES, TOL_DFW, make_inputs
from tests.test_lfw_gpu import assert_close

pytestmark = pytest.mark.gpu
SINGLE = 16                    # T2FW_FLAG_BF16_OPERANDS
MODES = [(torch.float32, 0), (torch.float32, SINGLE), (torch.float16, 0), (torch.float16, SINGLE), (torch.bfloat16, 0), (torch.bfloat16, SINGLE)]
GUARD = 4096


def guarded(shape, dtype):
    n = torch.Size(shape).numel()
    room = torch.full((n + 2 * GUARD,), 7, dtype=dtype, device="cuda")
    room[GUARD:GUARD + n] = float("nan")
    return room, room[GUARD:GUARD + n].view(shape)


def untouched(room):
    return bool((room[:GUARD] == 7).all()) and bool((room[-GUARD:] == 7).all())


@pytest.mark.parametrize("dtype,flags", MODES)
@pytest.mark.parametrize("B,T,n", [(3, 33, 2), (2, 64, 3), (2, 65, 2), (1, 200, 5), (9, 129, 2)])
def test_shares_and_sums_of_several_value_blocks(dtype, flags, B, T, n):
    from t2fw_amd import _lib
    lib, P, code, D = _lib.load(), _lib.ptr, _lib.DTYPE_CODE[dtype], 64 * n
    ts = make_inputs(B, T, D, 64, dtype, seed=T + n)
    q, k, v, s, go, gs = [t.cuda() for t in ts]
    st = _lib.current_stream_handle(v.device)
    out, delta, fin = torch.empty_like(v), torch.empty_like(v), torch.empty_like(s)
    _lib.check(lib.t2fw_dfw_forward_blocks(P(q), P(k), P(v), P(s), P(out), P(fin), P(delta), B, T, D, 64, code, flags, st))
    rooms, grads = zip(*[guarded(sh, dtype) for sh in ((B, n, T, 64), (B, n, T, 64), (B, T, D), (B, D, 64))])
    _lib.check(lib.t2fw_dfw_backward_blocks(P(go), P(gs), P(q), P(k), P(delta), P(fin), *[P(t) for t in grads], B, T, D, 64, code, flags, st))
    torch.cuda.synchronize()
    assert all(untouched(r) for r in rooms)
    tol = TOL_DFW[dtype] if not flags else (1e-2, 1e-2)      # single operands: 1e-2 of the largest element, as in tests/test_dfw_chunk_gpu.py
    qr, kr, vr, sr, gor, gsr = ts
    for i in range(n):
        c = slice(64 * i, 64 * i + 64)
        _, _, refs = dfw_reference_grads(qr, kr, vr[..., c], sr[:, c], gor[..., c], gsr[:, c])
        for name, g, r in zip(NAMES, (grads[0][:, i], grads[1][:, i], grads[2][..., c], grads[3][:, c]), refs):
            assert_close(g, r, dtype, name, tol=tol)
    size = lib.t2fw_dfw_backward_sums_workspace_bytes(B, T, D, 64, code, flags)
    assert (size > 0) == (dtype == torch.float32 or flags == SINGLE)
    if size == 0:
        return
    ws = torch.full((size + 2 * GUARD,), 7, dtype=torch.uint8, device="cuda")
    rooms, sums = zip(*[guarded(sh, dtype) for sh in ((B, T, 64), (B, T, 64), (B, T, D), (B, D, 64))])
    call = lambda nbytes: lib.t2fw_dfw_backward_sums(P(go), P(gs), P(q), P(k), P(delta), P(fin), *[P(t) for t in sums], B, T, D, 64, code, flags,
                                                     _lib.ctypes.c_void_p(ws.data_ptr() + GUARD), nbytes, st)
    assert call(size - 1) != 0
    _lib.check(call(size))
    torch.cuda.synchronize()
    assert all(untouched(r) for r in rooms) and untouched(ws)
    _, _, refs = dfw_reference_grads(*ts)
    for name, g, r in zip(NAMES, sums, refs):
        assert_close(g, r, dtype, name, tol=tol)
    assert torch.equal(sums[2], grads[2]) and torch.equal(sums[3], grads[3])


@pytest.mark.parametrize("dtype,flags", [m for m in MODES if m[0] == torch.float32 or m[1]])
def test_error_of_the_sums_against_that_of_the_shares(dtype, flags):
    """d_query and d_key against float64: the key side's chunks (the sums) no worse than its sequential form (the shares, rounded each
    and added up), where operands are single bf16 numbers as well; 1 % is what the two scatter by, in either direction"""
    from t2fw_amd import _lib
    from t2fw_amd.functional_dfw import DFWFunction
    lib, P, code, (B, T, n) = _lib.load(), _lib.ptr, _lib.DTYPE_CODE[dtype], (24, 777, 2)
    D = 64 * n
    q, k, v, s, go, gs = [t.cuda() for t in make_inputs(B, T, D, 64, dtype, seed=6)]
    st = _lib.current_stream_handle(v.device)
    out, delta, fin = torch.empty_like(v), torch.empty_like(v), torch.empty_like(s)
    _lib.check(lib.t2fw_dfw_forward_blocks(P(q), P(k), P(v), P(s), P(out), P(fin), P(delta), B, T, D, 64, code, flags, st))
    shares = [q.new_empty((B, n, T, 64)), q.new_empty((B, n, T, 64)), torch.empty_like(v), torch.empty_like(s)]
    _lib.check(lib.t2fw_dfw_backward_blocks(P(go), P(gs), P(q), P(k), P(delta), P(fin), *[P(t) for t in shares], B, T, D, 64, code, flags, st))
    size = lib.t2fw_dfw_backward_sums_workspace_bytes(B, T, D, 64, code, flags)
    ws = torch.empty(size, dtype=torch.uint8, device="cuda")
    sums = [torch.empty_like(t) for t in (q, k, v, s)]
    _lib.check(lib.t2fw_dfw_backward_sums(P(go), P(gs), P(q), P(k), P(delta), P(fin), *[P(t) for t in sums], B, T, D, 64, code, flags, P(ws), size, st))
    ins = [t.double().requires_grad_() for t in (q, k, v, s)]
    want = torch.autograd.grad(DFWFunction.apply(*ins), ins, (go.double(), gs.double()))
    for i in range(2):
        err = lambda t: ((t.double() - want[i]).norm() / want[i].norm()).item()
        assert err(sums[i]) <= 1.01 * err(shares[i].float().sum(1).to(dtype)), (i, err(sums[i]), err(shares[i].float().sum(1).to(dtype)))
