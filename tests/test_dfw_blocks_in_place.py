"""Delta rule, value widths 64 n read and written in place by the matrix-core kernels (t2fw_dfw_forward_blocks, and
t2fw_dfw_backward_sums or, for float16 tensors, t2fw_dfw_backward_blocks): the bits of the same kernels on copies of the blocks, at the edges of their blocks of 16 and
stages of 32 steps, and the arrays that they leave to the copies."""
import pytest
import torch

from tests.test_dfw_gpu import make_inputs

pytestmark = pytest.mark.gpu


def _on_copies(q, k, v, s, go, gs, nd):
    from t2fw_amd import functional_dfw as F
    B, T, D = v.shape
    cut = lambda t: t.view(B, T, nd, 64).transpose(1, 2).reshape(B * nd, T, 64).contiguous()
    join = lambda t: t.view(B, nd, T, 64).transpose(1, 2).reshape(B, T, D)
    rep = lambda t: t.unsqueeze(1).expand(B, nd, T, 64).reshape(B * nd, T, 64).contiguous()
    out, fin, delta = F._dfw_forward(rep(q), rep(k), cut(v), s.view(B * nd, 64, 64))
    d_q, d_k, d_v, d_s = F._dfw_backward(cut(go), gs.view(B * nd, 64, 64), rep(q), rep(k), delta, fin)
    total = lambda t: sum(t.view(B, nd, T, 64).float().unbind(1)).to(t.dtype)
    return join(out), fin.view(B, D, 64), total(d_q), total(d_k), join(d_v), d_s.view(B, D, 64)


def _apply(q, k, v, s, go, gs, change_after=False):
    from t2fw_amd.functional_dfw import DFWFunction
    ins = [t.detach().requires_grad_(True) for t in (q, k, v, s)]
    args = [t * 1 for t in ins] if change_after else ins
    out, fin = DFWFunction.apply(*args)
    if change_after:
        with torch.no_grad():
            args[0].zero_()
            args[1].zero_()
    return (out.detach(), fin.detach()) + torch.autograd.grad([out, fin], ins, [go, gs])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,T,nd", [(1, 1, 2), (3, 15, 2), (2, 16, 3), (2, 17, 2), (9, 32, 2), (2, 33, 4), (1, 64, 2), (2, 95, 5), (5, 129, 2)])
def test_same_bits_as_on_copies(dtype, B, T, nd):
    ts = [t.cuda() for t in make_inputs(B, T, 64 * nd, 64, dtype, seed=T + nd)]
    for a, b in zip(_apply(*ts), _on_copies(*ts, nd)):
        assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("which", [0, 1, 2, 4, 5])
def test_arrays_that_are_not_aligned(which):
    """one array starts an element after an aligned address: copies (inputs), or moved before the kernels (gradients).
    (With such a state the exact kernels run, as for 64 channels.)"""
    ts = [t.cuda() for t in make_inputs(2, 40, 128, 64, torch.bfloat16, seed=3)]
    want = _apply(*ts)
    room = torch.empty(ts[which].numel() + 1, dtype=torch.bfloat16, device="cuda")
    ts[which] = room[1:].view(ts[which].shape).copy_(ts[which])
    assert ts[which].data_ptr() % 16 and ts[which].is_contiguous()
    for a, b in zip(_apply(*ts), want):
        assert torch.equal(a, b)


def test_queries_and_keys_may_change_before_the_backward():
    ts = [t.cuda() for t in make_inputs(2, 40, 128, 64, torch.float32, seed=4)]
    for a, b in zip(_apply(*ts, change_after=True), _apply(*ts)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T", [1, 33])
def test_per_step_kernels_asked_for_between_forward_and_backward(dtype, T, monkeypatch):
    """the backward reads T2FW_FLAGS for itself: the per-step kernels, on the blocks that the forward left whole"""
    from t2fw_amd import functional_dfw as F
    q, k, v, s, go, gs = [t.cuda() for t in make_inputs(2, T, 192, 64, dtype, seed=5)]
    ins = [t.detach().requires_grad_(True) for t in (q, k, v, s)]
    res = F.DFWFunction.apply(*ins)
    kept = res[0].grad_fn.saved_tensors
    monkeypatch.setenv("T2FW_FLAGS", "1")
    got = torch.autograd.grad(res, ins, [go, gs])
    cut = lambda t: t.view(2, T, 3, 64).transpose(1, 2).reshape(6, T, 64).contiguous()
    rep = lambda t: t.unsqueeze(1).expand(2, 3, T, 64).reshape(6, T, 64).contiguous()
    d_q, d_k, d_v, d_s = F._dfw_backward(cut(go), gs.view(6, 64, 64), rep(q), rep(k), cut(kept[2]), kept[3].view(6, 64, 64))
    total = lambda t: sum(t.view(2, 3, T, 64).float().unbind(1)).to(dtype)
    want = total(d_q), total(d_k), d_v.view(2, 3, T, 64).transpose(1, 2).reshape(2, T, 192), d_s.view(2, 192, 64)
    for a, b in zip(got, want):
        assert a.shape == b.shape and torch.equal(a, b)


def test_what_the_entry_points_refuse():
    from t2fw_amd import _lib
    lib = _lib.load()
    t = [torch.zeros(1 << 16, device="cuda") for _ in range(7)]
    p = [_lib.ptr(x) for x in t]
    call = lambda ptrs, *a: lib.t2fw_dfw_forward_blocks(*ptrs, *a, None)
    assert call(p, 1, 1, 128, 64, _lib.F32, 0) == 0
    for bad in ((1, 1, 100, 64, _lib.F32, 0), (1, 1, 128, 128, _lib.F32, 0), (1, 1, 128, 64, _lib.F64, 0), (1, 0, 128, 64, _lib.F32, 0),
                (1, 1, 128, 64, _lib.F32, _lib.FLAG_FORCE_SCAN), (1, 1 << 25, 128, 64, _lib.F32, 0), (1, 1, 128, 64, 99, 0)):
        assert call(p, *bad) != 0, bad
    assert call(p[:2] + [_lib.ctypes.c_void_p(t[2].data_ptr() + 4)] + p[3:], 1, 1, 128, 64, _lib.F32, 0) != 0
    torch.cuda.synchronize()
