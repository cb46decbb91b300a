"""The forward with the chunks of a row side by side (csrc/lfw_par_fwd.hip): few rows of many steps, at the edges of its chunks of 64 and
of its batches of sixteen chunks, with and without heads and checkpoints, against the oracle and the sequential kernel
(T2FW_FLAG_BLOCKWISE keeps the forward there); rows that it hands over; the rule that chooses it."""
import pytest
import torch

from t2fw_amd.synthetic import make_config_inputs


def run(lib_call_flags, ins, H=1, C=64, ckpt=True):
    """(out, next, checkpoints, rows flagged, rows hinted, scratch bytes); inputs [B,T,64] or, with H > 1, [B,T,H,64]"""
    from t2fw_amd import _lib
    lib = _lib.load()
    x, f, q, k, fk, s = ins
    B, T = x.shape[:2]
    rows, code = B * H, _lib.DTYPE_CODE[x.dtype]
    out, nxt = torch.full_like(x, float("nan")), torch.full_like(s, float("nan"))
    ck = torch.full((rows, -(-T // C), 64, 64), float("nan"), dtype=x.dtype, device="cuda") if ckpt else None
    n = lib.t2fw_lfw_forward_workspace_bytes(rows, T, 64, 64, C, code, lib_call_flags)
    ws = torch.full((n,), 255, dtype=torch.uint8, device="cuda")
    extra = lib.t2fw_lfw_forward_scratch_bytes(B, T, H, 64, 64, C, code, lib_call_flags, ckpt)
    scratch = torch.full((extra + 4096,), 255, dtype=torch.uint8, device="cuda")
    P = _lib.ptr
    _lib.check(lib.t2fw_lfw_forward_scratch(P(x), P(f), P(q), P(k), P(fk), P(s), P(out), P(nxt), P(ck), B, T, H, 64, 64, C, code, lib_call_flags,
                                            P(ws), n, P(scratch), extra, _lib.current_stream_handle(x.device)))
    torch.cuda.synchronize()
    assert (scratch[extra:] == 255).all()
    pad = -(-rows // 8) * 8
    slots = ws.view(torch.int32).view(2, -1)[:, :2 * pad].view(2, 2, pad)[:, :, :rows].amax(1).cpu()
    return out, nxt, ck, slots[0], slots[1], extra


def inputs(B, T, dtype, seed, mean=2.0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = lambda *s: (torch.randn(s, generator=g, device="cuda") * 0.3).to(dtype)
    z = lambda *s: torch.sigmoid(torch.randn(s, generator=g, device="cuda") + mean).to(dtype)
    return [n(B, T, 64), z(B, T, 64), n(B, T, 64), n(B, T, 64), z(B, T, 64), n(B, 64, 64)]


def rel(a, b):
    return ((a.double() - b.double()).norm() / b.double().norm()).item()


def exact(ins):
    from t2fw_amd import LFWFunction
    with torch.no_grad():
        return LFWFunction.apply(*[t.double() for t in ins])           # the per-step kernels in float64


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,T", [(1, 833), (1, 1023), (2, 1024), (3, 1025), (9, 1087), (8, 1089), (1, 2048), (2, 2049), (33, 1100)])
def test_lengths_around_the_edges(dtype, B, T):
    """errors against float64 at most 1.1 times the sequential kernel's"""
    ins = inputs(B, T, dtype, seed=T)
    out, nxt, _, flags, hints, extra = run(0, ins, ckpt=False)
    assert extra > 0 and not flags.any() and not hints.any()
    s_out, s_nxt, _, _, _, none = run(8, ins, ckpt=False)
    assert none == 0
    r_out, r_nxt = exact(ins)
    assert rel(out, r_out) <= max(1.1 * rel(s_out, r_out), 1e-3), (rel(out, r_out), rel(s_out, r_out))
    assert rel(nxt, r_nxt) <= max(1.1 * rel(s_nxt, r_nxt), 1e-3), (rel(nxt, r_nxt), rel(s_nxt, r_nxt))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_checkpoints_and_heads(dtype):
    """checkpoints are the states that the sequential kernel leaves, to the rounding of either; heads are rows"""
    T = 64 * 125 - 7
    ins = inputs(8, T, dtype, seed=5, mean=3.0)
    out, nxt, ck, _, _, extra = run(0, ins)
    assert extra > 0
    s_out, s_nxt, s_ck, *_ = run(8, ins)
    for a, b in ((out, s_out), (nxt, s_nxt), (ck, s_ck)):
        assert rel(a, b) < 1e-2
    heads = [t.view(2, 4, T, 64).transpose(1, 2).contiguous() for t in ins[:5]] + [ins[5].view(2, 4, 64, 64)]
    h_out, h_nxt, h_ck, _, _, extra = run(0, heads, H=4)
    assert extra > 0
    assert torch.equal(h_out.transpose(1, 2).reshape(8, T, 64), out) and torch.equal(h_nxt.view(8, 64, 64), nxt) and torch.equal(h_ck, ck)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_rows_that_are_handed_over(dtype):
    """a gate above one, gates too small for a whole half chunk, a NaN among the values, an infinity among the queries: the sequential
    kernel's results for these rows, the others as they were"""
    ins = inputs(6, 1000, dtype, seed=6)
    clean = run(0, ins, ckpt=False)
    bad = [t.clone() for t in ins]
    bad[1][1, 700, 3] = 1.5
    bad[4][2, 64:96, 9] = 0.05
    bad[0][3, 500, 1] = float("nan")
    bad[2][4, 999, 63] = float("inf")
    got, seq = run(0, bad, ckpt=False), run(8, bad, ckpt=False)
    rows = torch.tensor([1, 2, 3, 4])
    for a, b, c in zip(got[:2], seq[:2], clean[:2]):
        assert torch.equal(a[rows].isnan(), b[rows].isnan())
        assert torch.equal(a[rows].nan_to_num(), b[rows].nan_to_num())
        assert torch.equal(a[[0, 5]], c[[0, 5]])
    assert torch.equal(got[3], seq[3]) and torch.equal(got[4][rows], seq[4][rows])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_zero_gates_stay(dtype):
    """an exactly zero gate counts as 2^-24, as in the sequential kernel: the form takes the row"""
    ins = inputs(4, 960, dtype, seed=7)
    ins[1][:, 100, 5] = 0
    ins[4][:, 500, 7] = 0
    out, nxt, _, flags, _, extra = run(0, ins, ckpt=False)
    assert extra > 0 and not flags.any()
    r_out, r_nxt = exact(ins)
    assert rel(out, r_out) < 1e-2 and rel(nxt, r_nxt) < 1e-2


@pytest.mark.gpu
def test_training_and_graph_replay():
    """a training step that takes it: gradients as with the sequential forward; replays of a captured call are the eager one"""
    import os
    from t2fw_amd import LFWFunction
    ins = inputs(4, 64 * 122, torch.float16, seed=8, mean=3.0)
    gos = [torch.randn_like(ins[0]), torch.randn_like(ins[5])]
    grads = []
    for flags in ("", "8"):
        os.environ["T2FW_FLAGS"] = flags
        try:
            args = [t.clone().requires_grad_() for t in ins]
            res = LFWFunction.apply(*args)
            grads.append([*res, *torch.autograd.grad(res, args, gos)])
        finally:
            del os.environ["T2FW_FLAGS"]
    assert not torch.equal(grads[0][0], grads[1][0])
    for a, b in zip(*grads):
        assert rel(a, b) < 1.5e-2
    static = [t.clone() for t in ins]
    with torch.no_grad():
        LFWFunction.apply(*static)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            res = LFWFunction.apply(*static)
        for seed in (8, 9, 10):
            for t, n in zip(static, inputs(4, 64 * 122, torch.float16, seed=seed, mean=3.0)):
                t.copy_(n)
            graph.replay()
            eager = LFWFunction.apply(*static)
            torch.cuda.synchronize()
            for a, b in zip(res, eager):
                assert torch.equal(a, b)


def test_where_it_is_chosen():
    from t2fw_amd import _lib
    size = _lib.load().t2fw_lfw_forward_scratch_bytes
    items = lambda rows, chunks: rows * chunks * (16384 + 8192 + 1024) + -(-rows * chunks * 4 // 256) * 256 + -(-rows * 4 // 256) * 256
    assert size(4, 1024, 1, 64, 64, 64, _lib.F16, 0, 0) == items(4, 16) and size(2, 1024, 4, 64, 64, 64, _lib.BF16, 0, 0) == items(8, 16)
    assert size(16, 8192, 1, 64, 64, 64, _lib.F16, 0, 1) == items(16, 128) and size(4, 1024, 1, 64, 64, 32, _lib.F16, 0, 0) > 0
    for call in ((4, 1024, 1, 64, 64, 64, _lib.F32, 0, 0), (4, 1024, 1, 128, 64, 64, _lib.F16, 0, 0), (4, 1024, 1, 64, 64, 64, _lib.F16, 1, 0), (4, 1024, 1, 64, 64, 64, _lib.F16, 4, 0),
                 (4, 512, 1, 64, 64, 64, _lib.F16, 0, 0), (96, 1024, 1, 64, 64, 64, _lib.F16, 0, 0), (128, 8192, 1, 64, 64, 64, _lib.F16, 0, 1), (16, 1024, 1, 64, 64, 64, _lib.F16, 0, 1),
                 (16, 8192, 1, 64, 64, 32, _lib.F16, 0, 1), (0, 1024, 1, 64, 64, 64, _lib.F16, 0, 0), (4, 1 << 24, 1, 64, 64, 64, _lib.F16, 0, 0), (1, 1 << 23, 4, 64, 64, 64, _lib.F16, 0, 0),
                 (1 << 40, 1024, 1, 64, 64, 64, _lib.F16, 0, 0), (4, 1024, 0, 64, 64, 64, _lib.F16, 0, 0), (-1, 1024, 1, 64, 64, 64, _lib.F16, 0, 0)):
        assert size(*call) == 0, call
