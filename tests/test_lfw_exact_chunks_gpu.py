"""The chunk-parallel exact kernels of the decay rule (T2FW_FLAG_EXACT_CHUNKS: float32 tensors, widths of up to 64)
against the float64 oracle, at the tolerance of the per-step kernels (TOL of test_lfw_gpu).  Sizes sit on the edges of the
kernels' pieces (8, 16 and 64 steps, 16 and 32 channels, eight chunks of the chain)."""
import pytest
import torch

from tests.lfw_cases import make_config_inputs, make_reference_test_inputs
from tests.test_lfw_gpu import NAMES, TOL, assert_close, check_all, oracle_all

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def exact_chunks(monkeypatch):
    monkeypatch.setenv("T2FW_FLAGS", "32")


F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


@pytest.mark.parametrize("B,T,D,K,dtype", [
    (1, 1, 64, 64, F32), (2, 7, 64, 64, F32), (2, 8, 64, 64, F32), (2, 9, 64, 64, F32), (2, 17, 64, 64, F32),
    (3, 64, 64, 64, F32), (2, 65, 64, 64, F32), (2, 127, 64, 64, F32), (2, 1000, 64, 64, F32), (2, 80, 1, 1, F32),
    (2, 8 * 64, 64, 64, F32), (2, 8 * 64 + 1, 64, 64, F32), (2, 13 * 64 - 5, 64, 64, F32), (2, 17 * 64 + 2, 64, 64, F32),
    (2, 8 * 64 + 1, 20, 40, F32), (2, 12 * 64, 40, 20, F32), (2, 15 * 64 - 1, 20, 40, F16), (1, 25 * 64 + 9, 9, 7, F32),
    (2, 80, 16, 17, F32), (1, 200, 63, 48, F32), (2, 65, 33, 64, F32), (2, 130, 64, 32, F32),
    (2, 150, 17, 5, F16), (2, 64, 64, 49, F16), (2, 150, 31, 32, BF16),
])
def test_edges(B, T, D, K, dtype):
    x, f, q, k, fk, s, go, gs = make_config_inputs(B, T, D, K, dtype, seed=T + D, in_scale=0.5, state_std=0.5, gate_mean=1.5)
    check_all((x, f, q, k, fk, s), go, gs, dtype)


def test_gates_down_to_one_sixty_fourth():
    x, f, q, k, fk, s, go, gs = make_reference_test_inputs(3, 300, 64, 64, F32, seed=5)
    check_all((x, f, q, k, fk, s), go, gs, F32)


@pytest.mark.parametrize("what", ["zero", "tiny", "above one", "one side's product overflows", "negative", "large values"])
@pytest.mark.parametrize("D,K,dtype", [(64, 64, F32), (20, 40, F32), (20, 40, BF16)])
def test_unusual_gates_and_values(what, D, K, dtype):
    """One row of three is out of the ordinary; gates above one send it through the whole sequence step by step."""
    x, f, q, k, fk, s, go, gs = make_config_inputs(3, 150, D, K, dtype, seed=3, in_scale=0.5, state_std=0.5)
    if what == "zero":
        f[1, 70, 3] = 0
        fk[1, 5, 7] = 0
        fk[2, 149, 0] = 0
    elif what == "tiny":
        f[1, 64:80] = 2.0 ** -20
    elif what == "above one":
        fk[1, 100, 2] = 1.25
    elif what == "one side's product overflows":
        f[1, :, :] = 2.0 ** -6
        fk[1, :, :] = 2.0 ** 5
    elif what == "negative":
        f[0, 30, 1] = -0.5
    else:
        x[1, 90] *= 2.0 ** 42
    check_all((x, f, q, k, fk, s), go, gs, dtype)


@pytest.mark.parametrize("T", [40, 100, 250, 400])
@pytest.mark.parametrize("D,K", [(64, 64), (33, 40)])
def test_rows_left_next_to_others(T, D, K):
    """Rows with a gate above one run step by step, on the workgroups of up to four of their chunks: one chunk to seven."""
    x, f, q, k, fk, s, go, gs = make_config_inputs(5, T, D, K, F32, seed=T, in_scale=0.5, state_std=0.5)
    f[1, T // 2, 3] = 1.25
    fk[4, 0, 7] = 1.25
    check_all((x, f, q, k, fk, s), go, gs, F32)


def _gate_gradients(x, f, q, k, fk, s, go, gs):
    """d_f and d_f_key in float64, and for each element the sum of the magnitudes of all products that it is made of"""
    x, f, q, k, fk, S, go, G = (t.double() for t in (x, f, q, k, fk, s, go, gs))
    T, A, H = x.shape[1], S.abs(), G.abs()
    outer = lambda a, b: a.unsqueeze(2) * b.unsqueeze(1)
    before = []
    for t in range(T):
        before.append((S, A))
        w = outer(f[:, t], fk[:, t])
        S, A = S * w + outer(x[:, t], k[:, t]), A * w + outer(x[:, t], k[:, t]).abs()
    grads, sizes = [[], []], [[], []]
    for t in reversed(range(T)):
        g = outer(go[:, t], q[:, t])
        G, H = G + g, H + g.abs()
        for out, w in ((grads, G * before[t][0]), (sizes, H * before[t][1])):
            out[0].append((w * fk[:, t].unsqueeze(1)).sum(2))
            out[1].append((w * f[:, t].unsqueeze(2)).sum(1))
        w = outer(f[:, t], fk[:, t])
        G, H = G * w, H * w
    back = lambda ts: torch.stack(ts[::-1], 1)
    return [(back(grads[i]), back(sizes[i])) for i in range(2)]


def check_gate_gradients(x, f, q, k, fk, s, go, gs):
    """Every gate gradient by itself, in units of the magnitudes that it is the sum of.  Bound: a product that is carried over n
    steps is rounded 2 n times in fp32 (the gates' product and the state), 2^-24 each and independent; where one product outweighs the
    rest that is sqrt(2 n) 2^-24, n up to 150, and twice that over so many elements.  The per-step kernels use 0.3 of it."""
    from t2fw_amd import LFWFunction
    assert x.shape[1] <= 150
    want = _gate_gradients(x, f, q, k, fk, s, go, gs)
    ins = [t.cuda().requires_grad_() for t in (x, f, q, k, fk, s)]
    got = torch.autograd.grad(LFWFunction.apply(*ins), [ins[1], ins[4]], [go.cuda(), gs.cuda()])
    for n, g, (w, size) in zip(("d_f", "d_f_key"), got, want):
        used = ((g.double().cpu() - w).abs() / (2 * 300 ** 0.5 * 2.0 ** -24 * size).clamp_min(1e-40)).max().item()
        print("%s: %.3g of the bound" % (n, used), flush=True)
        assert used <= 1, n


@pytest.mark.parametrize("what,value", [("one gate", 2.0 ** -20), ("one gate", 2.0 ** -21), ("whole chunk", 2.0 ** -6.2),
                                        ("whole chunk", 2.0 ** -6.3), ("every second gate", 2.0 ** -16), ("tiny gradients", 1e-30),
                                        ("large value", 2.0 ** 29), ("large value", 2.0 ** 31), ("large value", 2.0 ** 57), ("large value", 2.0 ** 59),
                                        ("large state", 2.0 ** 29), ("large state", 2.0 ** 31), ("large state", 2.0 ** 121)])
def test_limits_of_the_matrix_form(what, value):
    """64 x 64 float32: on both sides of each limit of the products (a chunk beyond one runs step by step, a row with inputs beyond
    2^58 or states beyond 2^120 over the whole sequence), with a chunk in range and a ragged one next to it.  T = 150: chunks of 64,
    64 and 22 steps."""
    x, f, q, k, fk, s, go, gs = make_config_inputs(2, 150, 64, 64, F32, seed=11, in_scale=0.5, state_std=0.5)
    if what == "one gate":
        f[0, 70, 3] = fk[0, 140, 5] = fk[1, 0, 0] = value
    elif what == "whole chunk":
        f[0, 64:128, 7] = value
        fk[1, 0:64, 9] = value
    elif what == "every second gate":
        f[0, ::2, 11] = fk[0, 1::2, 13] = value
    elif what == "tiny gradients":
        go[0], gs[0] = go[0] * value, gs[0] * value
    elif what == "large value":
        x[0, 80, 3] = value
        q[1, 80, 3] = value
    else:
        s[0, 5, 6] = value
        f[0, :, 5] = 0.5
    check_all((x, f, q, k, fk, s), go, gs, F32)
    check_gate_gradients(x, f, q, k, fk, s, go, gs)


@pytest.mark.parametrize("what,value,gate,tokens", [
    ("value", 1e6, 2.0 ** -20, 2), ("value", 1e9, 2.0 ** -20, 3), ("value", 1e10, 2.0 ** -20, 3), ("value", 1e12, 2.0 ** -20, 3),
    ("value", 1e15, 2.0 ** -10, 8), ("value, both gates", 1e5, 2.0 ** -20, 2),
    ("both gates", 1, 2.0 ** -20, 1), ("both gates", 1, 2.0 ** -17, 1), ("both gates", 1, 2.0 ** -12, 1), ("both gates", 1, 2.0 ** -20, 10),
    ("step", 1e9, 0.1, 45), ("step", 1e12, 0.1, 45), ("step", 1e15, 0.1, 45), ("query", 1e12, 2.0 ** -10, 6),
    ("loss ends", 0, 1, 1), ("loss ends, no state gradient", 0, 1, 1), ("no state", 0, 1, 1), ("gates of all sizes", 0, 1, 1),
    ("as usual", 0, 1, 1)])
def test_gate_gradients_element_by_element(what, value, gate, tokens):
    """A large value that small gates make the state forget, tokens whose gates are small on both sides, a loss that ends within a
    chunk.  T = 150: chunks of 64, 64 and 22 steps; the first and the last are out of the ordinary, in another row each."""
    x, f, q, k, fk, s, go, gs = make_config_inputs(3, 150, 64, 64, F32, seed=21, in_scale=0.125, state_std=0.1)
    for b, t in ((0, 5), (1, 130)):
        later = slice(t + 1, t + 1 + min(tokens, 150 - t - 1)) if what == "step" else slice(t + 10, t + 10 + tokens)
        if what.startswith("value"):
            x[b, t, 3] = value
            f[b, later, 3] = gate
        if what.endswith("both gates"):
            f[b, later], fk[b, later] = gate, gate
        if what == "step":
            x[b, t] *= value
            f[b, later], fk[b, later] = gate, 0.5
        if what == "query":
            q[b, t + 9, 3] = value
            fk[b, later, 3] = gate
    if what.startswith("loss ends"):
        go[0, 40:], go[1, 133:] = 0, 0
        gs[:2] = 0 if "no state" in what else gs[:2] * 1e-12
    if what == "no state":
        s[:] = 0
    if what == "gates of all sizes":             # 1/64 to 63/64, one per channel
        f[:] = fk[:] = torch.linspace(1 / 64, 63 / 64, 64)
    check_gate_gradients(x, f, q, k, fk, s, go, gs)


@pytest.mark.parametrize("value,small", [(2.0 ** 55, 2.0 ** -50), (2.0 ** 40, 2.0 ** -50), (2.0 ** 31, 2.0 ** -45), (2.0 ** 27, 2.0 ** -45), (1.0, 2.0 ** -45)])
def test_outputs_of_small_queries_after_a_large_value(value, small):
    """A value that key gates of 1/4 make the state forget, queries and keys so small that what is left of it is at the end of fp32's
    range: every output by itself, in units of the magnitudes that it is the sum of (bound as in the test above)."""
    from t2fw_amd import LFWFunction
    x, f, q, k, fk, s, go, gs = make_config_inputs(2, 100, 64, 64, F32, seed=22, in_scale=1.0, state_std=0.0)
    q, k = q * small, k * small
    f[:] = 1
    fk[:] = 0.9
    fk[0, 6:36] = 0.25
    x[0, 5] *= value
    S = A = s.double()
    want, size = [], []
    for t in range(100):
        w, xk = f[:, t].double().unsqueeze(2) * fk[:, t].double().unsqueeze(1), x[:, t].double().unsqueeze(2) * k[:, t].double().unsqueeze(1)
        S, A = S * w + xk, A * w + xk.abs()
        want.append((S @ q[:, t].double().unsqueeze(2)).squeeze(2))
        size.append((A @ q[:, t].double().abs().unsqueeze(2)).squeeze(2))
    with torch.no_grad():
        got = LFWFunction.apply(*[t.cuda() for t in (x, f, q, k, fk, s)])[0].double().cpu()
    used = ((got - torch.stack(want, 1)).abs() / (2 * 200 ** 0.5 * 2.0 ** -24 * torch.stack(size, 1))).max().item()
    print("outputs: %.3g of the bound" % used, flush=True)
    assert used <= 1


def test_error_of_the_matrix_form():
    """Relative error (2-norm) against the float64 kernels: what tokens share with tokens is fp64 but for P, rounded to fp32
    once, and the result is rounded once (2.4e-8 each); checkpoints, the adjoint between chunks and the products with them
    are fp32 sums (8e-8 of the part that a chunk's first and last tokens have of them).  Step by step the gate gradients
    are at 1.0e-7."""
    from t2fw_amd import LFWFunction
    x, f, q, k, fk, s, go, gs = make_config_inputs(8, 300, 64, 64, F32, seed=12)

    def run(dtype):
        ins = [t.cuda().to(dtype).requires_grad_() for t in (x, f, q, k, fk, s)]
        res = LFWFunction.apply(*ins)
        return list(res) + list(torch.autograd.grad(res, ins, [go.cuda().to(dtype), gs.cuda().to(dtype)]))

    for n, got, want in zip(("outputs", "next_state") + NAMES, run(F32), run(torch.float64)):
        assert ((got.double() - want).norm() / want.norm()).item() < 6e-8, n


def test_rows_left_take_no_longer_than_the_per_step_kernels(monkeypatch):
    """Every row of 96 x 1024 steps has a gate above one.  Measured 1.03 times the per-step kernels' time; 7.4 times when
    the workgroups that do such rows shared one die."""
    from t2fw_amd import LFWFunction
    ins = [t.cuda().requires_grad_() for t in make_config_inputs(96, 1024, 64, 64, F32, seed=2)[:6]]
    with torch.no_grad():
        ins[1][:, 500, 0] = 1.25
    grads = [torch.ones(96, 1024, 64, device="cuda"), torch.ones(96, 64, 64, device="cuda")]

    def fastest(flags):
        monkeypatch.setenv("T2FW_FLAGS", flags)
        best = float("inf")
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            torch.autograd.grad(LFWFunction.apply(*ins), ins, grads)
            b.record()
            b.synchronize()
            best = min(best, a.elapsed_time(b))
        return best

    assert fastest("32") < 2 * fastest("1")


def _same_where_finite(got, want, what, tol):
    got, want = got.detach().double().cpu(), want.detach().double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want)), what
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(got)], want[torch.isinf(want)]), what
    for g, w in zip(got, want):                            # row by row: one holds very large values
        ok = torch.isfinite(w)
        assert ((g - w)[ok].abs() <= tol[0] * w[ok].abs() + tol[1] * w[ok].abs().max()).all(), what


@pytest.mark.parametrize("what", ["infinite states, fast decay", "a product overflows, then decays", "the state overflows between chunks"])
@pytest.mark.parametrize("D,K,dtype", [(64, 64, F32), (20, 40, F32), (20, 40, BF16)])
def test_infinities_as_step_by_step(what, D, K, dtype, monkeypatch):
    """What the recurrence makes infinite stays so: the per-step kernels are the reference (sums differ in order only:
    their tolerance, per row)."""
    from t2fw_amd import LFWFunction
    T = 200
    x, f, q, k, fk, s, go, gs = make_config_inputs(3, T, D, K, dtype, seed=8, in_scale=0.5, state_std=0.5)
    if what == "infinite states, fast decay":
        s[1, 3, 5] = float("inf")
        gs[1, 2, 2] = float("-inf")
        f[1], fk[1] = 2.0 ** -6, 2.0 ** -6                 # a chunk's gate product is zero in fp32
    elif what == "a product overflows, then decays":
        f[1], fk[1] = 0.5, 0.5
        x[1, 70, 3], k[1, 70, 5] = 1e30, 1e30
        go[1, 120, 2], q[1, 120, 4] = 1e30, 1e30
    else:
        s[1, 3, 5] = 3e38
        x[1, 10, 3], k[1, 10, 5] = 1e19, 1e19
        f[1], fk[1] = 1.0, 1.0
        f[1, 140:], fk[1, 140:] = 2.0 ** -6, 2.0 ** -6
        x[1, :, 3] = x[1, :, 3].abs()
        k[1, :, 5] = k[1, :, 5].abs()

    def run(flags):
        monkeypatch.setenv("T2FW_FLAGS", flags)
        ins = [t.cuda().requires_grad_() for t in (x, f, q, k, fk, s)]
        res = LFWFunction.apply(*ins)
        return list(res) + list(torch.autograd.grad(res, ins, [go.cuda(), gs.cuda()]))

    want = run("1")
    assert not all(torch.isfinite(t).all() for t in want)
    for n, g, w in zip(("outputs", "next_state") + NAMES, run("32"), want):
        _same_where_finite(g, w, n, TOL[dtype])


def test_nan_stays_in_its_row():
    from t2fw_amd import LFWFunction
    ins = [t.cuda() for t in make_config_inputs(3, 150, 64, 64, F32, seed=4)[:6]]
    ref = LFWFunction.apply(*ins)
    ins[0][1, 70, 5] = float("nan")
    out, nxt = LFWFunction.apply(*ins)
    for a, r in ((out, ref[0]), (nxt, ref[1])):
        assert torch.equal(a[[0, 2]], r[[0, 2]])
    assert torch.isnan(out[1, 70:, 5]).all()
    # the row now runs step by step from its first state: the same terms, chunk states rounded in another order (both
    # orders are within TOL[F32] of the exact sums)
    assert_close(out[1, :70], ref[0][1, :70].cpu(), F32, "outputs before the NaN", tol=TOL[F32])


def test_head_strided_tensors():
    from t2fw_amd import LFWHeadsFunction
    B, T, H = 2, 100, 3
    heads = lambda t: t.view(B, H, T, -1).transpose(1, 2).contiguous().cuda()
    rows = lambda t: t.transpose(1, 2).reshape(B * H, T, -1)
    for D, K in ((64, 64), (40, 24)):
        x, f, q, k, fk, s, go, gs = make_config_inputs(B * H, T, D, K, F32, seed=9, in_scale=0.5, state_std=0.5)
        st = lambda t: t.view(B, H, D, K).contiguous().cuda()
        ins = [heads(t).requires_grad_() for t in (x, f, q, k, fk)] + [st(s).requires_grad_()]
        out, nxt = LFWHeadsFunction.apply(*ins)
        grads = torch.autograd.grad([out, nxt], ins, [heads(go), st(gs)])
        r_out, r_nxt, r_grads = oracle_all((x, f, q, k, fk, s), go, gs)
        assert_close(rows(out), r_out, F32, "outputs", tol=TOL[F32])
        assert_close(nxt.reshape(B * H, D, K), r_nxt, F32, "next_state", tol=TOL[F32])
        for n, g, r in zip(NAMES, grads, r_grads):
            assert_close(g.reshape(B * H, D, K) if n == "d_state" else rows(g), r, F32, n, tol=TOL[F32])
