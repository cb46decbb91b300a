"""The fp32 matrix-core kernels of the decay rule (T2FW_FLAG_TILES: float32 tensors, widths of up to 64) against the
float64 oracle, at the tolerance of the exact kernels (TOL of test_lfw_gpu).  Sizes sit on the edges of the kernels'
tiles (16 steps, 64 steps, 16 channels)."""
import pytest
import torch

from tests.lfw_cases import make_config_inputs, make_reference_test_inputs
from tests.test_lfw_gpu import NAMES, TOL, assert_close, check_all, oracle_all

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def tiles(monkeypatch):
    monkeypatch.setenv("T2FW_FLAGS", "32")


F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


@pytest.mark.parametrize("B,T,D,K,dtype", [
    (1, 16, 64, 64, F32), (2, 17, 64, 64, F32), (3, 64, 64, 64, F32), (2, 127, 64, 64, F32), (2, 129, 64, 64, F32),
    (2, 1000, 64, 64, F32), (2, 80, 1, 1, F32), (2, 80, 16, 17, F32), (1, 200, 63, 48, F32), (2, 65, 33, 64, F32),
    (2, 150, 17, 5, F16), (2, 64, 64, 49, F16), (2, 150, 31, 32, BF16),
])
def test_tile_edges(B, T, D, K, dtype):
    x, f, q, k, fk, s, go, gs = make_config_inputs(B, T, D, K, dtype, seed=T + D, in_scale=0.5, state_std=0.5, gate_mean=1.5)
    check_all((x, f, q, k, fk, s), go, gs, dtype)


def test_reference_gates_down_to_one_sixty_fourth():
    x, f, q, k, fk, s, go, gs = make_reference_test_inputs(3, 300, 64, 64, F32, seed=5)
    check_all((x, f, q, k, fk, s), go, gs, F32)


@pytest.mark.parametrize("what", ["zero", "tiny", "above one", "negative", "large values", "large state", "large gradient"])
@pytest.mark.parametrize("D,K,dtype", [(64, 64, F32), (20, 40, F32), (20, 40, BF16)])
def test_what_the_tiles_cannot_hold_runs_exactly(what, D, K, dtype):
    """One chunk of one row takes the exact recurrence, its neighbours do not; T ragged.  Large values: 2^40 and more
    are out of the operands' range; the tensors they reach are compared relative to their own largest element."""
    x, f, q, k, fk, s, go, gs = make_config_inputs(3, 150, D, K, dtype, seed=3, in_scale=0.5, state_std=0.5)
    if what == "zero":
        f[1, 70, 3] = 0
        fk[1, 5, 7] = 0
        fk[2, 149, 0] = 0
    elif what == "tiny":
        f[1, 64:80] = 2.0 ** -20
    elif what == "above one":
        fk[1, 100, 2] = 1.25
    elif what == "negative":
        f[0, 30, 1] = -0.5
    elif what == "large values":
        x[1, 90] *= 2.0 ** 42
    elif what == "large state":
        s[1] *= 2.0 ** 90
    else:
        gs[1] *= 2.0 ** 90
    check_all((x, f, q, k, fk, s), go, gs, dtype)


def test_head_strided_tensors():
    from t2fw_amd import LFWHeadsFunction
    B, T, H, D, K = 2, 100, 3, 40, 24
    x, f, q, k, fk, s, go, gs = make_config_inputs(B * H, T, D, K, F32, seed=9, in_scale=0.5, state_std=0.5)
    heads = lambda t: t.view(B, H, T, -1).transpose(1, 2).contiguous().cuda()
    st = lambda t: t.view(B, H, D, K).contiguous().cuda()
    ins = [heads(t).requires_grad_() for t in (x, f, q, k, fk)] + [st(s).requires_grad_()]
    out, nxt = LFWHeadsFunction.apply(*ins)
    grads = torch.autograd.grad([out, nxt], ins, [heads(go), st(gs)])
    r_out, r_nxt, r_grads = oracle_all((x, f, q, k, fk, s), go, gs)
    rows = lambda t: t.transpose(1, 2).reshape(B * H, T, -1)
    assert_close(rows(out), r_out, F32, "outputs", tol=TOL[F32])
    assert_close(nxt.reshape(B * H, D, K), r_nxt, F32, "next_state", tol=TOL[F32])
    for n, g, r in zip(NAMES, grads, r_grads):
        assert_close(g.reshape(B * H, D, K) if n == "d_state" else rows(g), r, F32, n, tol=TOL[F32])
