"""Training steps whose forward hints no row (every gate in the chunk-parallel backward's range) while values of a size that bfloat16
holds take an intermediate of it out of range: the row is declined for its results, and the launch that redoes it has to be there.
The hints are about gates alone.  Against the same step with the choice left to the device."""
import pytest
import torch

from t2fw_amd.synthetic import make_config_inputs


def test_no_hint_skips_the_extra_launch_for_small_values_only():
    from t2fw_amd import _lib
    from t2fw_amd.path_hint import choose_backward_flags as choose
    assert choose(0, 0, 96, True) == _lib.FLAG_NO_FIXUP and choose(0, 0, 96, False) == 0
    assert choose(0, None, 96, False) == 0 and choose(0, 96, 96, False) == choose(0, 96, 96, True) == _lib.FLAG_BLOCKWISE


# a gate of 1/4 on one channel (2^-64 over half a chunk, 2^-32 over 16 steps), or 16 steps of 0.05 in each half (2^-69 over 16 steps,
# where only the forward with the chunks of a row side by side sets no hint); lengths of either forward
@pytest.mark.gpu
@pytest.mark.parametrize("T", [128, 64 * 120])
@pytest.mark.parametrize("gates", ["quarter", "sixteen_small"])
@pytest.mark.parametrize("heads", [False, True])
def test_large_gradients_in_bfloat16(T, gates, heads, monkeypatch):
    from t2fw_amd import LFWFunction, LFWHeadsFunction
    x, f, q, k, fk, s, go, gs = make_config_inputs(4, T, 64, 64, torch.bfloat16, seed=40, gate_mean=3.0, state_std=0.1)
    if gates == "quarter":
        f[1, :, 0] = 0.25
    else:
        f[1, :, 0] = 1.0
        f[1].view(-1, 32, 64)[:, :16, 0] = 0.05
    go[1, :, 0] = 2.0 ** 60
    q[1], k[1] = 8.0, 8.0
    ins, go, gs = [t.cuda() for t in (x, f, q, k, fk, s)], go.cuda(), gs.cuda()
    fn = LFWFunction
    if heads:
        ins = [t.unsqueeze(2) for t in ins[:5]] + [ins[5].unsqueeze(1)]
        go, gs, fn = go.unsqueeze(2), gs.unsqueeze(1), LFWHeadsFunction
    got = []
    for hints in ("1", "0"):
        monkeypatch.setenv("T2FW_HOST_HINTS", hints)
        args = [t.clone().requires_grad_() for t in ins]
        res = fn.apply(*args)
        torch.cuda.synchronize()                     # the forward has completed: its hints are readable
        got.append(torch.autograd.grad(res, args, (go, gs)))
    for a, b in zip(*got):
        assert torch.isfinite(b).all()
        for r in range(4):                           # (another backward kernel where the row is hinted; bounds of tests/test_magnitudes_gpu.py)
            d, n = (a[r].double() - b[r].double()).norm(), b[r].double().norm()
            assert d <= (6e-2 if r == 1 else 2e-2) * n, r
