"""Gates made in the same step as the forward (lfw_forward of csrc/host.cpp on logits), in training: results and gradients of the same call
on gates made before it, the gradients of the logits from those of the gates.  Widths and types of every forward that may follow."""
import pytest
import torch

from t2fw_amd.synthetic import make_config_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,D,K,dtype", [(3, 70, 64, 64, torch.float16), (3, 70, 64, 64, torch.bfloat16), (2, 64 * 122, 64, 64, torch.float16),
                                           (3, 300, 17, 33, torch.float32), (3, 300, 17, 33, torch.float16), (2, 70, 128, 64, torch.bfloat16),
                                           (2, 1, 64, 64, torch.bfloat16)])
@pytest.mark.parametrize("heads", [True, False])
def test_logits_in_training(heads, B, T, D, K, dtype):
    from t2fw_amd import LFWFunction, LFWGatedFunction, LFWHeadsFunction, sigmoid_gates
    from t2fw_amd.functional_lfw import _gate_backward_inplace
    x, f, q, k, fk, s, go, gs = [t.cuda() for t in make_config_inputs(B, T, D, K, dtype, seed=4)]
    lf, lk = torch.randn_like(f) + 2, torch.randn_like(fk) + 2
    if heads:
        x, lf, q, k, lk, go = [t.unsqueeze(2) for t in (x, lf, q, k, lk, go)]
        s, gs = s.unsqueeze(1), gs.unsqueeze(1)
    f, fk = sigmoid_gates(lf, lk)

    def step(fn, ins, *more):
        args = [t.clone().requires_grad_() for t in ins]
        res = fn.apply(*args, *more)
        torch.cuda.synchronize()
        return [*res, *torch.autograd.grad(res, args, (go, gs))]
    got = step(LFWHeadsFunction, (x, lf, q, k, lk, s), True) if heads else step(LFWGatedFunction, (x, lf, q, k, lk, s))
    want = step(LFWHeadsFunction if heads else LFWFunction, (x, f, q, k, fk, s))
    _gate_backward_inplace(want[3], want[6], f, fk)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_a_graph_of_a_training_step_on_logits():
    """replays on new logits, with eager work between them, are the eager step to the bit"""
    from t2fw_amd import LFWHeadsFunction
    make = lambda seed: [t.cuda() for t in make_config_inputs(2, 130, 64, 64, torch.bfloat16, seed=seed)]
    h = lambda ts: [t.unsqueeze(2) for t in ts[:5]] + [ts[5].unsqueeze(1), ts[6].unsqueeze(2), ts[7].unsqueeze(1)]
    static = h(make(1))

    def step(ins):
        args = [t.requires_grad_() for t in ins[:6]]
        res = LFWHeadsFunction.apply(*args, True)
        return [*res, *torch.autograd.grad(res, args, ins[6:])]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step([t.detach() for t in static])
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = step([t.detach() for t in static])
    for seed in (2, 3, 4):
        new = h(make(seed))
        for a, b in zip(static, new):
            a.detach().copy_(b)
        graph.replay()
        eager = step([t.detach() for t in new])
        torch.cuda.synchronize()
        for a, b in zip(res, eager):
            assert torch.equal(a, b)
