"""Block copies made with their results in one step (blocks_of of csrc/host.cpp): parameters and plain tensors take it, tensor
subclasses the general path; the same results.  Gates made in the same step as the forward: the same bits as sigmoid_gates before it."""
import pytest
import torch

from t2fw_amd.synthetic import make_config_inputs

pytestmark = pytest.mark.gpu


class _Marked(torch.Tensor):
    """a tensor subclass with torch's own behaviour"""


@pytest.mark.parametrize("D,K", [(128, 64), (64, 128), (128, 192)])
def test_block_copies_of_plain_tensors_parameters_and_subclasses(D, K):
    from t2fw_amd import LFWFunction
    *ins, go, gs = [t.cuda() for t in make_config_inputs(2, 37, D, K, torch.float16, seed=3)]
    want = None
    for make in (lambda t: t.clone(), torch.nn.Parameter, lambda t: t.clone().as_subclass(_Marked)):
        args = [make(t).requires_grad_() for t in ins]
        res = LFWFunction.apply(*args)
        got = [t.as_subclass(torch.Tensor) for t in (*res, *torch.autograd.grad(res, args, (go, gs)))]
        want = want or got
        for a, b in zip(got, want):
            assert a.shape == b.shape and torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width,heads", [(64, True), (64, False), (17, True), (128, True)])
def test_gates_in_the_step_of_the_forward(width, heads, dtype):
    from t2fw_amd import LFWFunction, LFWGatedFunction, LFWHeadsFunction, sigmoid_gates
    x, f, q, k, fk, s, _, _ = [t.cuda() for t in make_config_inputs(3, 70, width, width, dtype, seed=4)]
    lf, lk = torch.randn_like(f), torch.randn_like(fk)
    gates = sigmoid_gates(lf, lk)
    if heads:
        h = lambda t: t.unsqueeze(2)
        got = LFWHeadsFunction.apply(h(x), h(lf), h(q), h(k), h(lk), s.unsqueeze(1), True)
        want = LFWHeadsFunction.apply(h(x), h(gates[0]), h(q), h(k), h(gates[1]), s.unsqueeze(1))
    else:
        got, want = LFWGatedFunction.apply(x, lf, q, k, lk, s), LFWFunction.apply(x, gates[0], q, k, gates[1], s)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
