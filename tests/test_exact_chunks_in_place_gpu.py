"""Exact chunk-parallel kernels of small calls, whose workgroups go through a row's chain themselves (chain_in_place of
csrc/lfw_xpar.hip): the bits of the chain's own launch, which the same rows take in a call of many more of them."""
import pytest
import torch

from t2fw_amd.synthetic import make_config_inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("D,K,T", [(1, 1, 65), (9, 5, 230), (16, 8, 8 * 64), (16, 16, 9 * 64 - 1), (33, 17, 385), (17, 40, 128), (5, 63, 7 * 64 + 1), (20, 40, 130),
                                   (16, 16, 48 * 64)])
def test_same_bits_as_with_the_chain_in_a_launch_of_its_own(D, K, T, dtype, monkeypatch):
    from t2fw_amd import LFWFunction
    monkeypatch.setenv("T2FW_FLAGS", "32")
    few = [t.cuda() for t in make_config_inputs(2, T, D, K, dtype, seed=T, in_scale=0.5, state_std=0.5)]
    few[1][1, T // 2, 0] = 1.25                     # a row left to the recurrence over the whole sequence
    up = lambda n: -(-n // 16) * 16
    chunks, state = -(-T // 64), up(D) * up(K)
    assert state // 256 * -(-chunks // 8) <= 6
    copies = (5 << 20) // (chunks * state) // (2 * chunks) + 1
    many = [t.repeat((copies,) + (1,) * (t.dim() - 1)) for t in few]
    res = []
    for *ins, go, gs in (few, many):
        args = [t.requires_grad_() for t in ins]
        out = LFWFunction.apply(*args)
        res.append([t[:2] for t in (*out, *torch.autograd.grad(out, args, (go, gs)))])
    for a, b in zip(*res):
        assert torch.equal(a, b)
