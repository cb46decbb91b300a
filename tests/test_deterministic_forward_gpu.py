"""torch.use_deterministic_algorithms: the forward of a row gives the same bits with and without gradients and whatever the rows beside it
(by default few rows of many steps run with their chunks side by side where that is faster)."""
import pytest
import torch

from tests.test_lfw_par_fwd_gpu import inputs

pytestmark = pytest.mark.gpu


@pytest.fixture
def deterministic():
    torch.use_deterministic_algorithms(True)
    yield
    torch.use_deterministic_algorithms(False)


@pytest.mark.parametrize("width", [64, 128])
def test_a_rows_bits_do_not_depend_on_the_call(width, deterministic):
    from t2fw_amd import LFWFunction
    ins = inputs(64, 1000, torch.float16, seed=5)
    if width == 128:
        ins = [torch.cat([t, t.flip(-1)], -1) for t in ins[:5]] + [ins[5].repeat(1, 2, 2)]
    few = [t[:4].clone() for t in ins]
    with torch.no_grad():
        res = [LFWFunction.apply(*few), LFWFunction.apply(*ins)]
    res.append(LFWFunction.apply(*[t.requires_grad_() for t in few]))
    for other in res[1:]:
        for a, b in zip(res[0], other):
            assert torch.equal(a, b[:4])


def test_activation_checkpointing(deterministic):
    """the recomputation is the first pass to the bit: what the layer after it keeps is what the backward sees"""
    from torch.utils.checkpoint import checkpoint
    from t2fw_amd import LFWFunction
    ins = [t.requires_grad_() for t in inputs(4, 1000, torch.float16, seed=6)]
    seen = []

    def layer(*a):
        out, _ = LFWFunction.apply(*[t * 1 for t in a])          # as a layer makes them: without gradients in the first pass
        seen.append(out.detach().clone())
        return out
    checkpoint(layer, *ins, use_reentrant=True).float().square().sum().backward()
    assert len(seen) == 2 and torch.equal(*seen)
