"""The forward with the chunks of a row side by side takes up to 420 MB of scratch: where the allocator has no room for it the call runs on
the sequential kernel, which needs none."""
import pytest
import torch

from tests.test_lfw_par_fwd_gpu import inputs, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grad", [False, True])
def test_without_room_for_the_scratch(grad):
    from t2fw_amd import LFWFunction
    ins = inputs(32, 32768, torch.float16, seed=3)                 # 16384 chunks; 134 MB a tensor, as much again for checkpoints
    out, nxt, *_, none = run(8, ins, ckpt=False)
    assert none == 0
    ins = [t.requires_grad_(grad) for t in ins]
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.empty_cache()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (360 << 20)) / total)
    try:
        got = LFWFunction.apply(*ins)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    for a, b in zip(got, (out, nxt)):
        assert torch.equal(a, b)
