"""Error of the forward with the chunks of a row side by side (csrc/lfw_par_fwd.hip) against float64: no larger than that of the
sequential kernel, over gates from near one down to the limit of what the form takes on both sides at once (2^-80 over half a chunk is a
constant gate of 0.177), states of 1 down to 1e-5, with and without values that add to them."""
import pytest
import torch

from tests.test_lfw_par_fwd_gpu import exact, inputs, rel, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("state", [1.0, 1e-3, 1e-5])
@pytest.mark.parametrize("gate", [0.9, 0.4, 0.25, 0.185])
def test_entering_states_under_small_gates(gate, state, dtype):
    """no values: the outputs are what is left of the entering state, a few tokens' worth; 4 % is what 4 x 4 x 64 numbers scatter"""
    g = torch.Generator(device="cuda").manual_seed(3)
    n = lambda *s: torch.randn(s, generator=g, device="cuda")
    u = lambda: (torch.rand((4, 1024, 64), generator=g, device="cuda") * 0.001 + gate).to(dtype)
    ins = [torch.zeros((4, 1024, 64), dtype=dtype, device="cuda"), u(), n(4, 1024, 64).to(dtype), n(4, 1024, 64).to(dtype), u(),
           (n(4, 64, 64) * state).to(dtype)]
    out, nxt, _, flags, _, extra = run(0, ins, ckpt=False)
    assert extra > 0 and not flags.any()
    s_out = run(8, ins, ckpt=False)[0]
    want = exact(ins)[0]
    assert rel(out, want) <= 1.04 * rel(s_out, want), (rel(out, want), rel(s_out, want))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,T,mean", [(4, 1024, 2.0), (12, 1000, 3.0), (32, 2050, 2.0), (9, 1087, 0.0), (9, 1087, 4.0)])
def test_gates_of_a_model(B, T, mean, dtype):
    ins = inputs(B, T, dtype, seed=T + B, mean=mean)
    out, nxt, _, _, _, extra = run(0, ins, ckpt=False)
    assert extra > 0
    s_out, s_nxt, *_ = run(8, ins, ckpt=False)
    for a, b, want in zip((out, nxt), (s_out, s_nxt), exact(ins)):
        assert rel(a, want) <= rel(b, want), (rel(a, want), rel(b, want))
