"""t2fw_lfw_forward with next_state in the place of s0 and t2fw_lfw_backward with d_s0 in that of g_state, on the exact
chunk-parallel kernels: small calls, whose workgroups would each read the whole starting state while others write there, leave the chain
over a row's chunks to a launch of its own.  Which of the two ran shows in the workspace: the launch puts the state (adjoint)
that enters a chunk in the place of the chunk's increment."""
import pytest
import torch

from t2fw_amd.synthetic import make_config_inputs

pytestmark = pytest.mark.gpu

CHUNKS = 32          # T2FW_FLAG_EXACT_CHUNKS


def call(D, K, T, dtype, aliased):
    """results of a forward and a backward call, and whether each had a launch for the chain"""
    from t2fw_amd import _lib
    lib = _lib.load()
    *ins, go, gs = [t.cuda() for t in make_config_inputs(5, T, D, K, dtype, seed=T, in_scale=0.5, state_std=0.5)]
    ins[1][1, T // 2, 0] = 1.25              # a row left to the recurrence over the whole sequence
    ins[5][0, 0, 0] = 2.0                    # not a chunk's increment
    gs[0, 0, 0] = 2.0
    code, P, nc, up = _lib.DTYPE_CODE[dtype], _lib.ptr, -(-T // 64), lambda n: -(-n // 16) * 16
    size = lib.t2fw_lfw_workspace_bytes(5, T, D, K, 64, code, CHUNKS)
    ws, st = torch.zeros(size, dtype=torch.uint8, device="cuda"), _lib.current_stream_handle(go.device)
    states = ws.view(torch.float32)[:5 * nc * up(D) * up(K)].view(5, nc, up(D), up(K))
    out, ckpt = torch.empty_like(ins[0]), torch.empty((5, nc, D, K), dtype=dtype, device="cuda")
    s0 = ins[5].clone()
    nxt = s0 if aliased else torch.empty_like(s0)
    _lib.check(lib.t2fw_lfw_forward(*[P(t) for t in ins[:5]], P(s0), P(out), P(nxt), P(ckpt), 5, T, D, K, 64, code, CHUNKS, P(ws), size, st))
    torch.cuda.synchronize()
    chained = [states[0, 0, 0, 0].item() == 2.0]
    grads = [torch.empty_like(t) for t in ins]
    g = gs.clone()
    if aliased:
        grads[5] = g
    _lib.check(lib.t2fw_lfw_backward(P(go), P(g), *[P(t) for t in ins], P(ckpt), *[P(t) for t in grads], 5, T, D, K, 64, code, CHUNKS, P(ws), size, st))
    torch.cuda.synchronize()
    chained.append(states[0, nc - 1, 0, 0].item() == 2.0)
    return [out, nxt, ckpt, *grads], chained


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("D,K,T", [(9, 5, 230), (16, 16, 9 * 64 - 1), (33, 17, 385), (5, 63, 449)])
def test_results_in_the_place_of_the_starting_state(D, K, T, dtype):
    want, chained = call(D, K, T, dtype, False)
    assert chained == [False, False]
    got, chained = call(D, K, T, dtype, True)
    assert chained == [True, True]
    for a, b in zip(got, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("D,K,T,chain", [(33, 17, 385, (False, False)), (33, 17, 8 * 64, (False, False)), (33, 17, 8 * 64 + 1, (True, True)),
                                         (63, 32, 300, (True, True)), (16, 16, 40 * 64, (False, False)), (16, 16, 48 * 64, (False, True)),
                                         (16, 16, 48 * 64 + 1, (True, True))])
def test_where_the_chain_has_a_launch(D, K, T, chain):
    """up to six batches of eight chunks per thread, and 5 x 2^20 floats read in all (five rows of 48 chunks: the backward's two
    sides read more)"""
    assert call(D, K, T, torch.float32, False)[1] == list(chain)
