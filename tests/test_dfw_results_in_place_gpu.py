"""The delta rule's backward with d_q and d_k in the place of q and k: the value side would leave the edges of the key side's chunks
there while q and k are still read, so the key side runs as one sequential pass."""
import pytest
import torch

from oracle.dfw_ref import dfw_reference_grads
from tests.test_dfw_chunk_gpu import run_abi
from tests.test_dfw_gpu import NAMES, TOL_DFW, make_inputs
from tests.test_lfw_gpu import assert_close

pytestmark = pytest.mark.gpu
SINGLE = 16                    # T2FW_FLAG_BF16_OPERANDS
MODES = [(torch.float32, 0), (torch.float32, SINGLE), (torch.float16, 0), (torch.float16, SINGLE), (torch.bfloat16, 0), (torch.bfloat16, SINGLE)]


@pytest.mark.parametrize("dtype,flags", MODES)
@pytest.mark.parametrize("T", [1, 64, 97, 200])
@pytest.mark.parametrize("blocks_entry", [False, True])
def test_gradients_in_the_place_of_queries_and_keys(dtype, flags, T, blocks_entry):
    from t2fw_amd import _lib
    lib, P, code, B = _lib.load(), _lib.ptr, _lib.DTYPE_CODE[dtype], 9
    ts = make_inputs(B, T, 64, 64, dtype, seed=T)
    _, _, refs = dfw_reference_grads(*ts)
    q, k, v, s, go, gs = [t.cuda() for t in ts]
    out, fin, delta, apart = run_abi(q, k, v, s, go, gs, flags)
    d_v, d_s = torch.empty_like(v), torch.empty_like(s)
    entry = lib.t2fw_dfw_backward_blocks if blocks_entry else lib.t2fw_dfw_backward
    _lib.check(entry(P(go), P(gs), P(q), P(k), P(delta), P(fin), P(q), P(k), P(d_v), P(d_s), B, T, 64, 64, code, flags,
                     _lib.current_stream_handle(v.device)))
    torch.cuda.synchronize()
    tol = TOL_DFW[dtype] if not flags else (1e-2, 1e-2)
    for name, g, r in zip(NAMES, (q, k, d_v, d_s), refs):
        assert_close(g, r, dtype, name, tol=tol)
    assert torch.equal(d_v, apart[2]) and torch.equal(d_s, apart[3])
