"""The forward with the chunks of a row side by side (csrc/lfw_par_fwd.hip) keeps two verdicts per row at the end of its scratch: by the
gates and states, which its last launch reads and does not write, and by the outputs, which it writes and does not read."""
import pytest
import torch

from tests.test_lfw_par_fwd_gpu import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B", [6, 40, 56])
def test_a_launch_does_not_write_the_verdict_that_it_reads(B, dtype):
    from t2fw_amd import _lib
    lib = _lib.load()
    T = 1000 if B < 40 else 64 * 100
    x, f, q, k, fk, s = ins = inputs(B, T, dtype, seed=6)
    q[1, T - 1, 63] = float("inf")           # outputs only
    f[2, 700, 3] = 1.5                       # gates
    x[B - 1, 500, 1] = float("nan")          # states, and outputs of the chunk that it is in
    code = _lib.DTYPE_CODE[dtype]
    n = lib.t2fw_lfw_forward_workspace_bytes(B, T, 64, 64, 64, code, 0)
    extra = lib.t2fw_lfw_forward_scratch_bytes(B, T, 1, 64, 64, 64, code, 0, 0)
    assert extra > 0
    ws = torch.full((n,), 255, dtype=torch.uint8, device="cuda")
    scratch = torch.full((extra + 4096,), 255, dtype=torch.uint8, device="cuda")
    out, nxt = torch.empty_like(x), torch.empty_like(s)
    P = _lib.ptr
    _lib.check(lib.t2fw_lfw_forward_scratch(*[P(t) for t in ins], P(out), P(nxt), None, B, T, 1, 64, 64, 64, code, 0, P(ws), n, P(scratch),
                                            extra, _lib.current_stream_handle(x.device)))
    torch.cuda.synchronize()
    assert (scratch[extra:] == 255).all()
    size = -(-8 * B // 256) * 256
    gates, outputs = scratch[extra - size:extra].view(torch.int32)[:2 * B].view(2, B).cpu()
    assert gates.nonzero().flatten().tolist() == [2, B - 1]
    assert outputs.nonzero().flatten().tolist() == [1]
    want = torch.empty_like(x), torch.empty_like(s)
    _lib.check(lib.t2fw_lfw_forward(*[P(t) for t in ins], P(want[0]), P(want[1]), None, B, T, 64, 64, 64, code, 0, P(ws), n,
                                    _lib.current_stream_handle(x.device)))
    for a, b in zip((out, nxt), want):
        for r in (1, 2, B - 1):
            assert torch.equal(a[r].isnan(), b[r].isnan()) and torch.equal(a[r].nan_to_num(), b[r].nan_to_num())
