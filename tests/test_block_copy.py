"""t2fw_block_copy against the same gather by torch (fp32 sums, one rounding): repeats, permutations, sums, empty arrays,
arrays that are not 16-byte aligned.  The sums are of at most three terms in the kernel's order, so results are equal."""
import pytest
import torch

ARRAYS = [
    ((3, 2, 5), (128 * 7, 0, 64)),                            # repeated
    ((3, 2, 5, 2), (64 * 21, 64, 64 * 4, 64 * 2)),            # permuted
    ((7, 2), (64 * 6, 64), 3, 64 * 2),                        # summed
    ((0, 4), (64, 64)),                                       # empty
    ((9,), (64,)),
]


def _check(dtype, device, shift):
    from t2fw_amd import _lib
    g = torch.Generator().manual_seed(1)
    srcs = [torch.randn(64 * 100 + shift, generator=g).to(dtype).to(device)[shift:] for _ in ARRAYS]
    dsts = [torch.full((*a[0], 64), 7.0, dtype=dtype, device=device) for a in ARRAYS]
    _lib.block_copy(_lib.block_plan(*ARRAYS), srcs, dsts)
    for (sizes, strides, *terms), s, d in zip(ARRAYS, srcs, dsts):
        n, ts = terms if terms else (1, 0)
        v = s.as_strided((*sizes, 64, n), (*strides, 1, ts)).float()
        want = v[..., 0].clone()
        for t in range(1, n):
            want += v[..., t]
        assert torch.equal(d, want.to(dtype))


def test_host_tensors():
    _check(torch.float32, "cpu", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shift", [0, 1])
def test_device_tensors(dtype, shift):
    _check(dtype, "cuda", shift)


def test_bad_arguments_are_refused():
    from t2fw_amd import _lib
    t = torch.zeros(128)
    for sizes, strides, *terms in (((-1,), (64,)), ((1,), (32,)), ((1,), (64,), 0, 0), ((1,), (64,), 2, 1)):
        descs = (_lib.BlockCopyDesc * 1).from_buffer_copy(_lib.block_plan((sizes, strides, *terms)))
        descs[0].src = descs[0].dst = t.data_ptr()
        with pytest.raises(RuntimeError):
            _lib.check(_lib.load().t2fw_block_copy(descs, 1, _lib.F32, None))
