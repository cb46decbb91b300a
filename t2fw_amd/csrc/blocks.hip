// Cuts tensors whose widths are multiples of 64 into 64-wide blocks and puts results together again: up to eight arrays
// in one launch, each a strided gather of 64-element vectors, optionally summed over the blocks that share a channel
// (fp32 sums, one rounding).  Pure streaming: a lane moves 16 bytes (one element where an address is not 16-byte
// aligned), so a vector is 8 lanes of a 16-bit type or 16 of fp32, and consecutive lanes write consecutive addresses.
//
// B=24, T=1024, 128 x 128 fp16, forward + backward: four launches, 61 us (3.7 TB/s), in the place of sixteen tensor
// operations, 144 us.
//
// The reference has one kernel for every width (t2fw/csrc/lfw_kernel.cu:105-121) and no counterpart of this.
#include "common.hpp"
#include "blocks.hpp"

namespace t2fw {
namespace {

constexpr int BC_THREADS = 256;

template <typename IO, int N> struct __attribute__((aligned(sizeof(IO) * N))) Piece {
    IO v[N];
};

template <typename IO, int N> __global__ __launch_bounds__(BC_THREADS) void block_copy_kernel(BlockCopyArgs p) {
    using P = Piece<IO, N>;
    constexpr int PER = 64 / N;                  // pieces of a vector
    const int64_t total = p.first[p.count] * PER;
    for (int64_t idx = (int64_t)blockIdx.x * BC_THREADS + threadIdx.x; idx < total; idx += (int64_t)gridDim.x * BC_THREADS) {
        const int64_t vec = idx / PER;
        const int part = (int)(idx % PER) * N;
        int i = 0;
        while (vec >= p.first[i + 1]) ++i;       // count <= 8; vec < first[count]
        const t2fw_block_copy_desc &d = p.a[i];
        const int64_t v = vec - p.first[i];
        uint32_t rest = (uint32_t)v;             // fewer than 2^31 vectors (checked by the host)
        int64_t off = part;
#pragma unroll
        for (int m = 3; m > 0; --m) {
            const uint32_t n = (uint32_t)d.size[m], q = rest / n;
            off += (int64_t)(rest - q * n) * d.stride[m];
            rest = q;
        }
        off += rest * d.stride[0];
        const IO *src = static_cast<const IO *>(d.src) + off;
        P r = *reinterpret_cast<const P *>(src);
        if (d.terms > 1) {
            float s[N];
#pragma unroll
            for (int e = 0; e < N; ++e) s[e] = to_acc(r.v[e]);
            for (int64_t t = 1; t < d.terms; ++t) {
                src += d.term_stride;
                const P w = *reinterpret_cast<const P *>(src);
#pragma unroll
                for (int e = 0; e < N; ++e) s[e] += to_acc(w.v[e]);
            }
#pragma unroll
            for (int e = 0; e < N; ++e) r.v[e] = from_acc<IO>(s[e]);
        }
        *reinterpret_cast<P *>(static_cast<IO *>(d.dst) + v * 64 + part) = r;
    }
}

template <typename IO> int launch(const BlockCopyArgs &a, bool aligned, hipStream_t stream) {
    constexpr int N = 16 / sizeof(IO);
    const int64_t pieces = a.first[a.count] * (aligned ? 64 / N : 64);
    if (pieces == 0) return T2FW_OK;
    const int64_t blocks = (pieces + BC_THREADS - 1) / BC_THREADS;
    const dim3 grid((unsigned)(blocks < 65536 ? blocks : 65536));
    if (aligned)
        hipLaunchKernelGGL((block_copy_kernel<IO, N>), grid, dim3(BC_THREADS), 0, stream, a);
    else
        hipLaunchKernelGGL((block_copy_kernel<IO, 1>), grid, dim3(BC_THREADS), 0, stream, a);
    return check_hip(hipGetLastError(), "block_copy_kernel launch");
}

}  // namespace

// The sizes are positive or the array is empty (checked by the caller); strides are element counts, multiples of 64.
int block_copy(BlockCopyArgs &a, int dtype, hipStream_t stream) {
    bool aligned = true;
    a.first[0] = 0;
    for (int i = 0; i < a.count; ++i) {
        const t2fw_block_copy_desc &d = a.a[i];
        a.first[i + 1] = a.first[i] + d.size[0] * d.size[1] * d.size[2] * d.size[3];
        if (a.first[i + 1] > 0x7fffffffLL) return fail(T2FW_ERR_UNSUPPORTED, "t2fw_block_copy: more than 2^31 vectors");
        aligned = aligned && reinterpret_cast<uintptr_t>(d.src) % 16 == 0 && reinterpret_cast<uintptr_t>(d.dst) % 16 == 0;
    }
    switch (dtype) {
        case T2FW_F32: return launch<float>(a, aligned, stream);
        case T2FW_F16: return launch<__half>(a, aligned, stream);
        case T2FW_BF16: return launch<__hip_bfloat16>(a, aligned, stream);
    }
    return fail(T2FW_ERR_BAD_DTYPE, "t2fw_block_copy takes fp32, fp16 or bf16 arrays");
}

}  // namespace t2fw
