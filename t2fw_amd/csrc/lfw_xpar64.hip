// Launch 3 of the chunk-parallel exact recurrence (lfw_xpar.hip) for fp32 tensors with 64 x 64 states.
//
// Chunks whose gates allow it run as products on fp64 matrix instructions (lfw_xpar64_mm.hpp), one workgroup of four
// waves per (row, chunk) [backward: and side].  Everything else runs in one more launch (4 and 6 us where it finds nothing
// to do; one kernel for both was 3 % faster then, and 8 % slower than the steps alone where every chunk has a zero gate): chunks
// with a gate below 2^-20 or a gate product below 2^-400, and those whose gate gradients have cancelled in the products, step by
// step, a state in a workgroup's registers, and rows that are left to the recurrence over the whole sequence on the per-step bodies.
//
// B = 96, T = 1024, measured: forward 53 us, backward 154 us, against 70 and 439 us for the same chunks step by step.
// Relative error against float64 (2-norm) 4.0e-8 outputs, 4.6e-8 gate gradients, 2.5e-8 states; step by step 8.5e-8, 1.03e-7
// and 5.1e-8.  What bounds the backward: the matrix instructions of a wave, 120 in fp64 (27 ns each) and 128 in fp32 (13.5),
// are 60 us at 12 waves per SIMD, its fp64 vector instructions, which do not run beside fp64 matrix instructions, about 35,
// and its 337 MB take 62 us at a large copy's rate; with two workgroups per CU these overlap in part.  Forms that were slower:
// products with the states in fp64, too (backward 163, forward 56, state error 2.5e-8); tiles of 16 steps with the state
// carried over them (operands in fp32: 199 us, twice the vector instructions); consecutive workgroups on chunks of one row in
// the place of one chunk of all rows (181 us).
//
// The steps: a lane is a row of the state (value channels; key channels on the backward's key side), a wave holds 16 of the
// other side's channels ("columns") in registers; lane l also holds the inputs of column l % 16, which DPP broadcasts within
// each row of 16 lanes as an operand of the multiplications: neither LDS nor scalar registers carry the inputs.  A
// contraction over columns, S_t q_t and the like, is lane-local; the four waves' shares meet in LDS, eight steps at a time.
// A state element costs 4 VALU instructions per step forward and 12.75 / 13.75 backward (value / key side: 3.75 + 3 to
// rebuild the states, the rest for the adjoint and the sums), the per-step kernels' arithmetic without their cross-lane
// sums.  Backward, per chunk: the states at steps 16, 32 and 48 (LDS) are rebuilt from the checkpoint, blocks of 16 steps
// are visited last to first, and per half block the eight states are rebuilt into registers and the adjoint runs back over
// them.  Tried and slower: rank-one terms on v_mfma_f32_4x4x1 (forward 115 us, backward 603), column vectors in scalar
// registers (105 and 1145: every wave misses the scalar cache once per step and array).
//
// A row that is left runs a tile of 16 channels per workgroup: 226 and 780 us where all of 96 rows x 1024 steps are
// (per-step kernels 228 and 822; one workgroup walking such a row in the layout of the steps: 335 and 1174).
#include "lfw_chunk.hpp"
#include "lfw_scan_body.hpp"
#include "lfw_xpar.hpp"
#include "lfw_xpar64_mm.hpp"

namespace t2fw {
namespace {

constexpr int XW_THREADS = 256;
constexpr int XW_COLS = 16;            // columns per wave
constexpr int XW_SEG = 8;              // steps whose inputs, states and sums are in flight together

// XW_SEG steps of one array, one value per lane.  p: the array at the segment's first step (wave-uniform), c: the lane's
// channel; steps from n on are read from the last one (and replaced by pad_steps).
__device__ __forceinline__ void load_steps(float (&r)[XW_SEG], const float *p, int c, int64_t ts, int n) {
#pragma unroll
    for (int j = 0; j < XW_SEG; ++j) r[j] = (p + min(j, n - 1) * ts)[(unsigned)c];
}
__device__ __forceinline__ void pad_steps(float (&r)[XW_SEG], int n, float pad) {
#pragma unroll
    for (int j = 0; j < XW_SEG; ++j) r[j] = j < n ? r[j] : pad;
}

// lane N of each row of 16, in every lane of the row
template <int N> __device__ __forceinline__ float bcast(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xf, 0xf, true));
}
// The compiler folds a broadcast into a multiplication but not into a multiply-add: those are written out.  Both blocks
// start with the two wait states that a DPP read of a register just written by the VALU needs.
//
// sum over the wave's columns of S times the column vector (chains of four, as the per-step kernel's lanes)
__device__ __forceinline__ float dot(const floatx4 (&S)[4], float col) {
    float a0, a1, a2, a3;
    asm("s_nop 1\n"
        "v_mul_f32_dpp %0, %4, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %1, %4, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %2, %4, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %3, %4, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %0, %4, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %1, %4, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %2, %4, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %3, %4, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %0, %4, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %1, %4, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %2, %4, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %3, %4, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %0, %4, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %1, %4, %18 row_newbcast:13 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %2, %4, %19 row_newbcast:14 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %3, %4, %20 row_newbcast:15 row_mask:0xf bank_mask:0xf\n"
        : "=&v"(a0), "=&v"(a1), "=&v"(a2), "=&v"(a3)
        : "v"(col), "v"(S[0][0]), "v"(S[0][1]), "v"(S[0][2]), "v"(S[0][3]), "v"(S[1][0]), "v"(S[1][1]), "v"(S[1][2]), "v"(S[1][3]), "v"(S[2][0]), "v"(S[2][1]), "v"(S[2][2]), "v"(S[2][3]), "v"(S[3][0]), "v"(S[3][1]), "v"(S[3][2]), "v"(S[3][3]));
    return (a0 + a1) + (a2 + a3);
}
// G += (column vector) (x) (row vector)
__device__ __forceinline__ void add_outer(floatx4 (&G)[4], float col, float row) {
    float g[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) g[n] = G[n / 4][n % 4];
    asm("s_nop 1\n"
        "v_fmac_f32_dpp %0, %16, %17 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %1, %16, %17 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %2, %16, %17 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %3, %16, %17 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %4, %16, %17 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %5, %16, %17 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %6, %16, %17 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %7, %16, %17 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %8, %16, %17 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %9, %16, %17 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %10, %16, %17 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %11, %16, %17 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %12, %16, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %13, %16, %17 row_newbcast:13 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %14, %16, %17 row_newbcast:14 row_mask:0xf bank_mask:0xf\n"
        "v_fmac_f32_dpp %15, %16, %17 row_newbcast:15 row_mask:0xf bank_mask:0xf\n"
        : "+v"(g[0]), "+v"(g[1]), "+v"(g[2]), "+v"(g[3]), "+v"(g[4]), "+v"(g[5]), "+v"(g[6]), "+v"(g[7]), "+v"(g[8]), "+v"(g[9]), "+v"(g[10]), "+v"(g[11]), "+v"(g[12]), "+v"(g[13]), "+v"(g[14]), "+v"(g[15])
        : "v"(col), "v"(row));
#pragma unroll
    for (int n = 0; n < 16; ++n) G[n / 4][n % 4] = g[n];
}

// What follows (volatile) does not start before v is there: keeps the steps apart, whose products would not fit the
// registers all at once.
__device__ __forceinline__ void settle(floatx4 (&v)[4]) {
    asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
}
__device__ __forceinline__ void settle(float &a, float &b, float &c, float &d) {
    asm volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}

// S <- S * (f (x) f_key) + x (x) k
template <int Q> __device__ __forceinline__ void step4(floatx4 &out, const floatx4 &S, float ca, float cf, float ra, float rf) {
    out[0] = fmaf(S[0], bcast<4 * Q + 0>(cf) * rf, bcast<4 * Q + 0>(ca) * ra);
    out[1] = fmaf(S[1], bcast<4 * Q + 1>(cf) * rf, bcast<4 * Q + 1>(ca) * ra);
    out[2] = fmaf(S[2], bcast<4 * Q + 2>(cf) * rf, bcast<4 * Q + 2>(ca) * ra);
    out[3] = fmaf(S[3], bcast<4 * Q + 3>(cf) * rf, bcast<4 * Q + 3>(ca) * ra);
}
__device__ __forceinline__ void step(floatx4 (&out)[4], const floatx4 (&S)[4], float ca, float cf, float ra, float rf) {
    step4<0>(out[0], S[0], ca, cf, ra, rf);
    step4<1>(out[1], S[1], ca, cf, ra, rf);
    step4<2>(out[2], S[2], ca, cf, ra, rf);
    step4<3>(out[3], S[3], ca, cf, ra, rf);
}
// G *= (column vector) (x) (row vector)
__device__ __forceinline__ void scale_outer(floatx4 (&G)[4], float col, float row) {
    float g[16];
    asm("s_nop 1\n"
        "v_mul_f32_dpp %0, %16, %17 row_newbcast:0 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %1, %16, %17 row_newbcast:1 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %2, %16, %17 row_newbcast:2 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %3, %16, %17 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %4, %16, %17 row_newbcast:4 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %5, %16, %17 row_newbcast:5 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %6, %16, %17 row_newbcast:6 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %7, %16, %17 row_newbcast:7 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %8, %16, %17 row_newbcast:8 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %9, %16, %17 row_newbcast:9 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %10, %16, %17 row_newbcast:10 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %11, %16, %17 row_newbcast:11 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %12, %16, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %13, %16, %17 row_newbcast:13 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %14, %16, %17 row_newbcast:14 row_mask:0xf bank_mask:0xf\n"
        "v_mul_f32_dpp %15, %16, %17 row_newbcast:15 row_mask:0xf bank_mask:0xf\n"
        : "=&v"(g[0]), "=&v"(g[1]), "=&v"(g[2]), "=&v"(g[3]), "=&v"(g[4]), "=&v"(g[5]), "=&v"(g[6]), "=&v"(g[7]), "=&v"(g[8]), "=&v"(g[9]), "=&v"(g[10]), "=&v"(g[11]), "=&v"(g[12]), "=&v"(g[13]), "=&v"(g[14]), "=&v"(g[15])
        : "v"(col), "v"(row));
#pragma unroll
    for (int n = 0; n < 16; ++n) G[n / 4][n % 4] *= g[n];
}

// 16 consecutive columns of row `row` of a [64][64] state, or 16 rows of column `row` (TRANSPOSED); p, col0 wave-uniform,
// p aligned to its elements
struct __attribute__((packed, aligned(4))) Float4 {
    float v[4];
};
template <bool TRANSPOSED> __device__ __forceinline__ void load_state(floatx4 (&S)[4], const float *p, int row, int col0) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (TRANSPOSED) {
#pragma unroll
            for (int e = 0; e < 4; ++e) S[q][e] = (p + (col0 + 4 * q + e) * XP_N)[(unsigned)row];
        } else {
            const Float4 v = *reinterpret_cast<const Float4 *>((p + col0 + 4 * q) + (unsigned)(row * XP_N));
#pragma unroll
            for (int e = 0; e < 4; ++e) S[q][e] = v.v[e];
        }
    }
}
__device__ __forceinline__ void store_state(float *p, const floatx4 (&S)[4], int row, int col0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<Float4 *>((p + col0 + 4 * q) + (unsigned)(row * XP_N)) = Float4{{S[q][0], S[q][1], S[q][2], S[q][3]}};
}

// ---- rows that are left ---------------------------------------------------------------------------
constexpr int XW_LEFT_TB = 16;
constexpr int XW_TILES = XP_N / 16;
__device__ __forceinline__ void left_row_forward(const XparFwdArgs &p, int64_t b, int chunk) {
    ScanFwdArgs s{};
    s.x = p.x; s.f = p.f; s.q = p.q; s.k = p.k; s.f_key = p.f_key; s.s0 = p.s0;
    s.out = p.out; s.next_state = p.next_state; s.ckpt = p.ckpt;
    s.B = p.B; s.T = p.T; s.D = XP_N; s.K = XP_N; s.NC = p.NC;
    s.C = XP_CHUNK; s.kg = 16; s.tb = XW_LEFT_TB; s.ntiles = XW_TILES; s.heads = p.heads;
    for (int tile = chunk; tile < XW_TILES; tile += (int)p.NC)
        scan::fwd_scan_body_kg<float, 4, 16, XW_LEFT_TB>(s, b, tile);
}
template <int SIDE> __device__ __forceinline__ void left_row_backward(const XparBwdArgs &p, int64_t b, int chunk) {
    ScanBwdArgs s{};
    s.g_out = p.g_out; s.g_state = p.g_state; s.x = p.x; s.f = p.f; s.q = p.q; s.k = p.k; s.f_key = p.f_key; s.ckpt = p.ckpt;
    s.d_x = p.d_x; s.d_f = p.d_f; s.d_q = p.d_q; s.d_k = p.d_k; s.d_f_key = p.d_f_key; s.d_s0 = p.d_s0;
    s.B = p.B; s.T = p.T; s.D = XP_N; s.K = XP_N; s.NC = p.NC;
    s.C = XP_CHUNK; s.kg = 16; s.use_sub = 1; s.ntiles = XW_TILES; s.heads = p.heads;
    for (int tile = chunk; tile < XW_TILES; tile += (int)p.NC)
        scan::bwd_scan_body_kg<float, 4, SIDE, 16, 1>(s, b, tile);
}

// ---- forward --------------------------------------------------------------------------------------
struct FwdSmem {
    float part[2][XW_SEG][4][XP_N];
};
__device__ __forceinline__ void forward_steps(const XparFwdArgs &p, FwdSmem &sm, int64_t b, int chunk) {
    auto &part = sm.part;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, col0 = XW_COLS * w;
    const int T = (int)p.T;
    int t_end = min(T, (chunk + 1) * XP_CHUNK);
    // the compiler must not see that the loop below runs eight times at most: it would keep the addresses of its passes
    // and need 134 registers, which leaves three waves per SIMD in the place of four
    asm("" : "+s"(t_end));
    const int64_t ts = (int64_t)p.heads * XP_N, line0 = uniform64(row_first_token(b, p.T, p.heads)) * XP_N;
    const float *const x = (const float *)p.x + line0, *const f = (const float *)p.f + line0;
    const float *const k = (const float *)p.k + line0 + col0, *const fk = (const float *)p.f_key + line0 + col0;
    const int cl = lane & 15;
    const float *const q = (const float *)p.q + line0 + col0;
    float *const out = (float *)p.out + line0;
    floatx4 S[4];
    load_state<false>(S, mm::entering_state(p, b * p.NC + chunk), lane, col0);
    int buf = 0;
    float rx[XW_SEG], rf[XW_SEG], ck[XW_SEG], cf[XW_SEG], cq[XW_SEG];
    auto fetch = [&](int t0) {
        const int n = t_end - t0;
        load_steps(rx, x + t0 * ts, lane, ts, n);
        load_steps(rf, f + t0 * ts, lane, ts, n);
        load_steps(ck, k + t0 * ts, cl, ts, n);
        load_steps(cf, fk + t0 * ts, cl, ts, n);
        load_steps(cq, q + t0 * ts, cl, ts, n);
        if (n < XW_SEG) {
            pad_steps(rx, n, 0.f);
            pad_steps(rf, n, 1.f);
            pad_steps(ck, n, 0.f);
            pad_steps(cf, n, 1.f);
        }
    };
    int t0 = chunk * XP_CHUNK;
    fetch(t0);
    for (; t0 < t_end; t0 += XW_SEG, buf ^= 1) {
        const int n = min(XW_SEG, t_end - t0);
        float cx[XW_SEG], cff[XW_SEG], kx[XW_SEG], kf[XW_SEG], kq[XW_SEG];
#pragma unroll
        for (int j = 0; j < XW_SEG; ++j) {
            cx[j] = rx[j]; cff[j] = rf[j]; kx[j] = ck[j]; kf[j] = cf[j]; kq[j] = cq[j];
        }
        if (t0 + XW_SEG < t_end) fetch(t0 + XW_SEG);
#pragma unroll
        for (int j = 0; j < XW_SEG; ++j) {
            step(S, S, kx[j], kf[j], cx[j], cff[j]);
            part[buf][j][w][lane] = dot(S, kq[j]);
        }
        __syncthreads();                 // the shares of this segment are there; the other buffer is free again
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int j = w + 4 * u;
            const float(*const s)[XP_N] = part[buf][j];
            if (j < n) (out + (t0 + j) * ts)[(unsigned)lane] = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
        }
    }
    if (t_end == T) store_state((float *)p.next_state + b * (XP_N * XP_N), S, lane, col0);
}

// Both kernels of a direction number their workgroups chunk by chunk.  The first does the chunks that the matrix
// instructions take and says which those were; the second does the others and the rows that are left.
//
// What the first says of a (row, chunk, side), in the place of the chunk's gate products, which launch 2 was the last to read.
// All results of those not done are stored again by the second.
__device__ __forceinline__ int32_t *not_done(const XparScratch &ws, int64_t item, int side) {
    return reinterpret_cast<int32_t *>(ws.tots + item * (2 * XP_N)) + side;
}
__global__ __launch_bounds__(XW_THREADS, 2) void lfw_xpar64_fwd_mm_kernel(XparFwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int64_t b = blockIdx.x % p.B;
    const int chunk = (int)(blockIdx.x / p.B);
    const int64_t item = b * p.NC + chunk;
    if (row_left(p.ws, b) || p.ws.chunk_flags[item] != 0) return;
    mm::Smem &sm = *reinterpret_cast<mm::Smem *>(smem);
    const bool done = (chunk + 1) * XP_CHUNK <= (int)p.T ? mm::forward_chunk<true>(p, sm, b, chunk) : mm::forward_chunk<false>(p, sm, b, chunk);
    if (threadIdx.x == 0) *not_done(p.ws, item, 0) = done ? 0 : 1;
}
__global__ __launch_bounds__(XW_THREADS, 4) void lfw_xpar64_fwd_steps_kernel(XparFwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int64_t b = blockIdx.x % p.B;
    const int chunk = (int)(blockIdx.x / p.B);
    const int64_t item = b * p.NC + chunk;
    const int out_of_range = p.ws.chunk_flags[item], rejected = *not_done(p.ws, item, 0);      // requested together
    if (row_left(p.ws, b))
        left_row_forward(p, b, chunk);
    else if ((out_of_range | rejected) != 0)
        forward_steps(p, *reinterpret_cast<FwdSmem *>(smem), b, chunk);
}

// ---- backward -------------------------------------------------------------------------------------
constexpr int XW_BLOCK = 2 * XW_SEG;
struct BwdSmem {
    float part[3][XW_SEG][4][XP_N];
    float start[3][XW_COLS][XW_THREADS];      // states at steps 16, 32 and 48 of a chunk, lane-private
};
static_assert(2 * sizeof(BwdSmem) <= 160 * 1024, "two workgroups must fit the LDS of one CU");

template <int SIDE> __device__ __forceinline__ void backward_side(const XparBwdArgs &p, BwdSmem &sm, int64_t b, int chunk) {
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, col0 = XW_COLS * w;
    const int64_t ts = (int64_t)p.heads * XP_N, line0 = uniform64(row_first_token(b, p.T, p.heads)) * XP_N;
    const float *const ra = (const float *)(SIDE ? p.k : p.x) + line0, *const rf = (const float *)(SIDE ? p.f_key : p.f) + line0;
    const float *const ru = (const float *)(SIDE ? p.q : p.g_out) + line0;
    const float *const ca = (const float *)(SIDE ? p.x : p.k) + line0 + col0, *const cf = (const float *)(SIDE ? p.f : p.f_key) + line0 + col0;
    const float *const cu = (const float *)(SIDE ? p.g_out : p.q) + line0 + col0;
    float *const d_a = (float *)(SIDE ? p.d_k : p.d_x) + line0, *const d_f = (float *)(SIDE ? p.d_f_key : p.d_f) + line0;
    float *const d_u = (float *)p.d_q + line0;
    const int cl = lane & 15;
    floatx4 S[4], G[4];

    // A chunk is a list of jobs of up to eight steps: `ahead` that advance S to the start of the last block of 16 steps,
    // then per block, last to first, an advance over its first half and the two halves in reverse (a last block of
    // eight steps or fewer: one).  The gates and values of a job are requested while the job before it computes.
    struct Job {
        int t0, n, blk;
        bool reverse, restart;               // restart: S is the state at the start of block blk
    };
    int tc = 0, len = 0, nblk = 0, ahead = 0, last_jobs = 0;
    auto enter_chunk = [&](int c) {
        tc = c * XP_CHUNK;
        len = (int)min((int64_t)XP_CHUNK, p.T - tc);
        nblk = (len + XW_BLOCK - 1) / XW_BLOCK;
        ahead = 2 * (nblk - 1);
        last_jobs = len - XW_BLOCK * (nblk - 1) > XW_SEG ? 3 : 1;
    };
    auto jobs = [&]() { return ahead + last_jobs + 3 * (nblk - 1); };
    auto job = [&](int q) {
        if (q < ahead) return Job{tc + XW_SEG * q, XW_SEG, q >> 1, false, q == 0};
        const int r = q - ahead, o = r - last_jobs;
        const int blk = r < last_jobs ? nblk - 1 : nblk - 2 - o / 3;
        const int sub = r < last_jobs ? (last_jobs == 3 ? r : 2) : o % 3;
        const int t0 = XW_BLOCK * blk + (sub == 1 ? XW_SEG : 0);
        return Job{tc + t0, min(XW_SEG, len - t0), blk, sub != 0, sub != 1};
    };
    float va[XW_SEG], vf[XW_SEG], ka[XW_SEG], kf[XW_SEG];              // of the job that runs
    float nva[XW_SEG], nvf[XW_SEG], nka[XW_SEG], nkf[XW_SEG];          // of the next one
    int next_n = 0;
    auto fetch = [&](const Job &b) {
        load_steps(nva, ra + b.t0 * ts, lane, ts, b.n);
        load_steps(nvf, rf + b.t0 * ts, lane, ts, b.n);
        load_steps(nka, ca + b.t0 * ts, cl, ts, b.n);
        load_steps(nkf, cf + b.t0 * ts, cl, ts, b.n);
        next_n = b.n;
    };
    auto take = [&]() {
        if (next_n < XW_SEG) {
            pad_steps(nva, next_n, 0.f);
            pad_steps(nvf, next_n, 1.f);
            pad_steps(nka, next_n, 0.f);
            pad_steps(nkf, next_n, 1.f);
        }
#pragma unroll
        for (int j = 0; j < XW_SEG; ++j) {
            va[j] = nva[j]; vf[j] = nvf[j]; ka[j] = nka[j]; kf[j] = nkf[j];
        }
    };

    // S over the eight steps of a job
    auto advance = [&](const Job &next) {
        fetch(next);
#pragma unroll
        for (int j = 0; j < XW_SEG; ++j) {
            settle(ka[j], kf[j], va[j], vf[j]);
            step(S, S, ka[j], kf[j], va[j], vf[j]);
            settle(S);
        }
    };
    // The segment [t0, t0 + n): its states rebuilt from S, the adjoint back over them, the sums stored.
    auto reverse = [&](int t0, int n, const Job &next) {
        float vu[XW_SEG], ku[XW_SEG];
        floatx4 st[XW_SEG + 1][4];
#pragma unroll
        for (int q = 0; q < 4; ++q) st[0][q] = S[q];
#pragma unroll
        for (int j = 0; j < XW_SEG; ++j) {
            settle(ka[j], kf[j], va[j], vf[j]);
            step(st[j + 1], st[j], ka[j], kf[j], va[j], vf[j]);
            settle(st[j + 1]);
            if (j == XW_SEG / 2) {
                load_steps(vu, ru + t0 * ts, lane, ts, n);
                load_steps(ku, cu + t0 * ts, cl, ts, n);
            }
        }
        pad_steps(vu, n, 0.f);
        pad_steps(ku, n, 0.f);
        __syncthreads();                 // the sums of the segment before have been read
#pragma unroll
        for (int j = XW_SEG - 1; j >= 0; --j) {
            settle(ku[j], kf[j], vu[j], vf[j]);
            if (j == XW_SEG / 2) fetch(next);
            add_outer(G, ku[j], vu[j]);      // G_t = g_t (x) q_t + ...
            floatx4 w_[4];
            sm.part[0][j][w][lane] = dot(G, ka[j]);                                      // d_x / d_k
            if (SIDE == 1) sm.part[2][j][w][lane] = dot(st[j + 1], ku[j]);               // d_q
#pragma unroll
            for (int q = 0; q < 4; ++q) w_[q] = G[q] * st[j][q];
            sm.part[1][j][w][lane] = dot(w_, kf[j]);                                     // d_f / d_f_key
            scale_outer(G, kf[j], vf[j]);
            settle(G);
        }
        __syncthreads();
#pragma unroll
        for (int o = 0; o < (SIDE ? 3 : 2); ++o)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int j = w + 4 * h;
                const float(*const s)[XP_N] = sm.part[o][j];
                if (j < n) ((o == 0 ? d_a : o == 1 ? d_f : d_u) + (t0 + j) * ts)[(unsigned)lane] = (s[0][lane] + s[1][lane]) + (s[2][lane] + s[3][lane]);
            }
    };

    const int64_t state = (b * p.NC + chunk) * (XP_N * XP_N);
    load_state<SIDE == 1>(G, p.ws.states + state, lane, col0);
    const float *const s0 = (const float *)p.ckpt + state;
    enter_chunk(chunk);
    const int njobs = jobs();
    fetch(job(0));
    for (int q = 0; q < njobs; ++q) {
        const Job now = job(q), next = job(min(q + 1, njobs - 1));
        take();
        if (now.restart) {
            if (now.blk == 0) {
                load_state<SIDE == 1>(S, s0, lane, col0);
            } else {
#pragma unroll
                for (int u = 0; u < XW_COLS; ++u) S[u / 4][u % 4] = sm.start[now.blk - 1][u][tid];
            }
        }
        if (now.reverse) {
            reverse(now.t0, now.n, next);
        } else {
            advance(next);
            if (q < ahead && (q & 1)) {
#pragma unroll
                for (int u = 0; u < XW_COLS; ++u) sm.start[q >> 1][u][tid] = S[u / 4][u % 4];
            }
        }
    }
    if (SIDE == 0 && chunk == 0) store_state((float *)p.d_s0 + b * (XP_N * XP_N), G, lane, col0);
}

__global__ __launch_bounds__(XW_THREADS, 2) void lfw_xpar64_bwd_mm_kernel(XparBwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int64_t pair = blockIdx.x >> 1, b = pair % p.B;
    const int chunk = (int)(pair / p.B);
    const int64_t item = b * p.NC + chunk;
    if (row_left(p.ws, b) || p.ws.chunk_flags[item] != 0) return;
    mm::Smem &sm = *reinterpret_cast<mm::Smem *>(smem);
    const bool full = (chunk + 1) * XP_CHUNK <= (int)p.T;
    bool done;
    if ((blockIdx.x & 1) == 0)
        done = full ? mm::backward_chunk<0, true>(p, sm, b, chunk) : mm::backward_chunk<0, false>(p, sm, b, chunk);
    else
        done = full ? mm::backward_chunk<1, true>(p, sm, b, chunk) : mm::backward_chunk<1, false>(p, sm, b, chunk);
    if (threadIdx.x == 0) *not_done(p.ws, item, blockIdx.x & 1) = done ? 0 : 1;
}
__global__ __launch_bounds__(XW_THREADS, 2) void lfw_xpar64_bwd_steps_kernel(XparBwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int64_t pair = blockIdx.x >> 1, b = pair % p.B;
    const int chunk = (int)(pair / p.B);
    const int64_t item = b * p.NC + chunk;
    const int out_of_range = p.ws.chunk_flags[item], rejected = *not_done(p.ws, item, blockIdx.x & 1);      // requested together
    const bool left = row_left(p.ws, b);
    if (!left && (out_of_range | rejected) == 0) return;
    BwdSmem &sm = *reinterpret_cast<BwdSmem *>(smem);
    if (left) {
        if ((blockIdx.x & 1) == 0)
            left_row_backward<0>(p, b, chunk);
        else
            left_row_backward<1>(p, b, chunk);
    } else if ((blockIdx.x & 1) == 0) {
        backward_side<0>(p, sm, b, chunk);
    } else {
        backward_side<1>(p, sm, b, chunk);
    }
}

}  // namespace

int xpar64_forward(const XparFwdArgs &a, hipStream_t stream) {
    const int rc = enable_lds(reinterpret_cast<const void *>(lfw_xpar64_fwd_mm_kernel), (int)sizeof(mm::Smem), "hipFuncSetAttribute(lfw_xpar64_fwd_mm_kernel)");
    if (rc) return rc;
    const dim3 grid((unsigned)(a.B * a.NC));
    hipLaunchKernelGGL(lfw_xpar64_fwd_mm_kernel, grid, dim3(XW_THREADS), sizeof(mm::Smem), stream, a);
    const size_t left = scan_fwd_lds_bytes(XW_LEFT_TB, 16, 4, 16), smem = left > sizeof(FwdSmem) ? left : sizeof(FwdSmem);
    hipLaunchKernelGGL(lfw_xpar64_fwd_steps_kernel, grid, dim3(XW_THREADS), smem, stream, a);
    return check_hip(hipGetLastError(), "lfw_xpar64 forward launches");
}

int xpar64_backward(const XparBwdArgs &a, hipStream_t stream) {
    const size_t left = scan_bwd_lds_bytes(scan::SegLen<4>::value, 16, 4, 16, XP_CHUNK, true);
    const size_t smem = left > sizeof(BwdSmem) ? left : sizeof(BwdSmem);
    int rc = enable_lds(reinterpret_cast<const void *>(lfw_xpar64_bwd_mm_kernel), (int)sizeof(mm::Smem), "hipFuncSetAttribute(lfw_xpar64_bwd_mm_kernel)");
    if (!rc) rc = enable_lds(reinterpret_cast<const void *>(lfw_xpar64_bwd_steps_kernel), (int)smem, "hipFuncSetAttribute(lfw_xpar64_bwd_steps_kernel)");
    if (rc) return rc;
    const dim3 grid((unsigned)(2 * a.B * a.NC));
    hipLaunchKernelGGL(lfw_xpar64_bwd_mm_kernel, grid, dim3(XW_THREADS), sizeof(mm::Smem), stream, a);
    hipLaunchKernelGGL(lfw_xpar64_bwd_steps_kernel, grid, dim3(XW_THREADS), smem, stream, a);
    return check_hip(hipGetLastError(), "lfw_xpar64 backward launches");
}

}  // namespace t2fw
