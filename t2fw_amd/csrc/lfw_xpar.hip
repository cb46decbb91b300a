// The exact per-step recurrence of the decay rule, chunk-parallel.
//
// The per-step kernels (lfw_scan.hip) carry a row's state through the whole sequence: their time is the number of steps
// times the latency of one step, on 1.5 workgroups per CU at 96 rows.  Here a row's chunks of 64 steps run side by side.
// Three launches per direction:
//   1  lfw_xpar_incr_kernel, a workgroup per (row, chunk): what the chunk adds to the state, sum_t (x_t A_t) (x) (k_t B_t)
//      with A_t, B_t the products of the gates after t to the chunk's end (backward: to the adjoint,
//      sum_t (g_t A_t) (x) (q_t B_t), products from the chunk's start up to t), and the chunk's gate products.  Plain
//      products, no inverses: as many roundings per term as the recurrence has.  The sum over the 64 steps runs on fp32
//      matrix instructions.
//   2  lfw_xpar_chain_kernel, elementwise: the chain over the chunks of a row; leaves the state at the START (the adjoint
//      at the END) of every chunk in fp32 in place of the increments and writes the checkpoints (64 x 64 fp32: those only,
//      19 -> 16 us, where the call has them).  Small calls do without it (chain_in_place).
//   3  lfw_xpar_fwd_kernel / lfw_xpar_bwd_kernel: the recurrence itself, step by step, within each chunk; the last chunk's
//      leaves the final state, the first one's d_s0.  64 x 64 fp32 (lfw_xpar64.hip): on fp64 matrix instructions where the
//      gates and values allow it, and one more launch for the chunks where they don't.
//
// A row is left to the recurrence over the whole sequence where the sums could differ from it by more than rounding:
//   * a gate of magnitude above one (or NaN): the product of one side's gates may overflow where the product of both
//     sides' does not;
//   * an input above XP_MAX_INPUT or a state above XP_MAX_STATE at a chunk's start or end (or NaN): with neither, no
//     state within a chunk exceeds 2^120 + 64 * 2^116 < 2^123.  What the recurrence makes infinite it keeps infinite; an
//     increment of decayed factors comes out finite, and infinity times a gate product that has underflowed is NaN.
// The workgroups of the row's first chunk (64 x 64 fp32: of the first four) do it in launch 3, the others of that row leave.
//
// B = 96, T = 1024, 64 x 64 fp32 (launch 3 in lfw_xpar64.hip): forward 31 + 16 + 54 + 4 us (220 per-step), backward 26 + 11 +
// 154 + 6 us (813).  13 rows, T = 385, 33 x 17 fp16, without launch 2: 6 + 20 us (76) and 6 + 38 us (251).
//
// Replaces lfw_cuda_fwd_kernel, lfw_cuda_bwd_kernel and the einsums of the reference
// (t2fw/csrc/lfw_kernel.cu:18-102, t2fw/csrc/lfw.cpp:45,84-93); semantics t2fw/torch.py:21-31.
#include <type_traits>

#include "lfw_par.hpp"
#include "lfw_scan_body.hpp"
#include "lfw_xpar.hpp"

namespace t2fw {
namespace {

constexpr int XI_THREADS = 512;
constexpr int XLS = 68;                // row stride, in floats, of the token-major tiles [64][XLS]

// What launches 1 and 2 read and write; BWD swaps the arrays and the direction of the products.
struct PassArgs {
    const void *val, *gate_val, *key, *gate_key;      // x f k f_key, or g_out f q f_key
    const void *first;                                 // s0, or g_state
    void *ckpt;                                        // may be null; null backward
    XparScratch ws;
    int64_t T, NC;
    int32_t D, K, heads;
};

// ---- launch 1 -------------------------------------------------------------------------------------
// Waves (side, 16 channels): lane (i, kg) owns channel 16 cb + i and tokens 16 m + 4 kg + j.
template <typename IO, bool BWD> __global__ __launch_bounds__(XI_THREADS) void lfw_xpar_incr_kernel(PassArgs p) {
    __shared__ __align__(16) float smem[2 * XP_CHUNK * XLS];
    const int64_t item = blockIdx.x, b = item / p.NC;
    const int chunk = (int)(item - b * p.NC);
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int side = w >> 2, cb = w & 3, i = lane & 15, kg = lane >> 4, c = 16 * cb + i;
    const int width = side ? p.K : p.D, Dp = xp_padded(p.D), Kp = xp_padded(p.K);
    const int n_tok = (int)min((int64_t)XP_CHUNK, p.T - (int64_t)chunk * XP_CHUNK);
    float *const VS = smem, *const KS = smem + XP_CHUNK * XLS;
    int bad = 0, small = 0;
    if (16 * cb < width) {                       // wave-uniform
        const int64_t off = uniform64((row_first_token(b, p.T, p.heads) + (int64_t)chunk * XP_CHUNK * p.heads) * width);
        const IO *const gp = (const IO *)(side ? p.gate_key : p.gate_val) + off;
        const IO *const ap = (const IO *)(side ? p.key : p.val) + off;
        const u32 ts = (u32)(p.heads * width);
        const bool ch_ok = c < width;
        const u32 cc = ch_ok ? (u32)c : 0u;
        // tokens past the end are read from the last one and act as identity
        IO rg[4][4], ra[4][4];
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32 o = (u32)min(16 * m + 4 * kg + j, n_tok - 1) * ts + cc;
                rg[m][j] = gp[o];
                ra[m][j] = ap[o];
            }
        float *const tile = side ? KS : VS;
        float carry = 1.0f;
#pragma unroll
        for (int mm = 0; mm < 4; ++mm) {
            const int m = BWD ? mm : 3 - mm;
            float g[4], l[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                g[j] = (ch_ok && 16 * m + 4 * kg + j < n_tok) ? to_acc(rg[m][j]) : 1.0f;
                bad |= !(fabsf(g[j]) <= 1.0f) ? 1 : 0;
                small |= !(g[j] >= XP_MM_MIN_GATE) ? 1 : 0;
            }
            float own;                           // product of the lane's four gates
            if (BWD) {                           // l: up to and with the token
                l[0] = g[0];
#pragma unroll
                for (int j = 1; j < 4; ++j) l[j] = l[j - 1] * g[j];
                own = l[3];
            } else {                             // l: after the token
                l[3] = 1.0f;
#pragma unroll
                for (int j = 2; j >= 0; --j) l[j] = l[j + 1] * g[j + 1];
                own = l[0] * g[0];
            }
            const u32 vb = __float_as_uint(own);
            const auto s16 = __builtin_amdgcn_permlane16_swap(vb, vb, false, false);     // {even row of the pair, odd row}
            const float ev = __uint_as_float(s16[0]), od = __uint_as_float(s16[1]);
            const u32 pb = __float_as_uint(ev * od);
            const auto s32 = __builtin_amdgcn_permlane32_swap(pb, pb, false, false);     // {rows 0-1, rows 2-3}
            const float lo = __uint_as_float(s32[0]), hi = __uint_as_float(s32[1]);
            const float rest = BWD ? ((kg & 1) ? ev : 1.0f) * ((kg & 2) ? lo : 1.0f)
                                   : ((kg & 1) ? 1.0f : od) * ((kg & 2) ? 1.0f : hi);
            const float base = carry * rest;
            carry *= lo * hi;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int t = 16 * m + 4 * kg + j;
                const float a = (ch_ok && t < n_tok) ? to_acc(ra[m][j]) : 0.0f;
                bad |= !(fabsf(a) <= XP_MAX_INPUT) ? 1 : 0;
                tile[t * XLS + c] = a * (base * l[j]);
            }
        }
        if (kg == 0) p.ws.tots[item * (Dp + Kp) + (side ? Dp : 0) + c] = carry;
    }
    const int any = __syncthreads_or(bad | small), left = any ? __syncthreads_or(bad) : 0;      // any: the same in every thread
    if (tid == 0) p.ws.chunk_flags[item] = left ? XP_ROW_LEFT : any ? XP_CHUNK_STEPS : 0;
    // wave w: key channels of blocks kb, value channels of block db; a lane stores four consecutive k of its d
    const int db = w & 3;
    if (16 * db >= p.D) return;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int kb = 2 * (w >> 2) + u;
        if (16 * kb >= p.K) break;
        // Steps close to where the products start weigh most: each group of 16 steps is summed by itself, and the
        // groups from the lightest to the heaviest, so that little is rounded at the size of the whole sum.
        floatx4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int nn = 0; nn < 4; ++nn) {
            const int n = BWD ? 3 - nn : nn;
            floatx4 m0 = {0.f, 0.f, 0.f, 0.f}, m1 = m0;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = (16 * n + 4 * kg + e) * XLS;
                const float kv = KS[row + 16 * kb + i], dv = VS[row + 16 * db + i];
                if (e & 1)
                    m1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv, dv, m1, 0, 0, 0);
                else
                    m0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kv, dv, m0, 0, 0, 0);
            }
            sum += m0 + m1;
        }
        *reinterpret_cast<float4 *>(p.ws.states + item * (Dp * Kp) + (16 * db + i) * Kp + 16 * kb + 4 * kg) =
            make_float4(sum[0], sum[1], sum[2], sum[3]);
    }
}

// ---- launch 2 -------------------------------------------------------------------------------------
// Four workgroups per row, a thread owns four consecutive k of one d.  The loads of a batch of chunks do not depend on
// the chain and are all issued before it.
constexpr int XC_THREADS = 256, XC_BATCH = 8;
template <typename IO, bool BWD> __global__ __launch_bounds__(XC_THREADS) void lfw_xpar_chain_kernel(PassArgs p) {
    const int64_t b = blockIdx.x >> 2;
    const int idx = (blockIdx.x & 3) * XC_THREADS + threadIdx.x, d = idx >> 4, k = (idx & 15) * 4;
    const int D = p.D, K = p.K, NC = (int)p.NC, Dp = xp_padded(D), Kp = xp_padded(K);
    int bad = 0;
    for (int c = threadIdx.x; c < NC; c += XC_THREADS) bad |= p.ws.chunk_flags[b * NC + c] & XP_ROW_LEFT;
    if (d < D && k < K) {
        const int64_t DK = (int64_t)D * K, o = d * K + k;
        float S[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            S[e] = k + e < K ? to_acc(((const IO *)p.first)[b * DK + o + e]) : 0.0f;
            bad |= !(fabsf(S[e]) <= XP_MAX_STATE) ? 1 : 0;
        }
        float *const st = p.ws.states + b * NC * (int64_t)(Dp * Kp) + d * Kp + k;
        const float *const tots = p.ws.tots + b * NC * (int64_t)(Dp + Kp);
        IO *const ckpt = p.ckpt != nullptr ? (IO *)p.ckpt + b * NC * DK + o : nullptr;
        // 64 x 64 fp32 states are read from the checkpoints, where those are asked for (lfw_xpar64.hip)
        const bool keep = !std::is_same<IO, float>::value || BWD || ckpt == nullptr || D != XP_N || K != XP_N;
        for (int n0 = 0; n0 < NC; n0 += XC_BATCH) {
            float4 m[XC_BATCH], tb[XC_BATCH];
            float ta[XC_BATCH];
#pragma unroll
            for (int u = 0; u < XC_BATCH; ++u) {
                const int n = min(n0 + u, NC - 1), c = BWD ? NC - 1 - n : n;
                m[u] = *reinterpret_cast<const float4 *>(st + (int64_t)c * (Dp * Kp));
                ta[u] = tots[c * (int64_t)(Dp + Kp) + d];
                tb[u] = *reinterpret_cast<const float4 *>(tots + c * (int64_t)(Dp + Kp) + Dp + k);
            }
#pragma unroll
            for (int u = 0; u < XC_BATCH; ++u) {
                if (n0 + u >= NC) break;
                const int c = BWD ? NC - 1 - (n0 + u) : n0 + u;
                if (keep) *reinterpret_cast<float4 *>(st + (int64_t)c * (Dp * Kp)) = make_float4(S[0], S[1], S[2], S[3]);
                if (!BWD && ckpt != nullptr) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (k + e < K) ckpt[c * DK + e] = from_acc<IO>(S[e]);
                }
                const float mv[4] = {m[u].x, m[u].y, m[u].z, m[u].w}, tv[4] = {tb[u].x, tb[u].y, tb[u].z, tb[u].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    S[e] = S[e] * (ta[u] * tv[e]) + mv[e];
                    bad |= (k + e >= K || fabsf(S[e]) <= XP_MAX_STATE) ? 0 : 1;
                }
            }
        }
    }
    const int any = __syncthreads_or(bad);
    if (threadIdx.x == 0) p.ws.row_flags[blockIdx.x] = any;
}

// Small calls without launch 2: every workgroup of launch 3 goes through its row's whole chain itself, all elements of the state in
// the same order (the verdict on a row is on all of them), and keeps the state at its own chunk's edge in LDS, [Dp][Kp] floats.
// The row's verdict.  What bounds it: one memory latency per batch of a thread's element (chain_is_in_place).  Three elements
// at a time were no faster (33 x 17: 72 us in the place of 71), with the gate products in LDS slower (75).
template <typename IO, bool BWD>
__device__ __forceinline__ bool chain_in_place(const XparScratch &ws, const void *first, int D, int K, int NC, int64_t b, int chunk, float *edge) {
    const int Dp = xp_padded(D), Kp = xp_padded(K), tid = threadIdx.x;
    int bad = 0;
    for (int c = tid; c < NC; c += SCAN_THREADS) bad |= ws.chunk_flags[b * NC + c] & XP_ROW_LEFT;
    const float *const st = ws.states + b * NC * (int64_t)(Dp * Kp), *const tots = ws.tots + b * NC * (int64_t)(Dp + Kp);
    for (int o = tid; o < Dp * Kp; o += SCAN_THREADS) {
        const int d = o / Kp, k = o - d * Kp;
        if (d >= D || k >= K) continue;
        float S = to_acc(((const IO *)first)[(b * D + d) * K + k]);
        bad |= !(fabsf(S) <= XP_MAX_STATE) ? 1 : 0;
        for (int n0 = 0; n0 < NC; n0 += XC_BATCH) {
            float m[XC_BATCH], ta[XC_BATCH], tb[XC_BATCH];
#pragma unroll
            for (int u = 0; u < XC_BATCH; ++u) {
                const int n = min(n0 + u, NC - 1), c = BWD ? NC - 1 - n : n;
                m[u] = st[c * (Dp * Kp) + o];
                ta[u] = tots[c * (Dp + Kp) + d];
                tb[u] = tots[c * (Dp + Kp) + Dp + k];
            }
#pragma unroll
            for (int u = 0; u < XC_BATCH; ++u) {
                if (n0 + u >= NC) break;
                if ((BWD ? NC - 1 - (n0 + u) : n0 + u) == chunk) edge[o] = S;
                S = S * (ta[u] * tb[u]) + m[u];
                bad |= fabsf(S) <= XP_MAX_STATE ? 0 : 1;
            }
        }
    }
    return __syncthreads_or(bad) != 0;
}

// ---- launch 3 -------------------------------------------------------------------------------------
// IN_PLACE: without launch 2 (chain_in_place; the state lies behind the body's LDS, `edge` bytes from its start).
// Workgroups are numbered chunk by chunk, all rows of a chunk together, so that those that may have a whole row to do come
// first and next to each other.  Numbered row by row, the ones with work were 16 chunks apart, all on the same one or two
// dies and shader engines: 96 rows x 1024 steps with a gate above one in each, 32 x 32 fp32, forward + backward 2050 us
// against 563 now and 752 on the per-step kernels; 64 x 64 7300, 1019, 992 (96 x 256 590, 277, 264; 16 x 1024 1430, 604,
// 909).
// One workgroup per (row, chunk, 16 value channels); base: the call over whole rows.
template <typename IO, int KPL, bool IN_PLACE> __global__ __launch_bounds__(SCAN_THREADS) void lfw_xpar_fwd_kernel(ScanFwdArgs base, XparScratch ws, int64_t NC, int edge) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float *const entering = reinterpret_cast<float *>(smem_raw + edge);
    const int64_t pair = blockIdx.x / base.ntiles, b = pair % base.B;
    const int tile = (int)(blockIdx.x - pair * base.ntiles), chunk = (int)(pair / base.B);
    const int64_t item = b * NC + chunk;
    bool left;
    if constexpr (IN_PLACE)
        left = chain_in_place<IO, false>(ws, base.s0, (int)base.D, (int)base.K, (int)NC, b, chunk, entering);
    else
        left = row_left(ws, b);
    if (left) {
        if (chunk == 0) scan::fwd_scan_body_kg<IO, KPL, 16>(base, b, tile);
        return;
    }
    const int64_t line = row_first_token(b, base.T, base.heads) + (int64_t)chunk * XP_CHUNK * base.heads;
    ScanFwdArgs a = base;
    a.x = (const IO *)base.x + line * base.D; a.f = (const IO *)base.f + line * base.D;
    a.q = (const IO *)base.q + line * base.K; a.k = (const IO *)base.k + line * base.K;
    a.f_key = (const IO *)base.f_key + line * base.K;
    a.out = (IO *)base.out + line * base.D;
    if constexpr (IN_PLACE) {
        if (base.ckpt != nullptr) {
            const int D = (int)base.D, K = (int)base.K, rows = min(16, D - 16 * tile);
            IO *const to = (IO *)base.ckpt + (item * D + 16 * tile) * K;
            for (int o = threadIdx.x; o < rows * K; o += SCAN_THREADS) to[o] = from_acc<IO>(entering[(16 * tile + o / K) * xp_padded(K) + o % K]);
        }
    }
    a.ckpt = nullptr;
    a.next_state = chunk == (int)NC - 1 ? (IO *)base.next_state + b * base.D * base.K : nullptr;
    a.s_stride = xp_padded(base.K);
    a.s_start = IN_PLACE ? entering : ws.states + item * (xp_padded(base.D) * xp_padded(base.K));
    a.T = min((int64_t)XP_CHUNK, base.T - (int64_t)chunk * XP_CHUNK);
    scan::fwd_scan_body_kg<IO, KPL, 16>(a, 0, tile);
}

// One workgroup per (row, chunk, 16 channels of one side); KV, KK: columns per lane on the value and on the key side.
template <typename IO, int KV, int KK, bool IN_PLACE> __global__ __launch_bounds__(SCAN_THREADS) void lfw_xpar_bwd_kernel(ScanBwdArgs base, XparScratch ws, int edge) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    float *const entering = reinterpret_cast<float *>(smem_raw + edge);
    const int nd = ((int)base.D + 15) / 16, per = nd + ((int)base.K + 15) / 16;
    const int64_t pair = blockIdx.x / per, b = pair % base.B;
    const int tile = (int)(blockIdx.x - pair * per), chunk = (int)(pair / base.B);
    const int64_t item = b * base.NC + chunk;
    ScanBwdArgs a = base;
    int64_t row = b;
    bool left;
    if constexpr (IN_PLACE)
        left = chain_in_place<IO, true>(ws, base.g_state, (int)base.D, (int)base.K, (int)base.NC, b, chunk, entering);
    else
        left = row_left(ws, b);
    if (left) {
        if (chunk != 0) return;
    } else {
        const int64_t line = row_first_token(b, base.T, base.heads) + (int64_t)chunk * XP_CHUNK * base.heads;
        a.x = (const IO *)base.x + line * base.D; a.f = (const IO *)base.f + line * base.D;
        a.g_out = (const IO *)base.g_out + line * base.D;
        a.q = (const IO *)base.q + line * base.K; a.k = (const IO *)base.k + line * base.K;
        a.f_key = (const IO *)base.f_key + line * base.K;
        a.ckpt = (const IO *)base.ckpt + item * (base.D * base.K);
        a.d_x = (IO *)base.d_x + line * base.D; a.d_f = (IO *)base.d_f + line * base.D;
        a.d_q = (IO *)base.d_q + line * base.K; a.d_k = (IO *)base.d_k + line * base.K;
        a.d_f_key = (IO *)base.d_f_key + line * base.K;
        a.d_s0 = chunk == 0 ? (IO *)base.d_s0 + b * base.D * base.K : nullptr;
        a.g_stride = xp_padded(base.K);
        a.g_end = IN_PLACE ? entering : ws.states + item * (xp_padded(base.D) * xp_padded(base.K));
        a.T = min((int64_t)XP_CHUNK, base.T - (int64_t)chunk * XP_CHUNK);
        a.NC = 1;
        row = 0;
    }
    if (tile < nd)
        scan::bwd_scan_body_kg<IO, KK, 0, 16, 1>(a, row, tile);
    else
        scan::bwd_scan_body_kg<IO, KV, 1, 16, 1>(a, row, tile - nd);
}

// Whether `tiles` workgroups per (row, chunk) go through the chain themselves: few batches of loads per thread, and not too much
// to read in all.  Two measures, with launch 2 / in place, us:
//   GPU time of forward + backward, fp16: 1 x 230 of 9 x 5 57 / 52, 16 x 1024 of 16 x 8 66 / 57, 64 x 512 of 16 x 16 73 / 66, 13 x 385 of
//   33 x 17 (six batches) 69 / 71, 16 x 512 of 63 x 32 (eight) 77 / 81.  Forwards one after the other: 13 x 385 of 33 x 17 24.6 / 24.5,
//   6 x 512 of 63 x 32 24.7 / 26.8.
//   A training step as issued, which the host bounds and which has two launches fewer of six: 16 x 700 of 16 x 8 151 / 141, 13 x 385 of
//   33 x 17 149 / 135, 6 x 512 of 63 x 32 153 / 141, 4 x 448 of 63 x 63 (sixteen batches) 150 / 141.
// The line lies at six batches, where a forward by itself breaks even: there a step that the host does not bound (replayed from a
// graph) loses 2 us of GPU time and one that it does gains 12; beyond it every forward would lose.
constexpr int64_t XC_IN_PLACE_READS = 5 << 20;             // floats
bool chain_is_in_place(int64_t B, int64_t NC, int D, int K, int tiles) {
    const int64_t state = (int64_t)xp_padded(D) * xp_padded(K);
    return state / SCAN_THREADS * ((NC + XC_BATCH - 1) / XC_BATCH) <= 6 && B * NC * tiles <= XC_IN_PLACE_READS / (NC * state);
}

template <typename IO, bool BWD> int entering_states(const PassArgs &p, int64_t B, bool in_place, hipStream_t stream) {
    hipLaunchKernelGGL((lfw_xpar_incr_kernel<IO, BWD>), dim3((unsigned)(B * p.NC)), dim3(XI_THREADS), 0, stream, p);
    const int rc = check_hip(hipGetLastError(), "lfw_xpar_incr_kernel launch");
    if (rc || in_place) return rc;
    hipLaunchKernelGGL((lfw_xpar_chain_kernel<IO, BWD>), dim3((unsigned)(4 * B)), dim3(XC_THREADS), 0, stream, p);
    return check_hip(hipGetLastError(), "lfw_xpar_chain_kernel launch");
}

template <typename IO> int forward(const XparFwdArgs &a, hipStream_t stream) {
    PassArgs p{};
    p.val = a.x; p.gate_val = a.f; p.key = a.k; p.gate_key = a.f_key;
    p.first = a.s0; p.ckpt = a.ckpt;
    p.ws = a.ws; p.T = a.T; p.NC = a.NC; p.D = a.D; p.K = a.K; p.heads = a.heads;
    const bool own = std::is_same<IO, float>::value && a.D == XP_N && a.K == XP_N;      // kernels of its own, which read the chain's results
    // without launch 2 every workgroup of launch 3 reads the state that the row starts from while others write results, which must
    // not lie where it does (next_state in the place of s0); the same for the adjoint in the backward
    const int64_t es = sizeof(IO), state = a.B * a.D * a.K * es;
    const bool in_place = !own && chain_is_in_place(a.B, a.NC, a.D, a.K, (a.D + 15) / 16) &&
                          !meets_any({a.s0, state}, {{a.next_state, state}, {a.out, a.B * a.T * a.D * es}, {a.ckpt, state * a.NC}});
    const int rc = entering_states<IO, false>(p, a.B, in_place, stream);
    if (rc) return rc;
    if (own) return xpar64_forward(a, stream);
    const int kpl = a.K <= 32 ? 2 : 4, tb = 32;
    ScanFwdArgs s{};
    s.x = a.x; s.f = a.f; s.q = a.q; s.k = a.k; s.f_key = a.f_key; s.s0 = a.s0;
    s.out = a.out; s.next_state = a.next_state; s.ckpt = a.ckpt;
    s.B = a.B; s.T = a.T; s.D = a.D; s.K = a.K; s.NC = a.ckpt != nullptr ? a.NC : 1;
    s.C = a.ckpt != nullptr ? XP_CHUNK : 1; s.kg = 16; s.tb = tb; s.ntiles = (a.D + 15) / 16; s.heads = a.heads;
    const dim3 grid((unsigned)(a.B * a.NC * s.ntiles));
    const size_t body = (scan_fwd_lds_bytes(tb, 16, kpl, 16) + 15) / 16 * 16, smem = body + (in_place ? 4 * xp_padded(a.D) * xp_padded(a.K) : 0);
    auto kern = in_place ? (kpl == 2 ? lfw_xpar_fwd_kernel<IO, 2, true> : lfw_xpar_fwd_kernel<IO, 4, true>)
                         : (kpl == 2 ? lfw_xpar_fwd_kernel<IO, 2, false> : lfw_xpar_fwd_kernel<IO, 4, false>);
    hipLaunchKernelGGL(kern, grid, dim3(SCAN_THREADS), smem, stream, s, a.ws, a.NC, (int)body);
    return check_hip(hipGetLastError(), "lfw_xpar_fwd_kernel launch");
}

template <typename IO> int backward(const XparBwdArgs &a, hipStream_t stream) {
    PassArgs p{};
    p.val = a.g_out; p.gate_val = a.f; p.key = a.q; p.gate_key = a.f_key;
    p.first = a.g_state;
    p.ws = a.ws; p.T = a.T; p.NC = a.NC; p.D = a.D; p.K = a.K; p.heads = a.heads;
    const bool own = std::is_same<IO, float>::value && a.D == XP_N && a.K == XP_N;
    const int64_t es = sizeof(IO), state = a.B * a.D * a.K * es, value = a.B * a.T * a.D * es, key = a.B * a.T * a.K * es;
    const bool in_place = !own && chain_is_in_place(a.B, a.NC, a.D, a.K, (a.D + 15) / 16 + (a.K + 15) / 16) &&
                          !meets_any({a.g_state, state}, {{a.d_s0, state}, {a.d_x, value}, {a.d_f, value}, {a.d_q, key}, {a.d_k, key}, {a.d_f_key, key}});
    const int rc = entering_states<IO, true>(p, a.B, in_place, stream);
    if (rc) return rc;
    if (own) return xpar64_backward(a, stream);
    ScanBwdArgs s{};
    s.g_out = a.g_out; s.g_state = a.g_state; s.x = a.x; s.f = a.f; s.q = a.q; s.k = a.k; s.f_key = a.f_key; s.ckpt = a.ckpt;
    s.d_x = a.d_x; s.d_f = a.d_f; s.d_q = a.d_q; s.d_k = a.d_k; s.d_f_key = a.d_f_key; s.d_s0 = a.d_s0;
    s.B = a.B; s.T = a.T; s.D = a.D; s.K = a.K; s.NC = a.NC; s.C = XP_CHUNK; s.kg = 16; s.use_sub = 1; s.heads = a.heads;
    const dim3 grid((unsigned)(a.B * a.NC * ((a.D + 15) / 16 + (a.K + 15) / 16)));
    const int kv = a.D <= 32 ? 2 : 4, kk = a.K <= 32 ? 2 : 4;
    const size_t body = (scan_bwd_lds_bytes(scan::SegLen<4>::value, 16, kv > kk ? kv : kk, 16, XP_CHUNK, true) + 15) / 16 * 16;
    const size_t smem = body + (in_place ? 4 * xp_padded(a.D) * xp_padded(a.K) : 0);
    auto pick = [&](auto flag) {
        constexpr bool IN = decltype(flag)::value;
        return kv == 4 ? (kk == 4 ? lfw_xpar_bwd_kernel<IO, 4, 4, IN> : lfw_xpar_bwd_kernel<IO, 4, 2, IN>)
                       : (kk == 4 ? lfw_xpar_bwd_kernel<IO, 2, 4, IN> : lfw_xpar_bwd_kernel<IO, 2, 2, IN>);
    };
    auto kern = in_place ? pick(std::true_type{}) : pick(std::false_type{});
    hipLaunchKernelGGL(kern, grid, dim3(SCAN_THREADS), smem, stream, s, a.ws, (int)body);
    return check_hip(hipGetLastError(), "lfw_xpar_bwd_kernel launch");
}

}  // namespace

int xpar_forward(const XparFwdArgs &a, int dtype, hipStream_t stream) {
    switch (dtype) {
        case T2FW_F32: return forward<float>(a, stream);
        case T2FW_F16: return forward<__half>(a, stream);
        case T2FW_BF16: return forward<__hip_bfloat16>(a, stream);
    }
    return fail(T2FW_ERR_UNSUPPORTED, "the chunk-parallel exact kernels take fp32, fp16 or bf16 tensors");
}

int xpar_backward(const XparBwdArgs &a, int dtype, hipStream_t stream) {
    switch (dtype) {
        case T2FW_F32: return backward<float>(a, stream);
        case T2FW_F16: return backward<__half>(a, stream);
        case T2FW_BF16: return backward<__hip_bfloat16>(a, stream);
    }
    return fail(T2FW_ERR_UNSUPPORTED, "the chunk-parallel exact kernels take fp32, fp16 or bf16 tensors");
}

}  // namespace t2fw
