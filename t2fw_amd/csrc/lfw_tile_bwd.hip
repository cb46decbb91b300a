// Backward pass of the decay rule on fp32 matrix cores, chunk-parallel (operands and lane layout: lfw_tile.hpp).
//
// A chunk is the 64 tokens between two checkpoints.  Four launches:
//   1  lfw_tile_incr_kernel, a workgroup per (row, chunk): the chunk's increment of the adjoint, sum_t (g_t a_t) (x) (q_t b_t)
//      with prefix products from the chunk's start (no inverses: any gates), and the chunk's gate products;
//   2  lfw_tile_scan_kernel, elementwise: the adjoint chain over the chunks of a row, last to first; leaves the adjoint
//      at the END of every chunk in place of the increments and writes d_s0;
//   3  lfw_tile_grads_kernel, a workgroup per (row, chunk): everything else.  Per tile of 16 tokens, with S the state
//      before it and G the adjoint after it, in the scalings of lfw_tile.hpp (o', q', x', k' leave out the token's own
//      write):
//        value side  o'_t = lo_d (qm_t . S') + sum_{s<t} P[t,s] xm_s       x'_t = up_d (km_t . G') + sum_{r>t} P[r,t] gm_r
//        key side    q'_t, k'_t: the same with W[t,s] = gm_t . xm_s instead of P[t,s] = qm_t . km_s
//        d_x_t = (x'_t + gm_t P[t,t]) / a'_t   d_k_t likewise   d_q_t = (q'_t + km_t W[t,t]) b'_t
//        f_t d_f_t = rowsum(G_end * S_end) + sum_{r>=t} (gm_r o'_r - xm_r x'_r)        (key side likewise)
//      A wave sweeps its slab of the state forwards over the four tiles, then its slab of the adjoint backwards;
//   4  lfw_tile_exact_kernel: the exact recurrence for the chunks that launch 3 left out (a list in the workspace): gates
//      outside [min_gate, 1] or operands out of range.  Chunks are independent once launch 2 is done.
//
// B = 96, T = 1024, 64 x 64 fp32: 23 + 11 + 117 + 4.5 us (nothing listed) against 801 us for the two per-step launches;
// 13 rows, T = 385, 33 x 17 fp16: 4.8 + 4.2 + 18.5 + 3.8 against 251 us.  Launch 3 needs 72 products of 16 x 16 x 16 per
// wave and chunk, 46 us of the chip's fp32 matrix rate at the first size.
//
// Replaces lfw_cuda_bwd_kernel and the six einsums of the reference
// (t2fw/csrc/lfw_kernel.cu:61-102, t2fw/csrc/lfw.cpp:84-93).
#include <algorithm>

#include "lfw_par.hpp"
#include "lfw_scan_body.hpp"
#include "lfw_tile.hpp"

namespace t2fw {
namespace {

using namespace tilem;

constexpr int TB_THREADS = 512;        // waves (side, channel block)

// f_t d_f_t comes out with the rounding of the terms it is the sum of (2^-24 of them for every type), and d_f_t is that
// over f_t: gates below this go to the exact recurrence, so that the division costs an fp32 gradient no more than the
// accuracy class of the exact kernels (2^-17 of the terms) and a 16-bit one less than its own rounding.
template <typename IO> struct MinGate { static constexpr float value = 0.0009765625f; };      // 2^-10
template <> struct MinGate<float> { static constexpr float value = 0.0078125f; };             // 2^-7

template <bool W64> __device__ __forceinline__ int nblocks(int n) { return W64 ? 4 : (n + 15) >> 4; }

// ---- launch 1 -------------------------------------------------------------------------------------
template <typename IO, bool W64, bool FULL>
__device__ __forceinline__ void incr_item(const TileBwdArgs &p, float *smem, int64_t item, int64_t b, int chunk) {
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int side = w >> 2, cb = w & 3, i = lane & 15, kg = lane >> 4, c = 16 * cb + i;
    const int T = (int)p.T, width = W64 ? CH_N : (side ? p.K : p.D);
    const int64_t off = uniform64((row_first_token(b, p.T, p.heads) + (int64_t)(chunk * TILE_CHUNK) * p.heads) * width);
    float *const GS = smem, *const QS = smem + TL_FLOATS;
    if (W64 || cb < nblocks<W64>(width)) {
        const u32 ts = (u32)(p.heads * width), lane_off = (u32)(4 * kg) * ts + (u32)min(c, width - 1);
        const int n_left = T - chunk * TILE_CHUNK - 4 * kg;
        const bool ch_ok = W64 || c < width;
        IO rg[4][4], ra[4][4];
        load_tile_tokens<IO, FULL>(rg, (const IO *)(side ? p.f_key : p.f) + off, lane_off, ts, n_left);
        load_tile_tokens<IO, FULL>(ra, (const IO *)(side ? p.q : p.g_out) + off, lane_off, ts, n_left);
        float *const tile = side ? QS : GS;
        float carry = 1.0f;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            float l[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float g = (ch_ok && (FULL || 16 * m + j < n_left)) ? to_acc(rg[m][j]) : 1.0f;
                l[j] = j == 0 ? g : l[j > 0 ? j - 1 : 0] * g;
            }
            const par::RowScan s = par::row_scan_mul(l[3], kg);
            const float first = carry * s.lower;
            carry *= s.all;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float a = (ch_ok && (FULL || 16 * m + j < n_left)) ? to_acc(ra[m][j]) : 0.0f;
                tile[(16 * m + 4 * kg + j) * TLS + c] = a * (first * l[j]);
            }
        }
        if (kg == 0) p.tots[(item * 2 + side) * CH_N + c] = carry;
    }
    __syncthreads();
    // wave w: rows k of blocks kb, column d of block db; a lane stores four consecutive k of its d
    const int db = w & 3, nbd = nblocks<W64>(W64 ? CH_N : p.D), nbk = nblocks<W64>(W64 ? CH_N : p.K);
    if (!W64 && db >= nbd) return;
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int kb = 2 * (w >> 2) + u;
        if (!W64 && kb >= nbk) break;
        floatx4 m0 = {0.f, 0.f, 0.f, 0.f}, m1 = m0;
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int row = (16 * n + 4 * kg + e) * TLS;
                const float kv = QS[row + 16 * kb + i], dv = GS[row + 16 * db + i];
                if (e & 1)
                    m1 = mfma4(kv, dv, m1);
                else
                    m0 = mfma4(kv, dv, m0);
            }
        *reinterpret_cast<float4 *>(p.gh + item * (CH_N * CH_N) + (16 * db + i) * CH_N + 16 * kb + 4 * kg) =
            make_float4(m0[0] + m1[0], m0[1] + m1[1], m0[2] + m1[2], m0[3] + m1[3]);
    }
}
template <typename IO, bool W64> __global__ __launch_bounds__(TB_THREADS) void lfw_tile_incr_kernel(TileBwdArgs p) {
    __shared__ __align__(16) float smem[2 * TL_FLOATS];
    const int64_t item = blockIdx.x, b = item / p.NC;
    const int chunk = (int)(item - b * p.NC);
    if (threadIdx.x == 0) {
        if (item == 0) p.list[0] = 0;
        p.flags[item] = 0;
    }
    if ((chunk + 1) * TILE_CHUNK <= (int)p.T)
        incr_item<IO, W64, true>(p, smem, item, b, chunk);
    else
        incr_item<IO, W64, false>(p, smem, item, b, chunk);
}

// ---- launch 2 -------------------------------------------------------------------------------------
// Four workgroups per row, a thread owns four consecutive k of one d.  The loads of a batch of chunks do not depend on
// the chain and are all issued before it.
constexpr int TS_THREADS = 256, TS_BATCH = 8;
template <typename IO, bool W64> __global__ __launch_bounds__(TS_THREADS) void lfw_tile_scan_kernel(TileBwdArgs p) {
    const int64_t b = blockIdx.x >> 2;
    const int idx = (blockIdx.x & 3) * TS_THREADS + threadIdx.x, d = idx >> 4, k = (idx & 15) * 4;
    const int D = W64 ? CH_N : p.D, K = W64 ? CH_N : p.K, NC = (int)p.NC;
    if (!W64 && (d >= D || k >= K)) return;
    float G[4];
    const IO *const gs = (const IO *)p.g_state + b * ((int64_t)D * K) + d * K + k;
#pragma unroll
    for (int e = 0; e < 4; ++e) G[e] = (W64 || k + e < K) ? to_acc(gs[e]) : 0.0f;
    float *const gh = p.gh + b * NC * (int64_t)(CH_N * CH_N) + d * CH_N + k;
    const float *const tots = p.tots + b * NC * (int64_t)(2 * CH_N);
    for (int top = NC - 1; top >= 0; top -= TS_BATCH) {
        float4 m[TS_BATCH], tb[TS_BATCH];
        float ta[TS_BATCH];
#pragma unroll
        for (int u = 0; u < TS_BATCH; ++u) {
            const int c = max(top - u, 0);
            m[u] = ldv4(gh + (int64_t)c * (CH_N * CH_N));
            ta[u] = tots[c * 2 * CH_N + d];
            tb[u] = ldv4(tots + c * 2 * CH_N + CH_N + k);
        }
#pragma unroll
        for (int u = 0; u < TS_BATCH; ++u) {
            if (top - u >= 0) {
                *reinterpret_cast<float4 *>(gh + (int64_t)(top - u) * (CH_N * CH_N)) = make_float4(G[0], G[1], G[2], G[3]);
                const bool ok = fabsf(G[0]) <= TILE_MAX_STATE && fabsf(G[1]) <= TILE_MAX_STATE &&
                                fabsf(G[2]) <= TILE_MAX_STATE && fabsf(G[3]) <= TILE_MAX_STATE;
                if (!ok) p.flags[b * NC + top - u] = 1;
                G[0] = G[0] * (ta[u] * tb[u].x) + m[u].x;
                G[1] = G[1] * (ta[u] * tb[u].y) + m[u].y;
                G[2] = G[2] * (ta[u] * tb[u].z) + m[u].z;
                G[3] = G[3] * (ta[u] * tb[u].w) + m[u].w;
            }
        }
    }
    IO *const ds = (IO *)p.d_s0 + b * ((int64_t)D * K) + d * K + k;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (W64 || k + e < K) ds[e] = from_acc<IO>(G[e]);
}

// ---- launch 3 -------------------------------------------------------------------------------------
struct GradSmem {
    float val[2][TL_FLOATS], adj[2][TL_FLOATS];      // xm / km, gm / qm of the two sides
    float vec[2][VEC_FLOATS], pt[2][4][PT_FLOATS], diag[2][CH_N];
    int bad[8];
};
static_assert(2 * ((sizeof(GradSmem) + 1279) / 1280 * 1280) <= 160 * 1024, "two workgroups must fit the LDS of one CU");

template <typename IO, bool W64, bool FULL, int SIDE> struct GradSide {
    const TileBwdArgs &p;
    GradSmem &sm;
    int64_t item, line0;
    int cb, i, kg, c, n_left, n_tok, width, owidth;
    u32 ts, lane_off;
    bool ch_ok;

    __device__ __forceinline__ GradSide(const TileBwdArgs &p_, GradSmem &sm_, int64_t item_, int64_t b, int chunk, int cb_, int lane)
        : p(p_), sm(sm_), item(item_), cb(cb_) {
        i = lane & 15; kg = lane >> 4; c = 16 * cb + i;
        width = W64 ? CH_N : (SIDE ? p.K : p.D);
        owidth = W64 ? CH_N : (SIDE ? p.D : p.K);
        line0 = uniform64(row_first_token(b, p.T, p.heads) + (int64_t)(chunk * TILE_CHUNK) * p.heads);
        ts = (u32)(p.heads * width);
        lane_off = (u32)(4 * kg) * ts + (u32)(W64 ? c : min(c, width - 1));
        n_tok = (int)p.T - chunk * TILE_CHUNK;
        n_left = n_tok - 4 * kg;
        ch_ok = W64 || c < width;
    }
    __device__ __forceinline__ bool tok_ok(int m, int j) const { return FULL || 16 * m + j < n_left; }
    // element (own channel, other side's channel 16 q + 4 kg + e) of a state whose rows are `stride` long
    __device__ __forceinline__ int st_off(int q, int e, int stride) const {
        const int o = 16 * q + 4 * kg + e;
        return SIDE ? o * stride + c : c * stride + o;
    }
    __device__ __forceinline__ bool el_ok(int q, int e) const { return W64 || (ch_ok && 16 * q + 4 * kg + e < owidth); }
    __device__ __forceinline__ void store4(IO *ubase, int m, const float (&v)[4]) const {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (tok_ok(m, j) && ch_ok) (ubase + (size_t)(16 * m + j) * ts)[lane_off] = from_acc<IO>(v[j]);
    }
    __device__ __forceinline__ void scale(floatx4 (&X)[4], const float *vec, int nbo) const {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!W64 && q >= nbo) break;
            const float4 v = ldv4(vec + 16 * q + 4 * kg);
            X[q][0] *= v.x; X[q][1] *= v.y; X[q][2] *= v.z; X[q][3] *= v.w;
        }
    }
    // rows of tokens 16 m + i of `tile` times the slab
    __device__ __forceinline__ floatx4 rows_times(const float *tile, int m, const floatx4 (&X)[4], int nbo) const {
        floatx4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            if (!W64 && q >= nbo) break;
            const float4 v = ldv4(tile + (16 * m + i) * TLS + 16 * q + 4 * kg);
            a0 = mfma4(v.x, X[q][0], a0);
            a1 = mfma4(v.y, X[q][1], a1);
            a0 = mfma4(v.z, X[q][2], a0);
            a1 = mfma4(v.w, X[q][3], a1);
        }
        return a0 + a1;
    }
    // X += (tokens of tile m of the other side)^T (x) (own tokens w)
    __device__ __forceinline__ void add_outer(floatx4 (&X)[4], const float *tile, int m, const float (&w)[4], int nbo) const {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (!W64 && q >= nbo) break;
                X[q] = mfma4(tile[(16 * m + 4 * kg + e) * TLS + 16 * q + i], w[e], X[q]);
            }
    }
    __device__ __forceinline__ void own_tokens(float (&v)[4], const float *tile, int m) const {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = tile[(16 * m + 4 * kg + e) * TLS + c];
    }

    __device__ __forceinline__ void run() const {
        const int nb = nblocks<W64>(width), nbo = nblocks<W64>(owidth), lane = 16 * kg + i;
        const bool active = W64 || cb < nb;
        float *const own_val = sm.val[SIDE], *const own_adj = sm.adj[SIDE];
        const float *const oth_val = sm.val[1 - SIDE], *const oth_adj = sm.adj[1 - SIDE], *const vec = sm.vec[1 - SIDE];
        const int64_t off = uniform64(line0 * width);
        float pre[4][4], rg0[4], lo[4], up[4];
        floatx4 S[4];
        u32 bad = (u32)p.flags[item];
        if (active) {
            IO rg[4][4], rv[4][4], ra[4][4];
            load_tile_tokens<IO, FULL>(rg, (const IO *)(SIDE ? p.f_key : p.f) + off, lane_off, ts, n_left);
            load_tile_tokens<IO, FULL>(rv, (const IO *)(SIDE ? p.k : p.x) + off, lane_off, ts, n_left);
            load_tile_tokens<IO, FULL>(ra, (const IO *)(SIDE ? p.q : p.g_out) + off, lane_off, ts, n_left);
            const IO *const s0 = (const IO *)p.ckpt + item * ((int64_t)(SIDE ? owidth : width) * (SIDE ? width : owidth));
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) S[q][e] = el_ok(q, e) ? to_acc(s0[st_off(q, e, SIDE ? width : owidth)]) : 0.0f;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                float g[4], inv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    g[j] = (tok_ok(m, j) && ch_ok) ? to_acc(rg[m][j]) : 1.0f;
                    bad |= !(g[j] <= 1.0f && g[j] >= MinGate<IO>::value) ? 1u : 0u;
                }
                rg0[m] = __builtin_amdgcn_rcpf(g[0]);
                const TileProducts tp = tile_products((g[0] * g[1]) * (g[2] * g[3]), kg);
                tile_scales(pre[m], inv, g, tp, kg);
                lo[m] = tp.lo; up[m] = tp.up;
                bad |= (tp.lo >= TILE_MIN_PRODUCT && tp.up >= TILE_MIN_PRODUCT) ? 0u : 1u;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const bool ok = tok_ok(m, j) && ch_ok;
                    const float v = (ok ? to_acc(rv[m][j]) : 0.0f) * inv[j], a = (ok ? to_acc(ra[m][j]) : 0.0f) * pre[m][j];
                    bad |= (fabsf(v) <= TILE_MAX_OPERAND && fabsf(a) <= TILE_MAX_OPERAND) ? 0u : 1u;
                    own_val[(16 * m + 4 * kg + j) * TLS + c] = v;
                    own_adj[(16 * m + 4 * kg + j) * TLS + c] = a;
                }
            }
            if (kg == 0) {
                float *v = sm.vec[SIDE] + c;
                v[0] = lo[0];
#pragma unroll
                for (int m = 0; m < 3; ++m) v[(m + 1) * CH_N] = up[m] * lo[m + 1];
                v[4 * CH_N] = up[3];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) bad |= fabsf(S[q][e]) <= TILE_MAX_STATE ? 0u : 1u;
        }
        {
            const int any = __any((int)bad);
            if (lane == 0) sm.bad[4 * SIDE + cb] = any;
        }
        __syncthreads();                         // tiles, factors and verdicts are there
        {
            int any = 0;
#pragma unroll
            for (int w = 0; w < 8; ++w) any |= sm.bad[w];
            if (__builtin_amdgcn_readfirstlane(any)) {      // the same in every wave of the workgroup
                if (SIDE == 0 && cb == 0 && lane == 0) p.list[1 + atomicAdd(p.list, 1)] = (int)item;
                return;
            }
        }
        {   // this side's product tile of token tile cb: [s][t], kept for s < t, and its diagonal
            floatx4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (!W64 && q >= nbo) break;
                const int o = (16 * cb + i) * TLS + 16 * q + 4 * kg;
                const float4 sv = ldv4(oth_val + o), tv = ldv4(oth_adj + o);
                a0 = mfma4(sv.x, tv.x, a0);
                a1 = mfma4(sv.y, tv.y, a1);
                a0 = mfma4(sv.z, tv.z, a0);
                a1 = mfma4(sv.w, tv.w, a1);
            }
            const floatx4 r = a0 + a1;
            float kept[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (4 * kg + j == i) sm.diag[SIDE][16 * cb + i] = r[j];
                kept[j] = 4 * kg + j < i ? r[j] : 0.0f;
            }
            *reinterpret_cast<float4 *>(pt_lane(sm.pt[SIDE][cb], i, kg)) = make_float4(kept[0], kept[1], kept[2], kept[3]);
        }
        __syncthreads();                         // product tiles are there
        if (!active) return;
        const float *const diag = sm.diag[SIDE];
        float du[4][4];
        IO *const d_adj = (IO *)p.d_q + off;                     // key side only
        scale(S, vec, nbo);
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            if (!FULL && 16 * m >= n_tok) break;
            par::lds_fence();
            const floatx4 st = rows_times(oth_adj, m, S, nbo);
            const float4 pv = ldv4(pt_lane(const_cast<float *>(sm.pt[SIDE][m]), i, kg));
            float vf[4], af[4], xh[4];
            own_tokens(vf, own_val, m);
            own_tokens(af, own_adj, m);
            floatx4 o = st * lo[m];
            o = mfma4(pv.x, vf[0], o);
            o = mfma4(pv.y, vf[1], o);
            o = mfma4(pv.z, vf[2], o);
            o = mfma4(pv.w, vf[3], o);
            const float tot = lo[m] * up[m];
#pragma unroll
            for (int e = 0; e < 4; ++e) xh[e] = vf[e] * up[m];
#pragma unroll
            for (int q = 0; q < 4; ++q) S[q] *= tot;
            add_outer(S, oth_val, m, xh, nbo);
#pragma unroll
            for (int j = 0; j < 4; ++j) du[m][j] = af[j] * o[j];
            if (SIDE == 1) {
                const float4 dg = ldv4(diag + 16 * m + 4 * kg);
                const float dgv[4] = {dg.x, dg.y, dg.z, dg.w};
                float dq[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) dq[j] = pre[m][j] * (o[j] + vf[j] * dgv[j]);
                store4(d_adj, m, dq);
            }
            scale(S, vec + (m + 1) * CH_N, nbo);
        }
        floatx4 G[4];
        {
            const float *const ge = p.gh + item * (CH_N * CH_N);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) G[q][e] = el_ok(q, e) ? ge[st_off(q, e, CH_N)] : 0.0f;
        }
        float carry = 0.0f;                      // rowsum(G_end * S_end), then plus the tokens already visited
        {
            float part = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) part += G[q][e] * S[q][e];
            carry = bwd::row_sums(part).all;
        }
        IO *const d_val = (IO *)(SIDE ? p.d_k : p.d_x) + off, *const d_gate = (IO *)(SIDE ? p.d_f_key : p.d_f) + off;
#pragma unroll
        for (int n = 3; n >= 0; --n) {
            if (!FULL && 16 * n >= n_tok) continue;
            par::lds_fence();
            scale(G, vec + (n + 1) * CH_N, nbo);
            floatx4 x = rows_times(oth_val, n, G, nbo) * up[n];
            float vf[4], af[4], gh[4];
            own_tokens(vf, own_val, n);
            own_tokens(af, own_adj, n);
            const float *const pt = sm.pt[SIDE][n] + (i >> 2) * TLS + 16 * kg + (i & 3);      // (t = 4 kg + e, s = i)
#pragma unroll
            for (int e = 0; e < 4; ++e) x = mfma4(pt[4 * e], af[e], x);
            if (n > 0) {
                const float tot = lo[n] * up[n];
#pragma unroll
                for (int e = 0; e < 4; ++e) gh[e] = af[e] * lo[n];
#pragma unroll
                for (int q = 0; q < 4; ++q) G[q] *= tot;
                add_outer(G, oth_adj, n, gh, nbo);
            }
            const float4 dg = ldv4(diag + 16 * n + 4 * kg);
            const float dgv[4] = {dg.x, dg.y, dg.z, dg.w};
            float dv[4], u[4], inv[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                inv[j] = __builtin_amdgcn_rcpf(pre[n][j]);
                dv[j] = inv[j] * (x[j] + af[j] * dgv[j]);
                u[j] = du[n][j] - vf[j] * x[j];
            }
            store4(d_val, n, dv);
            bwd::reverse_running_sum_swap(u, carry, kg);
            float dgt[4];
            dgt[0] = u[0] * rg0[n];
#pragma unroll
            for (int j = 1; j < 4; ++j) dgt[j] = u[j] * (pre[n][j - 1] * inv[j]);      // 1 / gate
            store4(d_gate, n, dgt);
        }
    }
};

template <typename IO, bool W64, bool FULL>
__device__ __forceinline__ void grads_item(const TileBwdArgs &p, GradSmem &sm, int64_t item, int64_t b, int chunk) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (w < 4)                       // wave-uniform; both sides meet the same two barriers
        GradSide<IO, W64, FULL, 0>(p, sm, item, b, chunk, w, lane).run();
    else
        GradSide<IO, W64, FULL, 1>(p, sm, item, b, chunk, w - 4, lane).run();
}
template <typename IO, bool W64> __global__ __launch_bounds__(TB_THREADS, 4) void lfw_tile_grads_kernel(TileBwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    GradSmem &sm = *reinterpret_cast<GradSmem *>(smem);
    const int64_t item = blockIdx.x, b = item / p.NC;
    const int chunk = (int)(item - b * p.NC);
    if ((chunk + 1) * TILE_CHUNK <= (int)p.T)
        grads_item<IO, W64, true>(p, sm, item, b, chunk);
    else
        grads_item<IO, W64, false>(p, sm, item, b, chunk);
}

// ---- launch 4 -------------------------------------------------------------------------------------
// Work items are (listed chunk, side, tile of 16 state rows); the grid is bounded and walks over them.  base: what all
// of them have in common (filled by the host, which keeps the body's loops as they are in the plain kernel).
constexpr int TE_GRID = 1024;
template <typename IO> __global__ __launch_bounds__(SCAN_THREADS) void lfw_tile_exact_kernel(TileBwdArgs p, ScanBwdArgs base) {
    const int nd = ((int)p.D + 15) / 16, nk = ((int)p.K + 15) / 16, per = nd + nk;
    const int64_t total = (int64_t)p.list[0] * per;
    for (int64_t idx = blockIdx.x; idx < total; idx += gridDim.x) {
        const int64_t item = p.list[1 + idx / per];
        const int tile = (int)(idx % per);
        const int64_t b = item / p.NC;
        const int chunk = (int)(item - b * p.NC);
        const int64_t line = row_first_token(b, p.T, p.heads) + (int64_t)(chunk * TILE_CHUNK) * p.heads;
        ScanBwdArgs a = base;
        a.x = (const IO *)p.x + line * p.D; a.f = (const IO *)p.f + line * p.D; a.g_out = (const IO *)p.g_out + line * p.D;
        a.q = (const IO *)p.q + line * p.K; a.k = (const IO *)p.k + line * p.K; a.f_key = (const IO *)p.f_key + line * p.K;
        a.ckpt = (const IO *)p.ckpt + item * ((int64_t)p.D * p.K);
        a.d_x = (IO *)p.d_x + line * p.D; a.d_f = (IO *)p.d_f + line * p.D;
        a.d_q = (IO *)p.d_q + line * p.K; a.d_k = (IO *)p.d_k + line * p.K; a.d_f_key = (IO *)p.d_f_key + line * p.K;
        a.g_end = p.gh + item * (CH_N * CH_N);
        a.T = min((int64_t)TILE_CHUNK, p.T - (int64_t)chunk * TILE_CHUNK);
        __syncthreads();                         // the item before no longer reads the LDS
        if (tile < nd)
            scan::bwd_scan_body_kg<IO, 4, 0, 16, 1>(a, 0, tile);
        else
            scan::bwd_scan_body_kg<IO, 4, 1, 16, 1>(a, 0, tile - nd);
    }
}

template <typename IO, bool W64> int launch(const TileBwdArgs &a, hipStream_t stream) {
    auto incr = lfw_tile_incr_kernel<IO, W64>;
    auto scan = lfw_tile_scan_kernel<IO, W64>;
    auto grads = lfw_tile_grads_kernel<IO, W64>;
    auto exact = lfw_tile_exact_kernel<IO>;
    int rc = enable_lds(reinterpret_cast<const void *>(grads), (int)sizeof(GradSmem), "hipFuncSetAttribute(tile gradient kernel)");
    if (rc) return rc;
    const int64_t items = a.B * a.NC;
    if (items > 0x0fffffffLL) return fail(T2FW_ERR_UNSUPPORTED, "B * chunks = %lld is too large", (long long)items);
    hipLaunchKernelGGL(incr, dim3((unsigned)items), dim3(TB_THREADS), 0, stream, a);
    if ((rc = check_hip(hipGetLastError(), "lfw_tile_incr_kernel launch"))) return rc;
    hipLaunchKernelGGL(scan, dim3((unsigned)(4 * a.B)), dim3(TS_THREADS), 0, stream, a);
    if ((rc = check_hip(hipGetLastError(), "lfw_tile_scan_kernel launch"))) return rc;
    hipLaunchKernelGGL(grads, dim3((unsigned)items), dim3(TB_THREADS), sizeof(GradSmem), stream, a);
    if ((rc = check_hip(hipGetLastError(), "lfw_tile_grads_kernel launch"))) return rc;
    const int per = (a.D + 15) / 16 + (a.K + 15) / 16;
    const int64_t grid = std::min<int64_t>(items * per, TE_GRID);
    const size_t smem = scan_bwd_lds_bytes(scan::SegLen<4>::value, 16, 4, 16, TILE_CHUNK, true);
    ScanBwdArgs base{};
    base.B = 1; base.NC = 1; base.D = a.D; base.K = a.K; base.C = TILE_CHUNK; base.heads = a.heads;
    base.kg = 16; base.use_sub = 1;
    hipLaunchKernelGGL(exact, dim3((unsigned)grid), dim3(SCAN_THREADS), smem, stream, a, base);
    return check_hip(hipGetLastError(), "lfw_tile_exact_kernel launch");
}

}  // namespace

int tile_backward(const TileBwdArgs &a, int dtype, hipStream_t stream) {
    const bool w64 = a.D == CH_N && a.K == CH_N;
    switch (dtype) {
        case T2FW_F32: return w64 ? launch<float, true>(a, stream) : launch<float, false>(a, stream);
        case T2FW_F16: return launch<__half, false>(a, stream);
        case T2FW_BF16: return launch<__hip_bfloat16, false>(a, stream);
    }
    return fail(T2FW_ERR_UNSUPPORTED, "the tile kernels take fp32, fp16 or bf16 tensors");
}

}  // namespace t2fw
