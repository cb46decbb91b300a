// Chunks of the exact recurrence (launch 3 of lfw_xpar.hip) on fp64 matrix instructions: fp32 tensors, 64 x 64 states.
//
// With the gate products from the chunk's first token, a_t[d] = f_0 .. f_t on the value side and b_t[k] on the key side,
//   xt_t = x_t / a_t    gs_t = g_t a_t    kt_t = k_t / b_t    qs_t = q_t b_t    P[t,s] = qs_t . kt_s    W[t,s] = gs_t . xt_s
// a chunk of 64 steps is a set of products with the state S0 before it and the adjoint G_end after it:
//   forward   o_t = a_t ( S0 qs_t + sum_{s<=t} P[t,s] xt_s )
//   backward  Gh = (a_63 (x) b_63) G_end,  o'_t = S0 qs_t + sum_{s<t} P[t,s] xt_s,  x'_t = Gh kt_t + sum_{r>t} P[r,t] gs_r
//             d_x_t = (x'_t + gs_t P[t,t]) / a_t;  d_k_t, d_q_t likewise from W (q', k': the two sides exchanged)
//             f_t d_f_t = beta - sum_{r<t} (gs_r o'_r - xt_r x'_r),  beta = rowsum(Gh * S0) + sum_t gs_t (S0 qs_t)
//
// Precision.  What tokens share with tokens is fp64, but for P and W, which are rounded to fp32 once.  What they share with
// S0 and G_end (Gh kt_t as a_63 times G_end with k_t times the gates after t) is an fp32 product in chains of 16 terms.  The
// running sum of the gate gradients cancels, but only against itself: P's terms from the same P in fp64, the states' from
// the same fp32 values, which enter beta and leave it again.  What is left of the cancellation is fp64 rounding of the LARGEST
// term so far, measured 2^-50 of it; a value that the gates have forgotten, a token whose gates are small on both sides or
// the end of the loss make the sum itself far smaller than that term.  MM_CANCELLED draws the line: a token of which less than
// 2^-26 of the largest term is left ends the chunk's use of these products, so that the remainder stays below 2^-24 of every
// gate gradient that is kept.  The measure of a token is the larger of f_t d_f_t and its own output's share of it, gs_t o'_t:
// the sum over the other side's channels may vanish by chance, both rarely do (no chunk of 600 with normal gates).
//
// Range: gates in [XP_MM_MIN_GATE, 1] with a product of at least MM_MIN_PRODUCT over the chunk: products of two scaled operands
// stay below 2^866 and factors of both sides above 2^-800.  Inputs, states and adjoints of at most MM_MAX_VALUE: where gate
// products make P or an operand of the states underflow fp32, 2^-150 is lost, times a value or an element of a state.  At 2^30
// that is 2^-24 of results of 2^-96 (with a limit of 2^58, values of 2^40 and queries and keys of 2^-50 gave outputs of 2^-95 that were wrong
// altogether).  Chunks outside it run step by step (lfw_xpar64.hip); launch 1 sees single gates, this
// workgroup the rest when it scales its operands, and the cancellation when it has the gradients.
//
// Lane layout: v_mfma_f64_16x16x4_f64 takes A[i][kg] and B[kg][i] in lane (i = lane & 15, kg = lane >> 4) and returns
// rows 4 j + kg of column i.  The rows of A are handed over in the order mm_row(i), which makes those rows 4 kg + j.
// A wave owns 16 channels of one side ("own"), its lane channel 16 cb + i and tokens 16 m + 4 kg + j: they are the B operand
// of what contracts over tokens, and a slab of the state (own channel, other side's channels 16 q + 4 kg + e) is the B
// operand of what contracts over the other side's channels.  That side's operands come from LDS, token-major fp64.
#pragma once

#include "lfw_chunk.hpp"
#include "lfw_xpar.hpp"

namespace t2fw {
namespace mm {

typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int MM_LS = 66;                          // row stride, in doubles, of the token-major operands [64][MM_LS]
constexpr int MM_FS = 68;                          // row stride, in floats, of the fp32 operands [64][MM_FS]
constexpr int MM_PS = 68;                          // a 16 x 16 product tile: element (t, s) at (s / 4) MM_PS + 4 t + s % 4
constexpr float MM_MIN_GATE = XP_MM_MIN_GATE;
constexpr double MM_MIN_PRODUCT = 0x1p-400;
constexpr float MM_MAX_VALUE = 0x1p30f;
constexpr unsigned MM_CANCELLED = 26u << 20;       // in the high word of a double: a factor of 2^26

struct Smem {
    // other side's kt / xt and qs / gs; after the products of tokens with tokens, adj [and backward val] make room for what is
    // multiplied with the states, in fp32 (state_operands)
    double val[XP_CHUNK * MM_LS], adj[XP_CHUNK * MM_LS];
    double tot[XP_N];                              // other side's gate products over the chunk
    float pt[10][4 * MM_PS];                       // product tiles (m, n), n <= m, at m (m + 1) / 2 + n
    float diag[XP_CHUNK];
    int bad[4];
};
static_assert(2 * ((sizeof(Smem) + 1279) / 1280 * 1280) <= 160 * 1024, "two workgroups must fit the LDS of one CU");

// Nothing moves across: keeps stages apart whose operands would not fit the registers all at once.
__device__ __forceinline__ void fence() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// What has been seen of the gates (as bits) and the inputs (sum of magnitudes: inf and NaN show, too).
// Launch 1 has sent chunks with a gate out of range elsewhere, so the gates' part always passes; without it the backward kernel
// keeps its gates longer and spills 36 registers in the place of 28 (96 x 1024 steps, both directions: 286.2 us for 284.5).
struct Seen {
    unsigned gate = 0;
    float inputs = 0.0f;
    __device__ __forceinline__ bool out_of_range() const {
        return gate > __float_as_uint(1.0f) - __float_as_uint(MM_MIN_GATE) || !(inputs <= MM_MAX_VALUE);
    }
};
// ... and the verdict on what has been looked at so far is taken, not put off with all values kept
__device__ __forceinline__ void fence(Seen &seen) {
    asm volatile("" : "+v"(seen.gate), "+v"(seen.inputs)::"memory");
    __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ int mm_row(int i) { return 4 * (i & 3) + (i >> 2); }
__device__ __forceinline__ doublex4 mfma(double a, double b, doublex4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4 ldv4(const float *p) { return *reinterpret_cast<const float4 *>(p); }
__device__ __forceinline__ constexpr int pt_index(int m, int n) { return m * (m + 1) / 2 + n; }

// Magnitudes are compared by their high words.
__device__ __forceinline__ unsigned magnitude(double v) {
    return (unsigned)((unsigned long long)__double_as_longlong(v) >> 32) & 0x7fffffffu;
}
// {value of the even row of 16 lanes of each pair, of the odd one}, {of rows 0-1, of rows 2-3} (v the same in both rows)
struct Pair { double a, b; };
__device__ __forceinline__ double words(unsigned lo, unsigned hi) {
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ Pair rows16(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)u, (unsigned)u, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    return {words(lo[0], hi[0]), words(lo[1], hi[1])};
}
__device__ __forceinline__ Pair rows32(double v) {
    const unsigned long long u = (unsigned long long)__double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)u, (unsigned)u, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(u >> 32), (unsigned)(u >> 32), false, false);
    return {words(lo[0], hi[0]), words(lo[1], hi[1])};
}
struct PairU { unsigned a, b; };
__device__ __forceinline__ PairU rows16(unsigned v) {
    const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    return {s[0], s[1]};
}
__device__ __forceinline__ PairU rows32(unsigned v) {
    const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return {s[0], s[1]};
}
__device__ __forceinline__ double reciprocal(double v) {
    const double r = __builtin_amdgcn_rcp(v);
    return fma(r, fma(-v, r, 1.0), r);
}

// One side's view of a chunk: lane (i, kg) of wave cb owns channel c = 16 cb + i and tokens 16 m + 4 kg + j.
template <bool FULL> struct Lane {
    int i, kg, c, n_left;                          // n_left: tokens from the lane's first one to the end of the sequence
    int64_t ts;                                    // bytes from a token to the next
    unsigned off;
    __device__ __forceinline__ Lane(int cb, int lane, int n_tok, int heads) : ts((int64_t)heads * (XP_N * 4)) {
        i = lane & 15; kg = lane >> 4; c = 16 * cb + i;
        n_left = n_tok - 4 * kg;
        off = (unsigned)(4 * kg) * (unsigned)ts + 4u * (unsigned)c;
    }
    __device__ __forceinline__ bool ok(int m, int j) const { return FULL || 16 * m + j < n_left; }
    // tokens past the end are read from the last one and replaced by `pad`
    __device__ __forceinline__ void load(float (&r)[4][4], const float *base, float pad) const {
        const char *const p = reinterpret_cast<const char *>(base);
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (FULL)
                    r[m][j] = *reinterpret_cast<const float *>((p + (16 * m + j) * ts) + off);
                else                               // the offset may be negative: the lane starts past the end
                    r[m][j] = *reinterpret_cast<const float *>(p + ((int64_t)off + min(16 * m + j, n_left - 1) * ts));
            }
        if (!FULL) {
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int j = 0; j < 4; ++j) r[m][j] = ok(m, j) ? r[m][j] : pad;
        }
    }
    __device__ __forceinline__ void store(float *base, int m, const float (&v)[4]) const {
        char *const p = reinterpret_cast<char *>(base);
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (ok(m, j)) *reinterpret_cast<float *>((p + (16 * m + j) * ts) + off) = v[j];
    }
};

// the four products (reciprocals) of a tile again, from the first (last) of them
__device__ __forceinline__ void products(double (&pre)[4], double first, const float (&g)[4]) {
    pre[0] = first;
#pragma unroll
    for (int j = 1; j < 4; ++j) pre[j] = pre[j - 1] * g[j];
}
__device__ __forceinline__ void reciprocals(double (&inv)[4], double last, const float (&g)[4]) {
    inv[3] = last;
#pragma unroll
    for (int j = 2; j >= 0; --j) inv[j] = inv[j + 1] * g[j + 1];
}
// Products from the chunk's start up to and with the lane's four tokens of a tile, and their reciprocals; carry: the
// product of the tiles before.
struct Scales { double pre[4], inv[4]; };
__device__ __forceinline__ Scales tile_scales(const float (&g)[4], int kg, double &carry, Seen &seen) {
    Scales s;
#pragma unroll
    for (int j = 0; j < 4; ++j) seen.gate = max(seen.gate, __float_as_uint(g[j]) - __float_as_uint(MM_MIN_GATE));
    const double own = ((double)g[0] * g[1]) * ((double)g[2] * g[3]);
    const Pair r = rows16(own), h = rows32(r.a * r.b);
    products(s.pre, carry * (((kg & 2) ? h.a : 1.0) * ((kg & 1) ? r.a : 1.0)) * g[0], g);
    carry *= h.a * h.b;
    reciprocals(s.inv, reciprocal(s.pre[3]), g);
    return s;
}
__device__ __forceinline__ double operand(float raw, double scale, Seen &seen) {
    seen.inputs += fabsf(raw);
    return raw * scale;
}

// The other side's operands of the wave's channels -> LDS.  qf: the lane's qs / gs in fp32; kf (SUFFIX): its values times the
// gates that follow them in the chunk.  Both are what multiplies a state: no factor is above one.
template <bool FULL, bool SUFFIX>
__device__ __forceinline__ bool stage_other(Smem &sm, const Lane<FULL> &ln, const float (&g)[4][4], const float (&v)[4][4], const float (&a)[4][4],
                                            float (&qf)[4][4], float (&kf)[4][4], Seen &seen) {
    double carry = 1.0, kept[4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        fence(seen);
        const Scales s = tile_scales(g[m], ln.kg, carry, seen);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int o = (16 * m + 4 * ln.kg + j) * MM_LS + ln.c;
            const double kt = operand(v[m][j], s.inv[j], seen), qs = operand(a[m][j], s.pre[j], seen);
            sm.val[o] = kt;
            sm.adj[o] = qs;
            qf[m][j] = (float)qs;
            if (SUFFIX) kept[m][j] = kt;
        }
    }
    if (SUFFIX) {
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
            for (int j = 0; j < 4; ++j) kf[m][j] = (float)(kept[m][j] * carry);
    }
    if (ln.kg == 0) sm.tot[ln.c] = carry;
    fence(seen);
    return !(carry >= MM_MIN_PRODUCT);
}

// The wave's share of the ten product tiles (m, n): (t, s) for s < t (INCL: s <= t) of the diagonal ones, whose diagonal
// goes to sm.diag.  Waves 0 to 3 take (3, n); then (2, 0) (2, 1) (2, 2) (1, 1); then (1, 0) and (0, 0).
template <bool INCL> __device__ __forceinline__ void product_tiles(Smem &sm, int w, int i, int kg, int n_tok) {
#pragma unroll 1
    for (int round = 0; round < 3; ++round) {
        int m = 3 - round, n = w;
        if (round == 1 && w == 3) { m = 1; n = 1; }
        if (round == 2) { m = 1 - w; n = 0; }
        if (m < 0) break;
        if (16 * m >= n_tok) continue;
        const double *const vp = sm.val + (16 * n + mm_row(i)) * MM_LS + 4 * kg, *const ap = sm.adj + (16 * m + i) * MM_LS + 4 * kg;
        doublex4 a0 = {0., 0., 0., 0.}, a1 = a0;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                a0 = mfma(vp[16 * q + e], ap[16 * q + e], a0);
                a1 = mfma(vp[16 * q + e + 1], ap[16 * q + e + 1], a1);
            }
        float kept[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float r = (float)(a0[j] + a1[j]);
            const int s = 4 * kg + j;
            if (!INCL && m == n && s == i) sm.diag[16 * m + i] = r;
            kept[j] = (m > n || (INCL ? s <= i : s < i)) ? r : 0.0f;
        }
        *reinterpret_cast<float4 *>(sm.pt[pt_index(m, n)] + kg * MM_PS + 4 * i) = make_float4(kept[0], kept[1], kept[2], kept[3]);
    }
}

// fp32 operands into the place of fp64 ones that all waves are done with
__device__ __forceinline__ float *state_operands(double *place) { return reinterpret_cast<float *>(place); }
template <bool FULL> __device__ __forceinline__ void store_operands(float *tile, const Lane<FULL> &ln, const float (&v)[4][4]) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) tile[(16 * m + 4 * ln.kg + j) * MM_FS + ln.c] = v[m][j];
}
// rows of tokens of tile m of an fp32 operand times a slab of the state: v_mfma_f32_16x16x4_f32, half the time of the
// fp64 form, whose rows come back as 4 kg + j.  Chains of 16 terms; nothing that cancels is made of these sums.
__device__ __forceinline__ doublex4 rows_times(const float *tile, int m, const float (&X)[4][4], int i, int kg) {
    const float *const p = tile + (16 * m + i) * MM_FS + 4 * kg;
    floatx4 acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 v = ldv4(p + 16 * q);
        const float av[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            acc[e] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], X[q][e], q ? acc[e] : floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    }
    const floatx4 sum = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    doublex4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = sum[j];
    return o;
}
// o + P[m, n] w  (own tokens w of tile n)
__device__ __forceinline__ doublex4 product_times(const Smem &sm, int m, int n, const double (&w)[4], doublex4 o, int i, int kg) {
    const float4 pv = ldv4(sm.pt[pt_index(m, n)] + kg * MM_PS + 4 * mm_row(i));
    o = mfma(pv.x, w[0], o);
    o = mfma(pv.y, w[1], o);
    o = mfma(pv.z, w[2], o);
    return mfma(pv.w, w[3], o);
}
// x + P[m, n]^T w  (own tokens w of tile m)
__device__ __forceinline__ doublex4 product_transposed_times(const Smem &sm, int m, int n, const double (&w)[4], doublex4 x, int i, int kg) {
    const float *const pt = sm.pt[pt_index(m, n)] + (i & 3) * MM_PS + 16 * kg + (i >> 2);      // (t = 4 kg + e, s = mm_row(i))
#pragma unroll
    for (int e = 0; e < 4; ++e) x = mfma(pt[4 * e], w[e], x);
    return x;
}
// X += sum over the chunk's tokens of (other side's operand) (x) (own tokens w), then times the chunk's products
template <typename F, int STRIDE>
__device__ __forceinline__ void add_outer(doublex4 (&X)[4], const F *operand, const double (&w)[4][4], int i, int kg) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int q = 0; q < 4; ++q) X[q] = mfma(operand[(16 * m + 4 * kg + e) * STRIDE + 16 * q + mm_row(i)], w[m][e], X[q]);
}
__device__ __forceinline__ void scale(doublex4 (&X)[4], const double *tot, double own, int kg) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) X[q][e] *= tot[16 * q + 4 * kg + e] * own;
}
// element (own channel c, other side's channel 16 q + 4 kg + e) of a [64][64] state; SIDE 0: own channels are its rows
template <int SIDE> __device__ __forceinline__ void load_slab(float (&X)[4][4], const float *st, int c, int kg) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int o = 16 * q + 4 * kg + e;
            X[q][e] = st[(unsigned)(SIDE ? o * XP_N + c : c * XP_N + o)];
        }
}
__device__ __forceinline__ void widen(doublex4 (&X)[4], const float (&raw)[4][4]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) X[q][e] = raw[q][e];
}
__device__ __forceinline__ void store_slab(float *st, const doublex4 (&X)[4], int c, int kg) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) st[(unsigned)(c * XP_N + 16 * q + 4 * kg + e)] = (float)X[q][e];
}

// Verdict of the four waves; a barrier after which the operands are there, too
__device__ __forceinline__ bool any_bad(Smem &sm, int w, int lane, bool bad) {
    const int any = __any((int)bad);
    if (lane == 0) sm.bad[w] = any;
    __syncthreads();
    return __builtin_amdgcn_readfirstlane(sm.bad[0] | sm.bad[1] | sm.bad[2] | sm.bad[3]) != 0;
}

// fp32: the state entering a chunk is its checkpoint, where those are asked for
__device__ __forceinline__ const float *entering_state(const XparFwdArgs &p, int64_t item) {
    return (p.ckpt != nullptr ? (const float *)p.ckpt : p.ws.states) + item * (XP_N * XP_N);
}

// false: the chunk is out of range, nothing has been stored
template <bool FULL> __device__ __forceinline__ bool forward_chunk(const XparFwdArgs &p, Smem &sm, int64_t b, int chunk) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t line0 = uniform64(row_first_token(b, p.T, p.heads) + (int64_t)chunk * XP_CHUNK * p.heads) * XP_N;
    const int n_tok = FULL ? XP_CHUNK : (int)p.T - chunk * XP_CHUNK;
    const Lane<FULL> ln(w, lane, n_tok, p.heads);
    const int i = ln.i, kg = ln.kg;
    Seen seen;
    float og[4][4], ov[4][4], oa[4][4], g[4][4], v[4][4], s0[4][4];
    ln.load(og, (const float *)p.f_key + line0, 1.0f);
    ln.load(ov, (const float *)p.k + line0, 0.0f);
    ln.load(oa, (const float *)p.q + line0, 0.0f);
    ln.load(g, (const float *)p.f + line0, 1.0f);
    ln.load(v, (const float *)p.x + line0, 0.0f);
    load_slab<0>(s0, entering_state(p, b * p.NC + chunk), ln.c, kg);
    float qf[4][4], unused[4][4];
    bool bad = stage_other<FULL, false>(sm, ln, og, ov, oa, qf, unused, seen);
    double xt[4][4], first[4], carry = 1.0;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        fence(seen);
        const Scales s = tile_scales(g[m], kg, carry, seen);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            xt[m][j] = operand(v[m][j], s.inv[j], seen);
        }
        first[m] = s.pre[0];
    }
    float states = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) states += fabsf(s0[q][e]);
    bad |= seen.out_of_range() || !(carry >= MM_MIN_PRODUCT) || !(states <= MM_MAX_VALUE);
    if (any_bad(sm, w, lane, bad)) return false;
    product_tiles<true>(sm, w, i, kg, n_tok);
    __syncthreads();
    float *const qs = state_operands(sm.adj);
    store_operands(qs, ln, qf);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        if (!FULL && 16 * m >= n_tok) break;
        fence();
        doublex4 o = rows_times(qs, m, s0, i, kg);
#pragma unroll
        for (int n = 0; n <= m; ++n) o = product_times(sm, m, n, xt[n], o, i, kg);
        double pre[4];
        products(pre, first[m], g[m]);
        float r[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) r[j] = (float)(o[j] * pre[j]);
        ln.store((float *)p.out + line0, m, r);
    }
    if (chunk == (int)p.NC - 1) {
        doublex4 S[4];
        widen(S, s0);
        add_outer<double, MM_LS>(S, sm.val, xt, i, kg);
        scale(S, sm.tot, carry, kg);
        store_slab((float *)p.next_state + b * (XP_N * XP_N), S, ln.c, kg);
    }
    return true;
}

// false: the chunk is out of range, or its gate gradients have cancelled; results that have been stored are no good
template <int SIDE, bool FULL> __device__ __forceinline__ bool backward_chunk(const XparBwdArgs &p, Smem &sm, int64_t b, int chunk) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int64_t line0 = uniform64(row_first_token(b, p.T, p.heads) + (int64_t)chunk * XP_CHUNK * p.heads) * XP_N;
    const int n_tok = FULL ? XP_CHUNK : (int)p.T - chunk * XP_CHUNK;
    const Lane<FULL> ln(w, lane, n_tok, p.heads);
    const int i = ln.i, kg = ln.kg;
    const int64_t state = (b * p.NC + chunk) * (XP_N * XP_N);
    Seen seen;
    float og[4][4], ov[4][4], oa[4][4], g[4][4], rv[4][4], ra[4][4], s0[4][4], g_end[4][4];
    ln.load(og, (const float *)(SIDE ? p.f : p.f_key) + line0, 1.0f);
    ln.load(ov, (const float *)(SIDE ? p.x : p.k) + line0, 0.0f);
    ln.load(oa, (const float *)(SIDE ? p.g_out : p.q) + line0, 0.0f);
    ln.load(g, (const float *)(SIDE ? p.f_key : p.f) + line0, 1.0f);
    ln.load(rv, (const float *)(SIDE ? p.k : p.x) + line0, 0.0f);
    ln.load(ra, (const float *)(SIDE ? p.q : p.g_out) + line0, 0.0f);
    load_slab<SIDE>(s0, (const float *)p.ckpt + state, ln.c, kg);
    load_slab<SIDE>(g_end, p.ws.states + state, ln.c, kg);
    float qf[4][4], kf[4][4];
    bool bad = stage_other<FULL, true>(sm, ln, og, ov, oa, qf, kf, seen);
    double v[4][4], a[4][4], first[4], last[4], tot = 1.0;
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        fence(seen);
        const Scales s = tile_scales(g[m], kg, tot, seen);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            v[m][j] = operand(rv[m][j], s.inv[j], seen);
            a[m][j] = operand(ra[m][j], s.pre[j], seen);
        }
        first[m] = s.pre[0];
        last[m] = s.inv[3];
    }
    float states = 0.0f;
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 4; ++e) states += fabsf(s0[q][e]) + fabsf(g_end[q][e]);
    bad |= seen.out_of_range() || !(tot >= MM_MIN_PRODUCT) || !(states <= MM_MAX_VALUE);
    if (any_bad(sm, w, lane, bad)) return false;
    product_tiles<false>(sm, w, i, kg, n_tok);
    __syncthreads();
    float *const qs = state_operands(sm.adj), *const ks = state_operands(sm.val);
    store_operands(qs, ln, qf);
    store_operands(ks, ln, kf);
    __syncthreads();
    double du[4][4], beta = 0.0;
    unsigned largest = 0;                          // of the terms of the gate gradients' running sum so far
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        if (!FULL && 16 * m >= n_tok) break;
        fence();
        doublex4 o = rows_times(qs, m, s0, i, kg);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            beta = fma(a[m][j], o[j], beta);
            largest = max(largest, magnitude(beta));
        }
#pragma unroll
        for (int n = 0; n <= m; ++n) o = product_times(sm, m, n, v[n], o, i, kg);
#pragma unroll
        for (int j = 0; j < 4; ++j) du[m][j] = a[m][j] * o[j];
        if (SIDE == 1) {
            const float4 dg = ldv4(sm.diag + 16 * m + 4 * kg);
            const float dgv[4] = {dg.x, dg.y, dg.z, dg.w};
            double pre[4];
            products(pre, first[m], g[m]);
            float dq[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) dq[j] = (float)(fma(v[m][j], (double)dgv[j], o[j]) * pre[j]);
            ln.store((float *)p.d_q + line0, m, dq);
        }
    }
    fence();
    {
        double part = 0.0;                         // rowsum(Gh * S0)
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) part = fma((double)g_end[q][e] * s0[q][e], sm.tot[16 * q + 4 * kg + e], part);
        beta = fma(part, tot, beta);
        const Pair r = rows16(beta), h = rows32(r.a + r.b);
        beta = h.a + h.b;                          // gate gradient of the tile's first token, times its gate
        const PairU lr = rows16(largest), lh = rows32(max(lr.a, lr.b));
        largest = max(max(lh.a, lh.b), magnitude(beta));
    }
    bad = false;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        if (!FULL && 16 * n >= n_tok) break;
        fence();
        doublex4 x = rows_times(ks, n, g_end, i, kg) * tot;
#pragma unroll
        for (int m = n; m < 4; ++m)
            if (FULL || 16 * m < n_tok) x = product_transposed_times(sm, m, n, a[m], x, i, kg);
        const float4 dg = ldv4(sm.diag + 16 * n + 4 * kg);
        const float dgv[4] = {dg.x, dg.y, dg.z, dg.w};
        double inv[4];
        reciprocals(inv, last[n], g[n]);
        float dv[4], dgt[4];
        double u[4];                               // what is gone after the lane's tokens up to and with the j-th
        unsigned terms[4];                         // largest of those
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            dv[j] = (float)(fma(a[n][j], (double)dgv[j], x[j]) * inv[j]);
            u[j] = fma(-v[n][j], x[j], du[n][j]);
            terms[j] = max(magnitude(du[n][j]), magnitude(u[j]));
            if (j > 0) {
                u[j] += u[j - 1];
                terms[j] = max(terms[j], terms[j - 1]);
            }
        }
        ln.store((float *)(SIDE ? p.d_k : p.d_x) + line0, n, dv);
        const Pair r = rows16(u[3]), h = rows32(r.a + r.b);
        const double first = beta - (((kg & 2) ? h.a : 0.0) + ((kg & 1) ? r.a : 0.0));
        beta -= h.a + h.b;
        const PairU lr = rows16(terms[3]), lh = rows32(max(lr.a, lr.b));
        const unsigned before = max(max(largest, (kg & 2) ? lh.a : 0u), (kg & 1) ? lr.a : 0u);
        largest = max(largest, max(lh.a, lh.b));
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const double left = j ? first - u[j - 1] : first;
            dgt[j] = (float)(left * reciprocal(g[n][j]));
            const bool lost = max(magnitude(left), magnitude(du[n][j])) + MM_CANCELLED < (j ? max(before, terms[j - 1]) : before);
            bad |= lost && ln.ok(n, j);
        }
        ln.store((float *)(SIDE ? p.d_f_key : p.d_f) + line0, n, dgt);
    }
    if (SIDE == 0 && chunk == 0) {
        doublex4 G[4];
        widen(G, g_end);
        scale(G, sm.tot, tot, kg);
        add_outer<float, MM_FS>(G, qs, a, i, kg);
        store_slab((float *)p.d_s0 + b * (XP_N * XP_N), G, ln.c, kg);
    }
    return !any_bad(sm, w, lane, bad);
}

}  // namespace mm
}  // namespace t2fw
