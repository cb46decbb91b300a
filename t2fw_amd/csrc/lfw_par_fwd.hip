// Forward pass with the chunks of a row side by side, D = K = 64, fp16 / bf16 (algebra, lane layout and helpers: lfw_par.hpp): for
// few rows of many steps, where the sequential kernel (lfw_chunk_fwd.hip) is a chain of 1.4 us per 64 tokens on a chip that is
// nearly empty.  Chunks of 64 tokens, four launches:
//   1  what a chunk adds to the state, M = sum_t xh_t (x) kh_t with xh, kh = x, k times the gates after t (factors of at most
//      one), and the chunk's gate products; one workgroup per (row, chunk)
//   2  the chain over a row's chunks, elementwise in fp32: S <- (tot_a (x) tot_b) S + M.  Leaves the state before each chunk,
//      scaled on the key side to the chunk's middle, as the bf16 operand that launch 3 reads, the checkpoints and the final state
//   3  o_t = a_t ( S0 qs_t + sum_{s <= t} P[t,s] xt_s ), one workgroup per (row, chunk)
//   4  the sequential kernel on the rows that this form cannot take (lfw_par.hpp: half a chunk's gate products below 2^-80, a gate
//      outside [0, 1]) or that have a result that is not finite (a NaN would reach the other tokens of its chunk); a workgroup of any other row reads its verdict and leaves
// Precision: bf16 operands, fp32 sums, increments and states (the chain's M and S are never rounded to 16 bits, the operand made
// of S is), gates below 2^-24 count as 2^-24, all as in the sequential kernel.  Three things keep the error at or below that
// kernel's, whose blocks are of 16 tokens.  A block's last token enters its increment without a rounding, which of 64 tokens is
// rarer: the xh come as two terms, head and remainder, and so do the P.  The state is scaled by powers of two, which rounds
// nothing (an initial state of bf16 stays what it is).  And the value side's share of that scale is applied to the product,
// in fp32: both sides' on the operand come to 2^-160, under which states of 1e-3 and less lost bits to the type's range.
// Error of the outputs against float64, bf16, sequential / here: 12 rows x 1000 steps 3.67e-3 / 3.30e-3, what is left of a state of
// 1e-5 under gates of 0.185 on both sides 2.24e-3 / 2.24e-3; without the three 3.68e-3 and 1.04e-2.  They cost 32 x 2050 0.8 us
// of 34.5 and the smaller calls nothing that shows.
//
// The reference's forward is one thread per state element and a loop over time (t2fw/csrc/lfw_kernel.cu:18-59).
#include "common.hpp"
#include "lfw_par.hpp"

namespace t2fw {
namespace {

using namespace par;

constexpr int PF_NT = 4, PF_CL = 16 * PF_NT;

// Product of the rows above this lane's row (identity for the last) and of all four
__device__ __forceinline__ RowScan row_scan_mul_above(float v, int kg) {
    const u32 vb = __float_as_uint(v);
    const auto s16 = __builtin_amdgcn_permlane16_swap(vb, vb, false, false);     // {even row of the pair, odd row}
    const float od = __uint_as_float(s16[1]);
    const float pair = __uint_as_float(s16[0]) * od;
    const u32 pb = __float_as_uint(pair);
    const auto s32 = __builtin_amdgcn_permlane32_swap(pb, pb, false, false);     // {rows 0-1, rows 2-3}
    const float hi = __uint_as_float(s32[1]);
    RowScan r;
    r.all = __uint_as_float(s32[0]) * hi;
    r.lower = ((kg & 1) ? 1.0f : od) * ((kg & 2) ? 1.0f : hi);
    return r;
}

// ---- launch 1: per-chunk increments and gate products ------------------------------------------------
constexpr int PF_INCR_SMEM = 3 * CM_BYTES;                // XH, KH, remainders of XH

template <typename IOE, bool HEADS> __global__ __launch_bounds__(PAR_THREADS) void lfw_par_fwd_incr_kernel(ParFwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NT = PF_NT, CL = PF_CL;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), l = tid & 63;
    const int side = w >> 2, cb = w & 3, i = l & 15, kg = l >> 4, c = 16 * cb + i;
    const int NC = (int)p.NC, T = (int)p.T;
    const int item = (int)blockIdx.x;
    const int64_t b = item / NC;
    const int chunk = item - (int)b * NC;
    const u32 ts = HEADS ? (u32)p.heads * CH_N : (u32)CH_N;
    const int n_left = T - (chunk * CL + 4 * kg);
    const int64_t chunk_off = wave_uniform(row_first_token(b, p.T, HEADS ? p.heads : 1) * CH_N + (int64_t)(chunk * CL) * ts);
    const u32 lane_off = (u32)(4 * kg) * ts + (u32)c;
    const u16 *const gate = reinterpret_cast<const u16 *>(side ? p.f_key : p.f) + chunk_off;
    const u16 *const val = reinterpret_cast<const u16 *>(side ? p.k : p.x) + chunk_off;
    RawTokens<NT> rg, rv;
    LaneChunk<NT> lc;
    float gt[NT][4], v[NT][4], after[NT][4];
    if (chunk * CL + CL <= T) {
        load_tokens<NT, true>(rg, gate, lane_off, ts, n_left);
        load_tokens<NT, true>(rv, val, lane_off, ts, n_left);
        gate_scan<IOE, NT, true, false, IOE::FLOOR_BITS>(lc, gt, rg, kg, n_left);
        to_floats<IOE, NT, true>(v, rv, n_left);
    } else {
        load_tokens<NT, false>(rg, gate, lane_off, ts, n_left);
        load_tokens<NT, false>(rv, val, lane_off, ts, n_left);
        gate_scan<IOE, NT, false, false, IOE::FLOOR_BITS>(lc, gt, rg, kg, n_left);
        to_floats<IOE, NT, false>(v, rv, n_left);
    }
    float carry = 1.0f;                          // product of the gates after the token, last tile first
#pragma unroll
    for (int m = NT - 1; m >= 0; --m) {
        float s[4];
        s[3] = 1.0f;
#pragma unroll
        for (int j = 2; j >= 0; --j) s[j] = s[j + 1] * gt[m][j + 1];
        const RowScan above = row_scan_mul_above(s[0] * gt[m][0], kg);
#pragma unroll
        for (int j = 0; j < 4; ++j) after[m][j] = carry * above.lower * s[j];
        carry *= above.all;
    }
    uint2 op[NT];
    scale_pack<NT>(op, v, after);
    store_cm<NT>(reinterpret_cast<u16 *>(smem + side * CM_BYTES), c, kg, op);
    if (side == 0) {
        uint2 rest[NT];
        scale_pack_rest<NT>(rest, op, v, after);
        store_cm<NT>(reinterpret_cast<u16 *>(smem + 2 * CM_BYTES), c, kg, rest);
    }
    if (kg == 0) {
        float *vec = p.vecs + (int64_t)item * (PF_NVEC * CH_N) + c;
        vec[side * CH_N] = carry;
        if (side == 1) vec[2 * CH_N] = pow2_below(lc.ref);
    }
    const int any_bad = __syncthreads_or((int)lc.bad);
    if (tid == 0) {
        p.chunk_flags[item] = any_bad ? 1 : 0;
        if (chunk == 0) p.declined[b] = p.declined[p.B + b] = 0;
    }
    // this wave's two tiles of the increment: rows d = 16 db + 4 kg + j, column k = 16 kb + i
    const u16 *const XH = reinterpret_cast<const u16 *>(smem), *const KH = reinterpret_cast<const u16 *>(smem + CM_BYTES),
              *const XR = reinterpret_cast<const u16 *>(smem + 2 * CM_BYTES);
    const int db = w & 3, kb0 = 2 * (w >> 2);
    uint4 xa[NT / 2], xr[NT / 2];
#pragma unroll
    for (int h = 0; h < NT / 2; ++h) {
        xa[h] = mat_rows_op(XH, 16 * db, h, i, kg);
        xr[h] = mat_rows_op(XR, 16 * db, h, i, kg);
    }
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int kb = kb0 + t;
        floatx4 m = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int h = 0; h < NT / 2; ++h) {
            const uint4 kh = mat_rows_op(KH, 16 * kb, h, i, kg);
            m = Bf16::mfma32(xa[h], kh, Bf16::mfma32(xr[h], kh, m));
        }
        float *const dst = p.incr + (int64_t)item * (CH_N * CH_N) + (16 * db + 4 * kg) * CH_N + 16 * kb + i;
#pragma unroll
        for (int j = 0; j < 4; ++j) dst[j * CH_N] = m[j];
    }
}

// ---- launch 2: the chain over the chunks of a row -----------------------------------------------------
// A workgroup owns eight rows of the state of one batch row, a thread two adjacent elements; sixteen chunks at a time, whose
// gate products go through LDS and whose increments are all in flight before the chain starts.
constexpr int PF_TPB = 256, PF_BATCH = 16, PF_VEC = 8 + 2 * CH_N;          // per chunk: totA of 8 rows; totB, refB
constexpr int PF_STAGE = (PF_BATCH * PF_VEC + PF_TPB - 1) / PF_TPB;

template <typename IOE> __global__ __launch_bounds__(PF_TPB) void lfw_par_fwd_scan_kernel(ParFwdArgs p) {
    __shared__ float vl[PF_STAGE * PF_TPB];
    const int64_t b = (int64_t)(blockIdx.x >> 6) * 8 + (blockIdx.x & 7);      // the eight slabs of a row on one XCD
    if (b >= p.B) return;
    const int slab = (int)((blockIdx.x >> 3) & 7), tid = threadIdx.x;
    const int dl = tid >> 5, d = slab * 8 + dl, k = (tid & 31) * 2;
    const int NC = (int)p.NC;
    const int64_t at = b * NC * (int64_t)(CH_N * CH_N) + d * CH_N + k;
    float S0, S1;
    {
        const u32 s = *reinterpret_cast<const u32 *>(reinterpret_cast<const u16 *>(p.s0) + b * (CH_N * CH_N) + d * CH_N + k);
        S0 = IOE::to_f32((u16)(s & 0xffffu));
        S1 = IOE::to_f32((u16)(s >> 16));
    }
    const float *const incr = p.incr + at;
    u16 *const states = p.states + at, *const ckpt = p.ckpt ? reinterpret_cast<u16 *>(p.ckpt) + at : nullptr;
    const float *const vecs = p.vecs + b * NC * (int64_t)(PF_NVEC * CH_N);
    for (int c0 = 0; c0 < NC; c0 += PF_BATCH) {
        float2 m[PF_BATCH];
#pragma unroll
        for (int u = 0; u < PF_BATCH; ++u) m[u] = *reinterpret_cast<const float2 *>(incr + (int64_t)min(c0 + u, NC - 1) * (CH_N * CH_N));
        __syncthreads();                                   // the previous batch's vectors are no longer read
        float tmp[PF_STAGE];
#pragma unroll
        for (int it = 0; it < PF_STAGE; ++it) {                                    // (the last pass goes past the batch, within vl)
            const int idx = tid + it * PF_TPB;
            const int u = idx / PF_VEC, wv = idx - u * PF_VEC;
            const int src = wv < 8 ? slab * 8 + wv : CH_N + wv - 8;                // totA; totB and refB
            tmp[it] = vecs[(int64_t)min(c0 + u, NC - 1) * (PF_NVEC * CH_N) + src];
        }
#pragma unroll
        for (int it = 0; it < PF_STAGE; ++it) vl[tid + it * PF_TPB] = tmp[it];
        __syncthreads();
        float tau0[PF_BATCH], tau1[PF_BATCH], sig0[PF_BATCH], sig1[PF_BATCH];
#pragma unroll
        for (int u = 0; u < PF_BATCH; ++u) {
            const float *v = vl + u * PF_VEC;
            const float ta = v[dl];
            const float2 tb = *reinterpret_cast<const float2 *>(v + 8 + k), rb = *reinterpret_cast<const float2 *>(v + 8 + CH_N + k);
            tau0[u] = ta * tb.x; tau1[u] = ta * tb.y;
            sig0[u] = PAR_STATE_SHIFT * rb.x; sig1[u] = PAR_STATE_SHIFT * rb.y;    // S0' is stored shifted
        }
#pragma unroll
        for (int u = 0; u < PF_BATCH; ++u) {
            const int c = c0 + u;
            if (c < NC) {
                *reinterpret_cast<u32 *>(states + (int64_t)c * (CH_N * CH_N)) = Bf16::pack2(S0 * sig0[u], S1 * sig1[u]);
                if (ckpt) *reinterpret_cast<u32 *>(ckpt + (int64_t)c * (CH_N * CH_N)) = IOE::pack2(S0, S1);
                S0 = S0 * tau0[u] + m[u].x;
                S1 = S1 * tau1[u] + m[u].y;
            }
        }
    }
    *reinterpret_cast<u32 *>(reinterpret_cast<u16 *>(p.next_state) + b * (CH_N * CH_N) + d * CH_N + k) = IOE::pack2(S0, S1);
    int bad = !(S0 * 0.0f + S1 * 0.0f == 0.0f);
    if (slab == 0)                    // any chunk the form cannot take
        for (int cc = tid; cc < NC; cc += PF_TPB) bad |= p.chunk_flags[b * NC + cc];
    const int any = __syncthreads_or(bad);
    if (tid == 0 && any) p.declined[b] = 1;              // launch 1 has cleared it
    if (slab == 0 && tid == 0) {
        p.row_flags[b] = p.row_flags[chunk_rows_padded(p.B) + b] = 0;
        if (p.par_hint != nullptr) p.par_hint[b] = p.par_hint[chunk_rows_padded(p.B) + b] = 0;
    }
}

// ---- launch 3: outputs ---------------------------------------------------------------------------------
// Waves 0 to 3: the value side, a block of 16 channels each; waves 4 to 7: the key side, whose operands go to LDS.  All eight share
// the ten tiles of P; the value side's waves then make the outputs, own channels and tokens in the lane that scales them.
constexpr int PO_QS = 0, PO_KT = PO_QS + CM_BYTES, PO_S0 = PO_KT + CM_BYTES, PO_PT = PO_S0 + CM_BYTES, PO_TILE = 64 * 8,
              PO_SMEM = PO_PT + 20 * PO_TILE;                   // P: heads, then remainders

template <typename IOE, bool HEADS, bool FULL> __device__ __forceinline__ void outputs_of(const ParFwdArgs &p, unsigned char *smem, int item) {
    constexpr int NT = PF_NT, CL = PF_CL;
    const int tid = threadIdx.x, w = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int cb = w & 3, i = lane & 15, kg = lane >> 4, c = 16 * cb + i;
    const int NC = (int)p.NC, T = (int)p.T;
    const int64_t b = item / NC;
    const int chunk = item - (int)b * NC;
    const u32 ts = HEADS ? (u32)p.heads * CH_N : (u32)CH_N;
    const int n_left = T - (chunk * CL + 4 * kg);
    const int64_t chunk_off = wave_uniform(row_first_token(b, p.T, HEADS ? p.heads : 1) * CH_N + (int64_t)(chunk * CL) * ts);
    const u32 lane_off = (u32)(4 * kg) * ts + (u32)c;
    u16 *const QS = reinterpret_cast<u16 *>(smem + PO_QS), *const KT = reinterpret_cast<u16 *>(smem + PO_KT), *const S0 = reinterpret_cast<u16 *>(smem + PO_S0);
    uint2 *const pt = reinterpret_cast<uint2 *>(smem + PO_PT);
    const int declined = p.declined[b];
    const uint4 state = *reinterpret_cast<const uint4 *>(p.states + (int64_t)item * (CH_N * CH_N) + tid * 8);
    LaneChunk<NT> lc;
    float gt[NT][4], inv[NT][4];
    uint2 xt[NT];
    if (w < 4) {
        RawTokens<NT> rg, rv;
        float v[NT][4];
        load_tokens<NT, FULL>(rg, reinterpret_cast<const u16 *>(p.f) + chunk_off, lane_off, ts, n_left);
        load_tokens<NT, FULL>(rv, reinterpret_cast<const u16 *>(p.x) + chunk_off, lane_off, ts, n_left);
        gate_scan<IOE, NT, FULL, true, IOE::FLOOR_BITS, true>(lc, gt, rg, kg, n_left);
        to_floats<IOE, NT, FULL>(v, rv, n_left);
        inverse_products<NT>(inv, lc, gt);
        scale_pack<NT>(xt, v, inv);
    } else {
        RawTokens<NT> rg, rv, ra;
        float v[NT][4], a[NT][4];
        load_tokens<NT, FULL>(rg, reinterpret_cast<const u16 *>(p.f_key) + chunk_off, lane_off, ts, n_left);
        load_tokens<NT, FULL>(rv, reinterpret_cast<const u16 *>(p.k) + chunk_off, lane_off, ts, n_left);
        load_tokens<NT, FULL>(ra, reinterpret_cast<const u16 *>(p.q) + chunk_off, lane_off, ts, n_left);
        gate_scan<IOE, NT, FULL, true, IOE::FLOOR_BITS, true>(lc, gt, rg, kg, n_left);
        to_floats<IOE, NT, FULL>(v, rv, n_left);
        to_floats<IOE, NT, FULL>(a, ra, n_left);
        inverse_products<NT>(inv, lc, gt);
        uint2 kt[NT], qs[NT];
        scale_pack<NT>(kt, v, inv);
        scale_pack<NT>(qs, a, lc.pre);
        store_cm<NT>(KT, c, kg, kt);
        store_cm<NT>(QS, c, kg, qs);
    }
    *reinterpret_cast<uint4 *>(S0 + (tid >> 3) * CMS + (tid & 7) * 8) = state;
    if (__builtin_amdgcn_readfirstlane(declined)) return;          // uniform over the workgroup: nothing in this launch writes it
    __syncthreads();
    const floatx4 zero = {0.f, 0.f, 0.f, 0.f};
    // tile (m, n), n <= m, of P at m (m + 1) / 2 + n: element [t = 16 m + i][s = 16 n + 4 kg + j] in lane (i, kg), s <= t
    for (int t = w; t < 10; t += 8) {
        const int m = t < 1 ? 0 : t < 3 ? 1 : t < 6 ? 2 : 3, n = t - m * (m + 1) / 2;
        const floatx4 r = Bf16::mfma32(tok_rows_op(KT, 16 * n, 1, i, kg), tok_rows_op(QS, 16 * m, 1, i, kg),
                                       Bf16::mfma32(tok_rows_op(KT, 16 * n, 0, i, kg), tok_rows_op(QS, 16 * m, 0, i, kg), zero));
        const floatx4 v = m == n ? mask<KEEP_ROW_LE_COL>(r, i, kg) : r;
        const uint2 head = packq<Bf16>(v[0], v[1], v[2], v[3]);
        pt[t * 64 + lane] = head;
        pt[(10 + t) * 64 + lane] = pack_rest(head, v[0], v[1], v[2], v[3]);
    }
    __syncthreads();
    if (w >= 4) return;
    u16 *const out = reinterpret_cast<u16 *>(p.out) + chunk_off;
    const uint4 s0a = mat_rows_op(S0, 16 * cb, 0, i, kg), s0b = mat_rows_op(S0, 16 * cb, 1, i, kg);
    const uint2 none = make_uint2(0u, 0u);
    const float ref = pow2_below(lc.ref);                          // pre * ref: from the chunk's start
    float chk = 0.f;
#pragma unroll
    for (int m = 0; m < NT; ++m) {
        const floatx4 old = Bf16::mfma32(tok_rows_op(QS, 16 * m, 1, i, kg), s0b, Bf16::mfma32(tok_rows_op(QS, 16 * m, 0, i, kg), s0a, zero));
        floatx4 acc = zero;
#pragma unroll
        for (int n0 = 0; n0 <= m; n0 += 2) {
            const int t = m * (m + 1) / 2 + n0;
            const uint4 x = cat(xt[n0], n0 + 1 <= m ? xt[n0 + 1] : none);
#pragma unroll
            for (int part = 10; part >= 0; part -= 10)
                acc = Bf16::mfma32(cat(pt[(part + t) * 64 + lane], n0 + 1 <= m ? pt[(part + t + 1) * 64 + lane] : none), x, acc);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float o = lc.pre[m][j] * acc[j] + (lc.pre[m][j] * ref) * (old[j] * PAR_STATE_UNSHIFT);
            if (FULL || 16 * m + j < n_left) {
                chk = __builtin_fmaf(o, 0.0f, chk);
                (out + (size_t)(16 * m + j) * ts)[lane_off] = cvt1<IOE>(o);
            }
        }
    }
    if (!(chk == 0.0f)) p.declined[p.B + b] = 1;
}

template <typename IOE, bool HEADS> __global__ __launch_bounds__(PAR_THREADS, 4) void lfw_par_fwd_out_kernel(ParFwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int item = (int)blockIdx.x;
    if ((item % (int)p.NC) * PF_CL + PF_CL <= (int)p.T)
        outputs_of<IOE, HEADS, true>(p, smem, item);
    else
        outputs_of<IOE, HEADS, false>(p, smem, item);
}

template <typename IOE, bool HEADS> int launch(const ParFwdArgs &a, hipStream_t stream) {
    const int64_t items = a.B * a.NC;
    hipLaunchKernelGGL((lfw_par_fwd_incr_kernel<IOE, HEADS>), dim3((unsigned)items), dim3(PAR_THREADS), PF_INCR_SMEM, stream, a);
    int rc = check_hip(hipGetLastError(), "lfw_par_fwd_incr_kernel launch");
    if (rc) return rc;
    hipLaunchKernelGGL((lfw_par_fwd_scan_kernel<IOE>), dim3((unsigned)(64 * ((a.B + 7) / 8))), dim3(PF_TPB), 0, stream, a);
    if ((rc = check_hip(hipGetLastError(), "lfw_par_fwd_scan_kernel launch"))) return rc;
    hipLaunchKernelGGL((lfw_par_fwd_out_kernel<IOE, HEADS>), dim3((unsigned)items), dim3(PAR_THREADS), PO_SMEM, stream, a);
    return check_hip(hipGetLastError(), "lfw_par_fwd_out_kernel launch");
}

}  // namespace

int par_forward(const ParFwdArgs &a, int dtype, hipStream_t stream) {
    if (a.heads < 1 || a.T * a.heads >= CHUNK_MAX_T || a.B * a.NC > PAR_FWD_MAX_ITEMS || a.B * a.T * CH_N >= 0x7fffffffLL)
        return fail(T2FW_ERR_UNSUPPORTED, "B=%lld T=%lld with %d heads is too large for the chunk-parallel forward", (long long)a.B, (long long)a.T, a.heads);
    if (dtype == T2FW_F16) return a.heads == 1 ? launch<Fp16, false>(a, stream) : launch<Fp16, true>(a, stream);
    if (dtype == T2FW_BF16) return a.heads == 1 ? launch<Bf16, false>(a, stream) : launch<Bf16, true>(a, stream);
    return fail(T2FW_ERR_UNSUPPORTED, "the chunk-parallel kernels take fp16 or bf16 tensors");
}

}  // namespace t2fw
