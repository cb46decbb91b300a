// Forward scan of the decay rule on fp32 matrix cores (algebra, lane layout and operand tiles: lfw_tile.hpp).
//
// One workgroup of eight waves per batch row, 64 tokens per stage.  Matrix wave w keeps S[16 w .. 16 w + 15][:] in
// accumulators for the whole sequence, prepares its own side's operands (x, f: the lane's own tokens, in registers) and
// stores the outputs.  Key wave w prepares channels 16 w .. of k, q, f_key for the next stage in LDS (two buffers).  A
// stage has two barriers: the operands of the stage are there; the four product tiles (one per matrix wave) are there.
//
// Bound by the serial chain of a row: per tile 16 + 16 + 4 dependent-ish matrix instructions of 32 cycles a wave, one
// row per compute unit.  B = 96, T = 1024, 64 x 64 fp32: 116 us (the per-step kernel: 224 us); 13 rows, T = 385,
// 33 x 17 fp16: 42 us (75 us).
//
// Replaces lfw_cuda_fwd_kernel + the output einsum of the reference
// (t2fw/csrc/lfw_kernel.cu:18-59, t2fw/csrc/lfw.cpp:45); semantics t2fw/torch.py:21-31.
#include <type_traits>

#include "lfw_tile.hpp"
#include "lfw_chunk_bwd_dev.hpp"

namespace t2fw {
namespace {

using namespace tilem;

constexpr int TF_THREADS = 512;
// Gates enter no smaller than this: a zero gate keeps its tile's products in range and lets 2^-48 of the state through,
// far below the fp32 rounding of the state before it.
constexpr float TILE_GATE_FLOOR = 3.552713678800501e-15f;      // 2^-48

struct FwdSmem {
    float km[2][TL_FLOATS], qm[2][TL_FLOATS], vec[2][VEC_FLOATS], pt[4][PT_FLOATS];
    int bad[2][4];
};

template <typename IO, bool W64> struct FwdRow {
    const TileFwdArgs &p;
    FwdSmem &sm;
    int64_t b, line0;
    int T, D, K, H, cb, i, kg, nfull, nst;

    __device__ __forceinline__ FwdRow(const TileFwdArgs &p_, FwdSmem &sm_, int wave, int lane) : p(p_), sm(sm_) {
        b = blockIdx.x;
        T = (int)p.T; D = W64 ? CH_N : p.D; K = W64 ? CH_N : p.K; H = p.heads;
        line0 = uniform64(row_first_token(b, p.T, H));
        cb = wave & 3; i = lane & 15; kg = lane >> 4;
        nfull = T / TILE_CHUNK;
        nst = (T + TILE_CHUNK - 1) / TILE_CHUNK;
    }
    __device__ __forceinline__ int blocks(int n) const { return W64 ? 4 : (n + 15) >> 4; }
    // gates, token by token; what does not exist (past the sequence, past the last channel) acts as identity
    template <bool FULL>
    __device__ __forceinline__ void gates(float (&g)[4], u32 &bad, const IO (&raw)[4], int m, int n_left, bool ch_ok) const {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float v = ((FULL || 16 * m + j < n_left) && (W64 || ch_ok)) ? to_acc(raw[j]) : 1.0f;
            bad |= !(v <= 1.0f && v >= 0.0f) ? 1u : 0u;
            g[j] = fmaxf(v, TILE_GATE_FLOOR);
        }
    }
    template <bool FULL>
    __device__ __forceinline__ float value(IO raw, int m, int j, int n_left, bool ch_ok) const {
        return ((FULL || 16 * m + j < n_left) && (W64 || ch_ok)) ? to_acc(raw) : 0.0f;
    }

    // ---- key waves ---------------------------------------------------------------------------------
    struct KeyRaw {
        IO g[4][4], k[4][4], q[4][4];
    };
    template <bool FULL> __device__ __forceinline__ void key_load(KeyRaw &r, int s) const {
        const int c = min(16 * cb + i, K - 1), t0 = s * TILE_CHUNK;
        const u32 ts = (u32)(H * K), lo = (u32)(4 * kg) * ts + (u32)c;
        const int64_t off = uniform64((line0 + (int64_t)t0 * H) * K);
        const int n_left = T - t0 - 4 * kg;
        load_tile_tokens<IO, FULL>(r.g, (const IO *)p.f_key + off, lo, ts, n_left);
        load_tile_tokens<IO, FULL>(r.k, (const IO *)p.k + off, lo, ts, n_left);
        load_tile_tokens<IO, FULL>(r.q, (const IO *)p.q + off, lo, ts, n_left);
    }
    template <bool FULL> __device__ __forceinline__ void key_prep(const KeyRaw &r, int s) const {
        const int n_left = T - s * TILE_CHUNK - 4 * kg, c = 16 * cb + i, buf = s & 1;
        const bool ch_ok = c < K;
        float lo[4], up[4];
        u32 bad = 0;
#pragma unroll
        for (int m = 0; m < 4; ++m) {
            float g[4], pre[4], inv[4];
            gates<FULL>(g, bad, r.g[m], m, n_left, ch_ok);
            const TileProducts tp = tile_products((g[0] * g[1]) * (g[2] * g[3]), kg);
            tile_scales(pre, inv, g, tp, kg);
            lo[m] = tp.lo; up[m] = tp.up;
            bad |= (tp.lo >= TILE_MIN_PRODUCT && tp.up >= TILE_MIN_PRODUCT) ? 0u : 1u;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float km = value<FULL>(r.k[m][j], m, j, n_left, ch_ok) * inv[j];
                const float qm = value<FULL>(r.q[m][j], m, j, n_left, ch_ok) * pre[j];
                bad |= (fabsf(km) <= TILE_MAX_OPERAND && fabsf(qm) <= TILE_MAX_OPERAND) ? 0u : 1u;
                sm.km[buf][(16 * m + 4 * kg + j) * TLS + c] = km;
                sm.qm[buf][(16 * m + 4 * kg + j) * TLS + c] = qm;
            }
        }
        if (kg == 0) {
            float *v = sm.vec[buf] + c;
            v[0] = lo[0];
#pragma unroll
            for (int m = 0; m < 3; ++m) v[(m + 1) * CH_N] = up[m] * lo[m + 1];
            v[4 * CH_N] = up[3];
        }
        const int any = __any((int)bad);
        if (i == 0 && kg == 0) sm.bad[buf][cb] = any;
    }
    __device__ __forceinline__ void run_key() const {
        const bool active = W64 || cb < blocks(K);          // wave-uniform
        KeyRaw r;
        if (active) {
            if (nfull > 0) {
                key_load<true>(r, 0);
                key_prep<true>(r, 0);
                key_load<true>(r, min(1, nfull - 1));
            } else {
                key_load<false>(r, 0);
                key_prep<false>(r, 0);
            }
        } else if (i == 0 && kg == 0) {
            sm.bad[0][cb] = 0;
            sm.bad[1][cb] = 0;
        }
        int s = 0;
        for (; s + 1 < nfull; ++s) {
            __syncthreads();
            __syncthreads();
            if (active) {
                key_prep<true>(r, s + 1);
                key_load<true>(r, min(s + 2, nfull - 1));
            }
        }
        for (; s < nst; ++s) {
            __syncthreads();
            __syncthreads();
            if (s + 1 < nst && active) {                    // the partial stage
                key_load<false>(r, s + 1);
                key_prep<false>(r, s + 1);
            }
        }
    }

    // ---- matrix waves ------------------------------------------------------------------------------
    struct ValRaw {
        IO g[4][4], x[4][4];
    };
    template <bool FULL> __device__ __forceinline__ void val_load(ValRaw &r, int s) const {
        const int c = min(16 * cb + i, D - 1), t0 = s * TILE_CHUNK;
        const u32 ts = (u32)(H * D), lo = (u32)(4 * kg) * ts + (u32)c;
        const int64_t off = uniform64((line0 + (int64_t)t0 * H) * D);
        const int n_left = T - t0 - 4 * kg;
        load_tile_tokens<IO, FULL>(r.g, (const IO *)p.f + off, lo, ts, n_left);
        load_tile_tokens<IO, FULL>(r.x, (const IO *)p.x + off, lo, ts, n_left);
    }
    __device__ __forceinline__ bool el_ok(int q, int e) const { return W64 || (16 * cb + i < D && 16 * q + 4 * kg + e < K); }
    __device__ __forceinline__ void store_state(IO *dst, const floatx4 (&S)[4]) const {
        const int d = 16 * cb + i;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (el_ok(q, e)) dst[d * K + 16 * q + 4 * kg + e] = from_acc<IO>(S[q][e]);
    }
    // the stage step by step, for what the tiles cannot hold (a gate outside [0, 1], products or operands out of range)
    __device__ __forceinline__ void exact_stage(floatx4 (&S)[4], int s) const {
        const int d = 16 * cb + i, dc = min(d, D - 1);
        const int n = min(T - s * TILE_CHUNK, TILE_CHUNK);
#pragma unroll 1
        for (int t = 0; t < n; ++t) {
            const int64_t line = line0 + (int64_t)(s * TILE_CHUNK + t) * H;
            const float xv = to_acc(((const IO *)p.x)[line * D + dc]), fv = to_acc(((const IO *)p.f)[line * D + dc]);
            float acc = 0.0f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if (!el_ok(q, e)) continue;
                    const int64_t o = line * K + 16 * q + 4 * kg + e;
                    S[q][e] = S[q][e] * (fv * to_acc(((const IO *)p.f_key)[o])) + xv * to_acc(((const IO *)p.k)[o]);
                    acc += S[q][e] * to_acc(((const IO *)p.q)[o]);
                }
            const float o = bwd::row_sums(acc).all;
            if (kg == 0 && d < D) ((IO *)p.out)[line * D + d] = from_acc<IO>(o);
        }
    }
    __device__ __forceinline__ void run_matrix() const {
        const int d = 16 * cb + i, nbk = blocks(K);
        const bool active = W64 || cb < blocks(D), ch_ok = d < D;
        floatx4 S[4];
        ValRaw r;
        if (active) {
            const IO *s0 = (const IO *)p.s0 + b * ((int64_t)D * K);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) S[q][e] = el_ok(q, e) ? to_acc(s0[d * K + 16 * q + 4 * kg + e]) : 0.0f;
            if (nfull > 0)
                val_load<true>(r, 0);
            else
                val_load<false>(r, 0);
        }
        auto stage = [&](int s, auto full_c) {
            constexpr bool FULL = decltype(full_c)::value;
            const int buf = s & 1, n_left = T - s * TILE_CHUNK - 4 * kg;
            const float *const KM = sm.km[buf], *const QM = sm.qm[buf], *const VEC = sm.vec[buf];
            __syncthreads();                     // the key side's operands of this stage are there
            float pre[4][4], xm[4][4], lo[4], up[4];
            u32 bad = 0;
            if (active) {
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    float g[4], inv[4];
                    gates<FULL>(g, bad, r.g[m], m, n_left, ch_ok);
                    const TileProducts tp = tile_products((g[0] * g[1]) * (g[2] * g[3]), kg);
                    tile_scales(pre[m], inv, g, tp, kg);
                    lo[m] = tp.lo; up[m] = tp.up;
                    bad |= (tp.lo >= TILE_MIN_PRODUCT && tp.up >= TILE_MIN_PRODUCT) ? 0u : 1u;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        xm[m][j] = value<FULL>(r.x[m][j], m, j, n_left, ch_ok) * inv[j];
                        bad |= fabsf(xm[m][j]) <= TILE_MAX_OPERAND ? 0u : 1u;
                    }
                }
                if (FULL) val_load<true>(r, min(s + 1, nfull - 1));
                if (p.ckpt != nullptr) store_state((IO *)p.ckpt + (b * p.NC + s) * ((int64_t)D * K), S);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int e = 0; e < 4; ++e) bad |= fabsf(S[q][e]) <= TILE_MAX_STATE ? 0u : 1u;
                bad |= (u32)(sm.bad[buf][0] | sm.bad[buf][1] | sm.bad[buf][2] | sm.bad[buf][3]);
            }
            {   // product tile `cb`: [s][t] = km_s . qm_t, kept for s <= t
                floatx4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (!W64 && q >= nbk) break;
                    const float4 kv = ldv4(KM + (16 * cb + i) * TLS + 16 * q + 4 * kg), qv = ldv4(QM + (16 * cb + i) * TLS + 16 * q + 4 * kg);
                    a0 = mfma4(kv.x, qv.x, a0);
                    a1 = mfma4(kv.y, qv.y, a1);
                    a0 = mfma4(kv.z, qv.z, a0);
                    a1 = mfma4(kv.w, qv.w, a1);
                }
                float4 v;
                v.x = 4 * kg + 0 <= i ? a0[0] + a1[0] : 0.f;
                v.y = 4 * kg + 1 <= i ? a0[1] + a1[1] : 0.f;
                v.z = 4 * kg + 2 <= i ? a0[2] + a1[2] : 0.f;
                v.w = 4 * kg + 3 <= i ? a0[3] + a1[3] : 0.f;
                *reinterpret_cast<float4 *>(pt_lane(sm.pt[cb], i, kg)) = v;
            }
            __syncthreads();                     // the product tiles are there
            if (!active) return;
            if (__any((int)bad)) {
                exact_stage(S, s);
                return;
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if (!W64 && q >= nbk) break;
                const float4 v = ldv4(VEC + 16 * q + 4 * kg);
                S[q][0] *= v.x; S[q][1] *= v.y; S[q][2] *= v.z; S[q][3] *= v.w;
            }
            const u32 ts = (u32)(H * D);
            IO *const out = (IO *)p.out + uniform64((line0 + (int64_t)s * TILE_CHUNK * H) * D);
            const u32 lane_off = (u32)(4 * kg) * ts + (u32)d;
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                if (!FULL && s * TILE_CHUNK + 16 * m >= T) break;
                floatx4 a0 = {0.f, 0.f, 0.f, 0.f}, a1 = a0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (!W64 && q >= nbk) break;
                    const float4 qv = ldv4(QM + (16 * m + i) * TLS + 16 * q + 4 * kg);
                    a0 = mfma4(qv.x, S[q][0], a0);
                    a1 = mfma4(qv.y, S[q][1], a1);
                    a0 = mfma4(qv.z, S[q][2], a0);
                    a1 = mfma4(qv.w, S[q][3], a1);
                }
                const float4 pv = ldv4(pt_lane(sm.pt[m], i, kg));
                floatx4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j) o[j] = (a0[j] + a1[j]) * lo[m];
                o = mfma4(pv.x, xm[m][0], o);
                o = mfma4(pv.y, xm[m][1], o);
                o = mfma4(pv.z, xm[m][2], o);
                o = mfma4(pv.w, xm[m][3], o);
                const float tot = lo[m] * up[m];
                float xh[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) xh[e] = xm[m][e] * up[m];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (!W64 && q >= nbk) break;
#pragma unroll
                    for (int e = 0; e < 4; ++e) S[q][e] *= tot;
                }
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        if (!W64 && q >= nbk) break;
                        S[q] = mfma4(KM[(16 * m + 4 * kg + e) * TLS + 16 * q + i], xh[e], S[q]);
                    }
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if ((FULL || 16 * m + j < n_left) && (W64 || ch_ok)) (out + (size_t)(16 * m + j) * ts)[lane_off] = from_acc<IO>(pre[m][j] * o[j]);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if (!W64 && q >= nbk) break;
                    const float4 v = ldv4(VEC + (m + 1) * CH_N + 16 * q + 4 * kg);
                    S[q][0] *= v.x; S[q][1] *= v.y; S[q][2] *= v.z; S[q][3] *= v.w;
                }
            }
        };
        for (int s = 0; s < nfull; ++s) stage(s, std::true_type{});
        if (nfull < nst) {
            if (active && nfull > 0) val_load<false>(r, nfull);
            stage(nfull, std::false_type{});
        }
        if (active) store_state((IO *)p.next_state + b * ((int64_t)D * K), S);
    }
};

template <typename IO, bool W64> __global__ __launch_bounds__(TF_THREADS) void lfw_tile_fwd_kernel(TileFwdArgs p) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const FwdRow<IO, W64> row(p, *reinterpret_cast<FwdSmem *>(smem), wave, lane);
    if (wave < 4)                    // wave-uniform; both kinds meet the same two barriers per stage
        row.run_matrix();
    else
        row.run_key();
}

template <typename IO, bool W64> int launch(const TileFwdArgs &a, hipStream_t stream) {
    auto kern = lfw_tile_fwd_kernel<IO, W64>;
    int rc = enable_lds(reinterpret_cast<const void *>(kern), (int)sizeof(FwdSmem), "hipFuncSetAttribute(tile forward kernel)");
    if (rc) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)a.B), dim3(TF_THREADS), sizeof(FwdSmem), stream, a);
    return check_hip(hipGetLastError(), "lfw_tile_fwd_kernel launch");
}

}  // namespace

int tile_forward(const TileFwdArgs &a, int dtype, hipStream_t stream) {
    const bool w64 = a.D == CH_N && a.K == CH_N;
    switch (dtype) {
        case T2FW_F32: return w64 ? launch<float, true>(a, stream) : launch<float, false>(a, stream);
        case T2FW_F16: return launch<__half, false>(a, stream);
        case T2FW_BF16: return launch<__hip_bfloat16, false>(a, stream);
    }
    return fail(T2FW_ERR_UNSUPPORTED, "the tile kernels take fp32, fp16 or bf16 tensors");
}

}  // namespace t2fw
