// Matrix-core form of the decay rule at the accuracy of the exact kernels: fp32 operands, fp32 accumulation, states of
// up to 64 x 64 of any width, fp32 / fp16 / bf16 tensors.
//
// Tokens are taken in tiles of 16.  Every factor of a tile is taken relative to its MIDDLE: with a_t[d] the product of
// the value-side gates from the tile's first token to t, lo = a_7 and up = a_15 / a_7 (eight gates each),
//   a'_t = a_t / lo    xm_t = x_t / a'_t    gm_t = g_t a'_t        (key side: b'_t, km_t = k_t / b'_t, qm_t = q_t b'_t)
// so that no factor spans more than eight gates.  A wave owns 16 channels of one side ("own" side, value channels d in
// the formulas below) and carries the slab S[16 d][64 k] in fp32 accumulators; per tile, with S the state before it,
//   S'      = S lo_k                                              (scaled to the middle of the tile on the other side)
//   o_t     = a'_t ( lo_d (qm_t . S') + sum_{s<=t} (qm_t . km_s) xm_s )
//   S_next  = up_k ( S' (lo_d up_d) + sum_s km_s (x) (xm_s up_d) )
// and up_k of a tile times lo_k of the next is one factor (rho_k).  All that is multiplied into S is <= 1; what is
// scaled up is scaled by at most eight gates.  The adjoint runs the same way backwards (lfw_tile_bwd.hip), and the
// key side is the same with the two sides exchanged and the state transposed.
//
// Lane layout: v_mfma_f32_16x16x4_f32 takes A[i][kg] and B[kg][i] in lane (i = lane & 15, kg = lane >> 4) and returns
// rows 4 kg + j of column i.  A lane of wave (side, cb) owns channel 16 cb + i and tokens 16 m + 4 kg + j of its side.
// In fp32 the accumulator of a slab (row = other side's channel 16 q + 4 kg + e, column = own channel i) is at once the
// B operand of a product that contracts over the other side's channels, so the state never moves; a lane's own
// scaled tokens are the B operand of what contracts over tokens.  The other side's operands come from LDS, token-major
// [64][TLS] fp32: rows of tokens as 16-byte reads, columns as four 4-byte reads, both without bank conflicts.
#pragma once

#include "common.hpp"
#include "lfw_chunk.hpp"

namespace t2fw {

struct TileFwdArgs {
    const void *x, *f, *q, *k, *f_key, *s0;
    void *out, *next_state, *ckpt;     // ckpt may be null; else one state per 64 steps
    int64_t B, T, NC;
    int32_t D, K, heads;
};

struct TileBwdArgs {
    const void *g_out, *g_state, *x, *f, *q, *k, *f_key, *ckpt;
    void *d_x, *d_f, *d_q, *d_k, *d_f_key, *d_s0;
    float *gh;                         // scratch [B * NC][64][64]: adjoint increment of a chunk, then the adjoint at its end
    float *tots;                       // scratch [B * NC][2][64]: the chunk's gate products, value side and key side
    int32_t *flags;                    // scratch [B * NC]: the adjoint at the chunk's end is out of the tiles' range
    int32_t *list;                     // scratch [1 + B * NC]: number of chunks left to the exact recurrence, their items
    int64_t B, T, NC;
    int32_t D, K, heads;
};

constexpr int TILE_CHUNK = 64;         // tokens between checkpoints and per workgroup of the backward
int tile_forward(const TileFwdArgs &a, int dtype, hipStream_t stream);
int tile_backward(const TileBwdArgs &a, int dtype, hipStream_t stream);

#if defined(__HIPCC__)
namespace tilem {

constexpr int TLS = 68;                // row stride, in floats, of the token-major tiles [64][TLS]
constexpr int TL_FLOATS = TILE_CHUNK * TLS;
constexpr int PT_FLOATS = 4 * TLS;     // a 16 x 16 product tile: element (t, s) at (s / 4) TLS + 4 t + s % 4
constexpr int VEC_FLOATS = 5 * CH_N;   // per chunk and side: lo of tile 0, rho of tiles 0..2, up of tile 3

// An eight-gate product below this, or a scaled operand above TILE_MAX_OPERAND (inf and NaN included), sends the chunk
// to the exact recurrence: sums of 64 products of two operands times a third stay below 2^124.
constexpr float TILE_MIN_PRODUCT = 8.673617379884035e-19f;      // 2^-60
constexpr float TILE_MAX_OPERAND = 274877906944.0f;             // 2^38
constexpr float TILE_MAX_STATE = 1.2089258196146292e24f;        // 2^80

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// a value that is the same in every lane, moved to scalar registers
__device__ __forceinline__ int64_t uniform64(int64_t v) {
    const u32 lo = __builtin_amdgcn_readfirstlane((u32)(unsigned long long)v);
    const u32 hi = __builtin_amdgcn_readfirstlane((u32)((unsigned long long)v >> 32));
    return (int64_t)(((unsigned long long)hi << 32) | lo);
}

// The lane's tokens of one array over a chunk: [m][j] is token 16 m + 4 kg + j.  ubase: the array at the chunk's first
// token, channel 0 (wave-uniform); lane_off = 4 kg ts + c.  n_left: tokens from the lane's first one to the end of the
// sequence; tokens past it are read from the last one (and replaced when they are used).
template <typename IO, bool FULL>
__device__ __forceinline__ void load_tile_tokens(IO (&r)[4][4], const IO *ubase, u32 lane_off, u32 ts, int n_left) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (FULL) {
                r[m][j] = (ubase + (size_t)(16 * m + j) * ts)[lane_off];
            } else {
                const int o = min(16 * m + j, n_left - 1);           // may be negative: the lane starts past the end
                r[m][j] = ubase[(int)lane_off + o * (int)ts];
            }
        }
}

// Products over the sixteen lanes-rows of a tile: l = the lane's own four-gate product
struct TileProducts {
    float below, above;      // product of the rows of the same half below / above this lane's row (one row at most)
    float lo, up;            // products of the two halves (rows 0-1, rows 2-3)
};
__device__ __forceinline__ TileProducts tile_products(float l, int kg) {
    const u32 vb = __float_as_uint(l);
    const auto s16 = __builtin_amdgcn_permlane16_swap(vb, vb, false, false);     // {even row of the pair, odd row}
    const float ev = __uint_as_float(s16[0]), od = __uint_as_float(s16[1]);
    const float pair = ev * od;
    const u32 pb = __float_as_uint(pair);
    const auto s32 = __builtin_amdgcn_permlane32_swap(pb, pb, false, false);     // {rows 0-1, rows 2-3}
    TileProducts r;
    r.lo = __uint_as_float(s32[0]);
    r.up = __uint_as_float(s32[1]);
    r.below = (kg & 1) ? ev : 1.0f;
    r.above = (kg & 1) ? 1.0f : od;
    return r;
}

// a'_t and 1 / a'_t of the lane's four tokens of a tile.  For the tokens of the upper half a'_t is the product of the
// gates from the middle to t; for those of the lower half 1 / a'_t is the product of the gates after t up to the middle.
// Either way the smaller of the two is a plain product and the other its reciprocal.
__device__ __forceinline__ void tile_scales(float (&pre)[4], float (&inv)[4], const float (&g)[4], const TileProducts &tp, int kg) {
    const bool upper = kg >= 2;
    float e[4];
    if (upper) {
        e[0] = tp.below * g[0];
#pragma unroll
        for (int j = 1; j < 4; ++j) e[j] = e[j - 1] * g[j];
    } else {
        e[3] = tp.above;
#pragma unroll
        for (int j = 2; j >= 0; --j) e[j] = e[j + 1] * g[j + 1];
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float r = __builtin_amdgcn_rcpf(e[j]);
        pre[j] = upper ? e[j] : r;
        inv[j] = upper ? r : e[j];
    }
}

// product tile, result orientation [s = 4 kg + j][t = i] -> LDS, ready as an A operand: lane (i, kg) reads its own four
// floats back for A[t = i][s = 4 kg + e]
__device__ __forceinline__ float *pt_lane(float *pt, int i, int kg) { return pt + kg * TLS + 4 * i; }

__device__ __forceinline__ float4 ldv4(const float *p) { return *reinterpret_cast<const float4 *>(p); }

}  // namespace tilem
#endif

}  // namespace t2fw
