// Exact per-step recurrence, chunk-parallel: states of up to 64 x 64 of any width, fp32 / fp16 / bf16 tensors
// (lfw_xpar.hip).
#pragma once

#include "common.hpp"

namespace t2fw {

constexpr int XP_CHUNK = 64;           // tokens per chunk, and between checkpoints
constexpr int XP_N = 64;               // the widest state
constexpr float XP_MAX_INPUT = 0x1p58f, XP_MAX_STATE = 0x1p120f;      // lfw_xpar.hip
constexpr float XP_MM_MIN_GATE = 0x1p-20f;                             // lfw_xpar64_mm.hpp
constexpr int XP_ROW_LEFT = 1, XP_CHUNK_STEPS = 2;                     // chunk_flags: a smaller gate (64 x 64 fp32: step by step)
// A chunk's state in the scratch: [D][K], both rounded up to whole tiles of 16 channels.
__host__ __device__ constexpr int xp_padded(int64_t width) { return (int)((width + 15) / 16 * 16); }

struct XparScratch {
    float *states;                     // [B * NC][D][K], padded: a chunk's increment, then the state (adjoint) entering it
    float *tots;                       // [B * NC][D + K], padded: a chunk's gate products, value side and key side
    int32_t *chunk_flags;              // [B * NC]
    int32_t *row_flags;                // [B][4]: the row is left to the recurrence over the whole sequence
};

// a value that is the same in every lane, moved to scalar registers
__device__ __forceinline__ int64_t uniform64(int64_t v) {
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long long)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((unsigned long long)v >> 32));
    return (int64_t)(((unsigned long long)hi << 32) | lo);
}

// the row is left to the recurrence over the whole sequence
__device__ __forceinline__ bool row_left(const XparScratch &ws, int64_t b) {
    const int4 v = *reinterpret_cast<const int4 *>(ws.row_flags + 4 * b);
    return __builtin_amdgcn_readfirstlane(v.x | v.y | v.z | v.w) != 0;
}

struct XparFwdArgs {
    const void *x, *f, *q, *k, *f_key, *s0;
    void *out, *next_state, *ckpt;     // ckpt may be null; else one state per chunk
    XparScratch ws;
    int64_t B, T, NC;
    int32_t D, K, heads;
};

struct XparBwdArgs {
    const void *g_out, *g_state, *x, *f, *q, *k, *f_key, *ckpt;
    void *d_x, *d_f, *d_q, *d_k, *d_f_key, *d_s0;
    XparScratch ws;
    int64_t B, T, NC;
    int32_t D, K, heads;
};

int xpar_forward(const XparFwdArgs &a, int dtype, hipStream_t stream);
int xpar_backward(const XparBwdArgs &a, int dtype, hipStream_t stream);
// launch 3 for fp32 tensors with D = K = 64 (lfw_xpar64.hip)
int xpar64_forward(const XparFwdArgs &a, hipStream_t stream);
int xpar64_backward(const XparBwdArgs &a, hipStream_t stream);

}  // namespace t2fw
