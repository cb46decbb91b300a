// Argument blocks and host entry points of the delta-rule kernels (dfw_scan.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace t2fw {

struct DfwFwdArgs {
    const void *q, *k, *v, *s0;
    void *out, *final_state, *delta;
    int64_t B, T, D, M;
    int32_t kg, tb, ntiles;
    int32_t blocks;                    // matrix-core kernels: value blocks of 64 (at least 1); B counts (row, block) pairs
};

struct DfwBwdArgs {
    const void *g_out, *g_state, *q, *k, *delta, *final_state;
    void *d_q, *d_k, *d_v, *d_s0;
    int64_t B, T, D, M;
    int32_t kg, tb, ntiles;
    int32_t blocks;                    // matrix-core kernels: value blocks of 64 (at least 1); B counts (row, block) pairs
    void *states, *adjoints;           // null, or arrays of the shape and type of d_q and d_k (per block), for the key side's chunks;
                                       // without blocks d_q and d_k themselves.  d_q and d_k are then sums over the blocks.
};

// Whether the key side runs in chunks of 64 tokens: a state at a chunk's edge (one or two bf16 planes of 64 x 64) has to fit where the
// chunk's 64 tokens of a result go.
constexpr bool dfw_key_chunks_ok(size_t elem_bytes, bool split_operands) { return elem_bytes == 4 || !split_operands; }

int dfw_forward(const DfwFwdArgs &a, int dtype, hipStream_t stream);
int dfw_backward(const DfwBwdArgs &a, int dtype, hipStream_t stream);
// block-wise matrix-core kernels: M = 64, D = 64 `blocks` (each a recurrence of its own), fp32 / fp16 / bf16 tensors, 16-byte
// aligned pointers (dfw_chunk_fwd.hip, dfw_chunk_bwd.hip)
int dfw_chunk_forward(const DfwFwdArgs &a, int dtype, bool split_operands, hipStream_t stream);
int dfw_chunk_backward(const DfwBwdArgs &a, int dtype, bool split_operands, hipStream_t stream);
int dfw_key_chunks(const DfwBwdArgs &a, int dtype, bool split_operands, hipStream_t stream);       // dfw_key.hip; the second launch of the above

}  // namespace t2fw
