// Argument block and host entry point of the block copy kernel (blocks.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

#include "../../include/t2fw_hip.h"

namespace t2fw {

struct BlockCopyArgs {
    t2fw_block_copy_desc a[T2FW_BLOCK_COPY_MAX];
    int64_t first[T2FW_BLOCK_COPY_MAX + 1];      // vectors of 64 elements before array i
    int32_t count;
};

int block_copy(BlockCopyArgs &a, int dtype, hipStream_t stream);

}  // namespace t2fw
