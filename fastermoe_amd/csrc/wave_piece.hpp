// Which piece of which row a wave of a streaming kernel works on (device code).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace fmoe {

// piece number of the calling wave, in scalar registers
__device__ __forceinline__ int64_t wave_piece(int waves_per_block) {
    return (int64_t)blockIdx.x * waves_per_block + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
}

// n / d for n >= 0, d >= 1, both the same in all lanes.  A 64-bit division by a number the compiler does not know takes some
// 150 instructions, and two of them were a sixth of a pass over rows of 4 KiB (8192 tokens combined from eight rows each in
// bf16: 60 us with, 51 without; 32768 tokens of 8 KiB, top-2: 150 and 128; 16384 of 2 KiB: 22.6 and 18.6); operands that fit
// 32 bits, nearly always, take 20.
__device__ __forceinline__ int64_t div_small(int64_t n, int64_t d) {
    if (((uint64_t)n | (uint64_t)d) >> 32) return n / d;
    return (int64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)n / (uint32_t)d));
}

}  // namespace fmoe
