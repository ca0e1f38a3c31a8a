// Words of rows that workgroups of one launch hand to each other (chain.hip): all ones until they are written, so what is written is never all ones.
#pragma once
#include <stdint.h>

namespace fh {

constexpr uint32_t NOT_YET = ~0u;

// Numbers that are handed off: the one fp16, and fp32, NaN that reads as NOT_YET loses its sign.
__host__ __device__ inline __attribute__((always_inline)) uint32_t written2(uint32_t w) {
    if ((w & 0xFFFFu) == 0xFFFFu) w ^= 0x8000u;
    return w >= 0xFFFF0000u ? w ^ 0x80000000u : w;
}
__host__ __device__ inline __attribute__((always_inline)) uint32_t written1(uint32_t w) { return w == NOT_YET ? w ^ 0x80000000u : w; }

}  // namespace fh
