// Exchange between the four rows of 16 lanes of a wave (gfx950).
#pragma once

#include <hip/hip_runtime.h>

namespace lanes {

// A lane's value and that of the lane 32 (16) away, in the same order for both lanes: one instruction that swaps halves
// (rows) of two registers, in the vector ALU, where a shuffle goes through the LDS pipe and comes back some 100 cycles later.
struct Both {
    float lo, hi;
};
__device__ __forceinline__ Both both32(float v) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    return {__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1])};
}
__device__ __forceinline__ Both both16(float v) {
    const uint32_t b = __builtin_bit_cast(uint32_t, v);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    return {__builtin_bit_cast(float, (uint32_t)r[0]), __builtin_bit_cast(float, (uint32_t)r[1])};
}

// Over the lanes of the same place in the four rows; every lane gets the result.
__device__ __forceinline__ float rows_sum(float v) {
    const Both a = both16(v);
    const Both b = both32(a.lo + a.hi);
    return b.lo + b.hi;
}
__device__ __forceinline__ float rows_max(float v) {
    const Both a = both16(v);
    const Both b = both32(fmaxf(a.lo, a.hi));
    return fmaxf(b.lo, b.hi);
}

} // namespace lanes
