// Exchanges between the lanes of a wavefront that turn the matrix units' layout of sums into runs of one row.
#pragma once
#include <hip/hip_runtime.h>

namespace fgx {
namespace {

// a's lanes 32 - 63 and b's lanes 0 - 31 change places
__device__ __forceinline__ void swap_halves(uint32_t& a, uint32_t& b) {
    const auto both = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = both[0];
    b = both[1];
}
// a's odd runs of 16 lanes and b's even ones
__device__ __forceinline__ void swap_rows(uint32_t& a, uint32_t& b) {
    const auto both = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = both[0];
    b = both[1];
}
// the same for floats (of their own: clang's bit cast of a vector's element is that of element 0)
__device__ __forceinline__ void swap_halves(float& a, float& b) {
    const auto both = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
    a = __builtin_bit_cast(float, (uint32_t)both[0]);
    b = __builtin_bit_cast(float, (uint32_t)both[1]);
}
__device__ __forceinline__ void swap_rows(float& a, float& b) {
    const auto both = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
    a = __builtin_bit_cast(float, (uint32_t)both[0]);
    b = __builtin_bit_cast(float, (uint32_t)both[1]);
}

}  // namespace
}  // namespace fgx
