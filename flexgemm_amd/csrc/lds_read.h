// Transposing LDS read (ds_read_b64_tr_b16): in a group of 16 lanes, lane s names 4 adjacent columns of K row s / 4 and receives 4 K
// values of column s.  Issued as inline assembly: through the compiler builtin every such read is preceded by a conservative
// s_waitcnt vmcnt(0) (the compiler cannot tell it apart from the LDS areas the in-flight direct-to-LDS loads are filling),
// which would drain the whole ring each step.  The price is that the result must be waited for by hand: lds_wait_all() ties the
// registers to an s_waitcnt lgkmcnt(0).
#pragma once
#include <stdint.h>

namespace fgx {
namespace {

using i16x4 = short __attribute__((ext_vector_type(4)));

__device__ __forceinline__ i16x4 lds_read_tr16(const unsigned char* p) {
    const uint32_t addr = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p;
    i16x4 r;
    asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(r) : "v"(addr));
    return r;
}
// the same with the address given as an LDS byte address plus a constant that goes into the instruction's offset field
template <int OFFSET>
__device__ __forceinline__ i16x4 lds_read_tr16_at(uint32_t addr) {
    static_assert(OFFSET >= 0 && OFFSET < 65536, "the offset field is 16 bits wide");
    i16x4 r;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFFSET));
    return r;
}
template <int N>
__device__ __forceinline__ void lds_wait_all(i16x4 (&r)[N]) {
    static_assert(N % 4 == 0, "fragments come in groups of four registers pairs");
#pragma unroll
    for (int i = 0; i < N; i += 4)
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(r[i]), "+v"(r[i + 1]), "+v"(r[i + 2]), "+v"(r[i + 3]));
}

}  // namespace
}  // namespace fgx
