// Waiting for this wavefront's vector-memory operations.
#pragma once
#include <hip/hip_runtime.h>

namespace fgx {
namespace {

// s_waitcnt with only the vector-memory counter constrained (gfx9 encoding: vmcnt = imm[3:0] | imm[15:14] << 4,
// expcnt = imm[6:4], lgkmcnt = imm[11:8]; all-ones = unconstrained)
template <int N>
__device__ __forceinline__ void wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// s_waitcnt vmcnt(n) for a wave-uniform n in [LO, HI]: the count is an immediate, so a binary tree of scalar branches
// picks the instruction.
template <int LO, int HI>
__device__ __forceinline__ void wait_vmcnt_in(int n) {
    if constexpr (LO == HI) {
        wait_vmcnt<LO>();
    } else {
        constexpr int MID = (LO + HI) / 2;
        if (n <= MID) wait_vmcnt_in<LO, MID>(n);
        else wait_vmcnt_in<MID + 1, HI>(n);
    }
}

}  // namespace
}  // namespace fgx
