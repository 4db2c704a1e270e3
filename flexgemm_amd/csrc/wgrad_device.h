// Device-side pieces shared by the weight-gradient kernels (wgrad_gemm.hip, wgrad_sweep.hip, wgrad_narrow.hip, conv_stem.hip): vector
// types, the MFMA wrappers, buffer resources, rows that are not finite.
#pragma once
#include <type_traits>

#include "fgx_common.h"
#include "lds_read.h"
#include "vmem_wait.h"

namespace fgx {
namespace {

using f16x8 = _Float16 __attribute__((ext_vector_type(8)));
using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));
using f32x16 = float __attribute__((ext_vector_type(16)));
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));
using i16x8 = short __attribute__((ext_vector_type(8)));

struct F16 { using type = _Float16; };
struct BF16 { using type = __bf16; };
struct F32 { using type = float; };
struct F32Units { using type = float; };      // multiplied on the fp32 matrix units rather than in bf16 parts

template <typename T> __device__ __forceinline__ T from_float(float x);
template <> __device__ __forceinline__ _Float16 from_float<_Float16>(float x) { return (_Float16)x; }
template <> __device__ __forceinline__ float from_float<float>(float x) { return x; }
// v_cvt_pk_bf16_f32: to nearest even, NaN stays NaN (bit for bit what shifts and adds give, over all 2^32 values; those took a branch per value)
template <> __device__ __forceinline__ __bf16 from_float<__bf16>(float x) { return (__bf16)x; }

constexpr int kMaxV = 32;
constexpr int kXcds = 8;
// Balanced item lists of the streaming weight gradient: words [0..3] = {workgroups, items, tiles per (block, offset),
// kItemListMagic}, then head[workgroups], then next[items]; kItemListEnd closes a chain.
constexpr uint32_t kItemListEnd = 0xFFFFFFFFu, kItemListMagic = 0x4C495354u;
constexpr int kItemListHeader = 4;

#define FGX_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
#define FGX_GLOBAL_PTR(p) ((const __attribute__((address_space(1))) void*)(p))
#define FGX_CONST_PTR(p) ((const __attribute__((address_space(4))) uint32_t*)(uintptr_t)(p))      // words no launch in flight writes

struct SegTable {
    uint32_t seg[kMaxV + 1];   // pair offsets per kernel offset
};

template <typename Tag> __device__ __forceinline__ void mma16(f32x16& acc, const i16x8& a, const i16x8& b);
template <> __device__ __forceinline__ void mma16<F16>(f32x16& acc, const i16x8& a, const i16x8& b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
}
template <> __device__ __forceinline__ void mma16<BF16>(f32x16& acc, const i16x8& a, const i16x8& b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}
template <> __device__ __forceinline__ void mma16<F32>(f32x16&, const i16x8&, const i16x8&) {}

// Rows of grad_out with an infinity or a NaN, for the kernels that multiply a missing neighbor as zeros: 0 * infinity is NaN
// where the sum over the pairs has no such term.  A workgroup whose sums come out finite met none; one with a sum that is not goes
// over its rows again, leaves such rows out of the matrix product and adds their pairs one by one.
__device__ __forceinline__ bool all_finite(const f32x16& a) {
    bool ok = true;
#pragma unroll
    for (int e = 0; e < 16; ++e) ok = ok && fabsf(a[e]) < __builtin_inff();
    return ok;
}
// whether nothing that is added changes the sum any more: NaN in every element with a column below `cols` and a row below `rows`
// (element e of lane l: row first_row + 8 * (e / 4) + 4 * (l / 32) + e % 4, column first_col + l % 32)
__device__ __forceinline__ bool all_nan(const f32x16& a, int lane, int first_row, int rows, int first_col, int cols) {
    bool nan = true;
#pragma unroll
    for (int e = 0; e < 16; ++e) nan = nan && (a[e] != a[e] || first_row + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3) >= rows);
    return nan || first_col + (lane & 31) >= cols;
}
constexpr uint32_t exponent16(F16) { return 0x7C00u; }
constexpr uint32_t exponent16(BF16) { return 0x7F80u; }
// the rows of the wavefront's fragment (bit 8 * half + j: element j of a lane of that half) where some lane has one
template <typename Tag>
__device__ __forceinline__ uint32_t nonfinite_rows(const i16x8& f) {
    constexpr uint32_t E = exponent16(Tag{});
    uint32_t rows = 0u;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const unsigned long long have = __ballot(((uint32_t)(uint16_t)f[j] & E) == E);
        rows |= ((have & 0xFFFFFFFFull) ? 1u : 0u) << j | ((have >> 32) ? 1u : 0u) << (8 + j);
    }
    return rows;
}
__device__ __forceinline__ void drop_rows(i16x8& f, uint32_t rows, int half) {
#pragma unroll
    for (int j = 0; j < 8; ++j)
        if ((rows >> (8 * half + j)) & 1u) f[j] = 0;
}

// eight ones in the 16-bit type, as a fragment
template <typename Tag> __device__ __forceinline__ i16x8 ones16() {
    constexpr short one = sizeof(typename Tag::type) == 2 && __is_same(typename Tag::type, _Float16) ? (short)0x3C00 : (short)0x3F80;
    return i16x8{one, one, one, one, one, one, one, one};
}

constexpr uint32_t kOobOffset = 0xFF000000u;

using rsrc_t = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>): a loop whose counter is a compile-time constant
template <int N, int I = 0, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<N, I + 1>(f);
    }
}

// wait until the LDS reads before the newest N have returned; the registers are tied to the wait so that the
// compiler cannot move their first use above it
template <int N, int R>
__device__ __forceinline__ void lds_wait_but(i16x4 (&r)[R]) {
    static_assert(N >= 0 && N < 16 && R % 4 == 0, "lgkmcnt is a 4-bit counter");
#if defined(__HIP_DEVICE_COMPILE__)   // (the host pass only needs the kernel's signature; it has no such registers)
#pragma unroll
    for (int i = 0; i < R; i += 4)
        asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(r[i]), "+v"(r[i + 1]), "+v"(r[i + 2]), "+v"(r[i + 3]) : "n"(N));
#endif
}

// bounds[v * (nb + 1) + b] = first pair of offset v whose output row is >= b * block_rows
__global__ void __launch_bounds__(256) block_bounds_kernel(const uint32_t* __restrict__ sig_o, SegTable tab, int V,
                                                           unsigned nb, unsigned block_rows,
                                                           uint32_t* __restrict__ bounds) {
    const unsigned t = blockIdx.x * 256 + threadIdx.x;
    if (t >= (unsigned)V * (nb + 1)) return;
    const unsigned v = t / (nb + 1), b = t % (nb + 1);
    uint32_t lo = tab.seg[v], hi = tab.seg[v + 1];
    const uint64_t target = (uint64_t)b * block_rows;
    while (lo < hi) {
        uint32_t mid = lo + ((hi - lo) >> 1);
        if ((uint64_t)sig_o[mid] < target) lo = mid + 1;
        else hi = mid;
    }
    bounds[t] = lo;
}

}  // namespace
}  // namespace fgx
