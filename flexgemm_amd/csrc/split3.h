// fp32 matrix products on the bf16 matrix units.
#pragma once
#include "fgx_common.h"

namespace fgx {
namespace {

using bf16x8 = __bf16 __attribute__((ext_vector_type(8)));
using u32x4 = uint32_t __attribute__((ext_vector_type(4)));

// fp32 products on the bf16 units, which multiply sixteen times as fast.  Eight values of a lane as sums of three bf16 values: each is what
// the ones before leave, rounded to nearest, so the first is off by 2^-9 of the value, two by 2^-18, three by nothing (24 bits).
// Of the nine products of two such sums the six down to 2^-18 are added, smallest first; the three left out are 2^-26
// of the product together, an eighth of a rounding to fp32, and 16 values of K share six roundings where the fp32 unit rounds
// every other one (error of an output against 64 bits, 96 channels: 1.56e-7, fp32 units 1.90e-7).
// Both operands are multiplied by 2^24 first: the last bit of any fp32 value is then 2^-125 or more, so that no part falls below the normal numbers and every
// finite value under 2^104 is its three parts, the subnormal ones too; the sums are 2^48 times as large.
// What they cannot stand for: an infinity, a larger value or a sum past 2^80 leaves an infinity or NaN behind it, and products that fall below the normal numbers
// are lost, which a sum (of up to 2^22 products) shows that is not 2^24 times as large as all of them, 2^-79 (2^-127 of the result).  The
// kernels look at their sums (split3_holds) and repeat a tile on the fp32 units.  (A sum of zero is one whose products are under half of the smallest subnormal.)
constexpr float kSplit3Scale = 0x1p24f, kSplit3Unscale = 0x1p-48f;
struct Split3 {
    bf16x8 part[3];
};
// scale: kSplit3Scale, or that negated.  BY_DOT: what a part leaves of its value comes from one dot product of the pair of parts with (-1, 0) or (0, -1) instead
// of a shift or mask and a subtraction, to the same bits (a difference of two such values is exact).  For the weight gradient it makes up for the scaling
// (us, unscaled, scaled, by dot products: 96 channels, 38 720 voxels 83 88 84, 166 232 235 254 239; 64 channels 141 149 139; 128 channels 502 521 479);
// between products of 32 x 32 it waits for longer than it saves (streaming product, 166 232 voxels x 128 channels 425 443 455; pairs product level).
template <bool BY_DOT = false>
__device__ __forceinline__ Split3 split3(const u32x4& lo, const u32x4& hi, float scale = kSplit3Scale) {
    using bf16x2 = __bf16 __attribute__((ext_vector_type(2)));
    using f32x2 = float __attribute__((ext_vector_type(2)));
    float x[4], y[4];
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        x[p] = __builtin_bit_cast(float, p < 2 ? lo[p * 2] : hi[p * 2 - 4]) * scale;
        y[p] = __builtin_bit_cast(float, p < 2 ? lo[p * 2 + 1] : hi[p * 2 - 3]) * scale;
    }
    uint32_t less_lo = 0, less_hi = 0, out[3][4];
    if (BY_DOT) {           // (-1, 0) and (0, -1) in bf16, as words: as inline constants they could be read as fp32
        asm("s_mov_b32 %0, 0x0000bf80" : "=s"(less_lo));
        asm("s_mov_b32 %0, 0xbf800000" : "=s"(less_hi));
    }
#pragma unroll
    for (int t = 0; t < 3; ++t) {
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const f32x2 xy = {x[p], y[p]};
            out[t][p] = __builtin_bit_cast(uint32_t, __builtin_convertvector(xy, bf16x2));
        }
        if (t == 2) break;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            if constexpr (BY_DOT) {
                const bf16x2 part = __builtin_bit_cast(bf16x2, out[t][p]);
                x[p] = __builtin_amdgcn_fdot2_f32_bf16(part, __builtin_bit_cast(bf16x2, less_lo), x[p], false);
                y[p] = __builtin_amdgcn_fdot2_f32_bf16(part, __builtin_bit_cast(bf16x2, less_hi), y[p], false);
            } else {
                x[p] -= __builtin_bit_cast(float, out[t][p] << 16);
                y[p] -= __builtin_bit_cast(float, out[t][p] & 0xFFFF0000u);
            }
        }
    }
    Split3 s;
#pragma unroll
    for (int t = 0; t < 3; ++t) {
        const u32x4 words = {out[t][0], out[t][1], out[t][2], out[t][3]};
        s.part[t] = __builtin_bit_cast(bf16x8, words);
    }
    return s;
}
// (of the sum as it is, 2^48 times the result) neither an infinity, NaN nor other than zero below 2^-79
__device__ __forceinline__ bool split3_holds(float sum) {
    const uint32_t u = __builtin_bit_cast(uint32_t, sum) << 1;
    return u == 0u || u - (48u << 24) < (207u << 24);
}
// the six products, smallest first, of 32 x 32 over 16 values of K or 16 x 16 over 32
constexpr int kSplit3Products = 6;
template <typename Acc>
__device__ __forceinline__ void mma_split3(Acc& acc, const Split3& a, const Split3& b, int product) {
    constexpr int kOfA[kSplit3Products] = {2, 0, 1, 1, 0, 0}, kOfB[kSplit3Products] = {0, 2, 1, 0, 1, 0};
    const bf16x8 x = a.part[kOfA[product]], y = b.part[kOfB[product]];
    if constexpr (sizeof(Acc) == 64) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, acc, 0, 0, 0);
    else acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, acc, 0, 0, 0);
}
template <typename Acc>
__device__ __forceinline__ void mma_split3(Acc& acc, const Split3& a, const Split3& b) {
#pragma unroll
    for (int p = 0; p < kSplit3Products; ++p) mma_split3(acc, a, b, p);
}

}  // namespace
}  // namespace fgx
