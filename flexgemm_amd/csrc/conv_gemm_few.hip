// Gather GEMM of few voxels under a small weight (16-bit types, forward): one launch, split over the wavefronts of a workgroup.
//
// The tiled kernel stages rows and weight through LDS, step after step with a barrier each, and needs split K (and a launch to add the
// pieces up) to put so few tiles on more than a handful of CUs: what bounds it is that chain of steps and the second launch.  Here a
// workgroup owns 16 rows and up to 64 columns; its eight wavefronts share the (offset, 32-channel slab) units, fetch map entry, row
// piece and weight piece of four units at a time straight into registers in the matrix instruction's layout, and add their sums in
// LDS in wavefront order (fixed: the same sums on every run).  The chain is two loads, at most a few rounds of them.
// Figures at fgx_conv_gemm_few_pays.
#include "gemm_device.h"

namespace fgx {
namespace {

constexpr int kFewRows = 16, kFewWaves = 8, kFewUnits = 4;

template <typename Tag> __device__ __forceinline__ void mma_16(f32x4& acc, const u32x4& a, const u32x4& b);
template <> __device__ __forceinline__ void mma_16<F16>(f32x4& acc, const u32x4& a, const u32x4& b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), acc, 0, 0, 0);
}
template <> __device__ __forceinline__ void mma_16<BF16>(f32x4& acc, const u32x4& a, const u32x4& b) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
}

// NC: column tiles of 16 in the workgroup.  Products are (weight piece) x (row piece): lane l then holds row l % 16 and the four
// columns 4 * (l / 16) ... + 3 of a tile.
template <typename Tag, int NC>
__global__ void __launch_bounds__(64 * kFewWaves)
few_rows_kernel(const typename Tag::type* __restrict__ src, const typename Tag::type* __restrict__ weight, const typename Tag::type* __restrict__ bias,
                const uint32_t* __restrict__ map, uint32_t n, int V, int Ci, int Co, int activation, typename Tag::type* __restrict__ out) {
    using T = typename Tag::type;
    __shared__ f32x4 sums[kFewWaves][NC][64];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l16 = lane & 15, k8 = (lane >> 4) * 8;
    const uint32_t row = blockIdx.x * kFewRows + l16;
    const int col0 = blockIdx.y * (16 * NC);
    const int slabs = (Ci + 31) / 32, units = V * slabs;
    const u32x4 zero = {0u, 0u, 0u, 0u};
    f32x4 acc[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) acc[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int u0 = wave; u0 < units; u0 += kFewWaves * kFewUnits) {
        uint32_t id[kFewUnits];
#pragma unroll
        for (int j = 0; j < kFewUnits; ++j) {
            const int u = u0 + j * kFewWaves;
            id[j] = u < units && row < n ? map[(size_t)row * V + u / slabs] : FGX_EMPTY32;
        }
        u32x4 a[kFewUnits], w[kFewUnits][NC];
#pragma unroll
        for (int j = 0; j < kFewUnits; ++j) {
            const int u = u0 + j * kFewWaves, v = u / slabs, k = u % slabs * 32 + k8;
            const bool inside = u < units && k < Ci;                    // (channels are whole pieces of eight)
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int co = col0 + c * 16 + l16;
                w[j][c] = inside && co < Co ? *reinterpret_cast<const u32x4*>(weight + ((size_t)co * V + v) * Ci + k) : zero;
            }
            a[j] = inside && id[j] != FGX_EMPTY32 ? *reinterpret_cast<const u32x4*>(src + (size_t)id[j] * Ci + k) : zero;
        }
#pragma unroll
        for (int j = 0; j < kFewUnits; ++j)
#pragma unroll
            for (int c = 0; c < NC; ++c) mma_16<Tag>(acc[c], w[j][c], a[j]);
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) sums[wave][c][lane] = acc[c];
    __syncthreads();
    if (wave >= NC || row >= n) return;
    const int col = col0 + wave * 16 + (lane >> 4) * 4;
    f32x4 total = sums[0][wave][lane];
#pragma unroll
    for (int w = 1; w < kFewWaves; ++w) total += sums[w][wave][lane];
    T x[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = from_float<T>(activate(total[e] + (bias != nullptr && col + e < Co ? to_float<T>(bias[col + e]) : 0.f), activation));
    T* dst = out + (size_t)row * Co + col;
    if (Co % 4 == 0) {                                                  // (a run of four is inside or outside as a whole)
        if (col < Co) *reinterpret_cast<uint64_t*>(dst) = __builtin_bit_cast(uint64_t, x);
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (col + e < Co) dst[e] = x[e];
    }
}

int few_col_tiles(int Co) { return Co <= 16 ? 1 : Co <= 32 ? 2 : 4; }

template <typename Tag>
void launch_few(const void* src, const void* weight, const void* bias, const uint32_t* map, size_t n, int V, int Ci, int Co, int activation, void* out,
                hipStream_t s) {
    using T = typename Tag::type;
    const int nc = few_col_tiles(Co);
    const dim3 grid(cdiv(n, (size_t)kFewRows), cdiv((size_t)Co, (size_t)(16 * nc)));
    auto kern = nc == 1 ? few_rows_kernel<Tag, 1> : nc == 2 ? few_rows_kernel<Tag, 2> : few_rows_kernel<Tag, 4>;
    kern<<<grid, 64 * kFewWaves, 0, s>>>((const T*)src, (const T*)weight, (const T*)bias, map, (uint32_t)n, V, Ci, Co, activation, (T*)out);
}

}  // namespace
}  // namespace fgx

using namespace fgx;

extern "C" {

// One round of units (27 offsets under up to 32 channels, 8 under up to 128), and at most 110 MB of weight, which every 16 rows read once
// more (from L2).  Measured (us a layer, kept cache, tiled or streaming kernel -> this):  32 -> 32 channels: 187 voxels 10.9 -> 6.9, 864
// 11.0 -> 6.6, 8 600 14.7 -> 7.6, 23 600 (81 MB) 18.8 -> 13.3, 34 000 (118 MB) 21.0 and 20.3;  32 -> 64: 8 600 16.5 -> 10.6, 34 000
// (235 MB) 19.6 and 29.7;  32 -> 128: 6 100 18.1 -> 10.8.   Two rounds, by sixteen wavefronts, gain a tenth to a third between 864 and
// 3 758 voxels of 64 channels (11.5 -> 10.0, 14.9 -> 10.1) and lose elsewhere (128 -> 128: 864 voxels 14.5 and 17.4): not built.
int fgx_conv_gemm_few_pays(int dtype, size_t n, int Ci, int Co, int V) {
    if ((dtype != FGX_F16 && dtype != FGX_BF16) || n == 0 || Ci < 8 || Ci % 8 || Co < 1 || V < 1 || V > 32) return 0;
    if (V * ((Ci + 31) / 32) > kFewWaves * kFewUnits) return 0;
    return (double)cdiv(n, (size_t)kFewRows) * V * Ci * Co * 2.0 <= 110e6;
}

int fgx_conv_gemm_few(int dtype, const void* src, const void* weight, const void* bias, const uint32_t* map, size_t n, int Ci, int Co, int V,
                      int activation, void* out, fgx_stream_t stream) {
    FGX_CHECK_ARG(dtype == FGX_F16 || dtype == FGX_BF16, "fgx_conv_gemm_few: 16-bit types only, got dtype %d", dtype);
    FGX_CHECK_ARG(V >= 1 && Ci >= 8 && Ci % 8 == 0 && Co >= 1, "fgx_conv_gemm_few: bad shape Ci=%d Co=%d V=%d", Ci, Co, V);
    FGX_CHECK_ARG(n <= ((size_t)1 << 24) && (Co + 15) / 16 <= 65535, "fgx_conv_gemm_few: too many rows or columns");
    FGX_CHECK_ARG(activation == FGX_ACT_NONE || activation == FGX_ACT_RELU, "fgx_conv_gemm_few: unknown activation %d", activation);
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(src && weight && map && out, "fgx_conv_gemm_few: null buffer");
    FGX_CHECK_ARG((((uintptr_t)src | (uintptr_t)weight) & 15) == 0 && ((uintptr_t)out & 7) == 0, "fgx_conv_gemm_few: src and weight must be 16-byte aligned, out 8-byte");
    if (dtype == FGX_F16) launch_few<F16>(src, weight, bias, map, n, V, Ci, Co, activation, out, (hipStream_t)stream);
    else launch_few<BF16>(src, weight, bias, map, n, V, Ci, Co, activation, out, (hipStream_t)stream);
    FGX_CHECK_LAUNCH("fgx_conv_gemm_few");
    return FGX_OK;
}

}  // extern "C"
