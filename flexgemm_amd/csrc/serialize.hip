// Space-filling-curve codes of voxel coordinates for gfx950: z-order (Morton) and Hilbert, encode / decode, and the
// "sort coordinates along the curve" pass the generic sparse convolution uses for its output coordinates.
//
// Semantics follow flex_gemm/kernels/cuda/serialize/z_order.h:22-40 and hilbert.h:22-118: x, y, z contribute bit i to
// code bits 3i+2, 3i+1, 3i; the batch index sits above the 3*bit_length spatial bits; the Hilbert code is the Morton
// code of Skilling's "transpose" of the point (J. Skilling, Programming the Hilbert curve, 2004).  The batch index is
// widened before it is shifted for both curves (the reference's z-order path shifts it as a 32-bit value, which loses
// it for 64-bit codes with bit_length >= 11).
//
// All three passes are streaming: 16 bytes of coordinates and 4 or 8 bytes of code per voxel, 16-byte vector accesses on the
// coordinate side.  The z-order shuffles are about 40 vector instructions and hide behind the memory traffic (5.3 M voxels: 17 us
// each way, 6.3 TB/s).  The Hilbert codes are the Morton code taken through a state machine in LDS, two bits per axis at a time;
// worked out bit by bit instead, 261 instructions to encode and 216 to decode filled the SIMDs for 30 us.
#include <cstring>
#include <string.h>

#include <rocprim/rocprim.hpp>

#include "fgx_common.h"

namespace fgx {
namespace {

constexpr int kBlock = 256;
constexpr int kZOrder = 1, kHilbert = 2;      // SerializationMode values of flex_gemm/ops/spconv/__init__.py:20-24

// Bits i with (i / run) % 3 == 0: runs of `run` ones, two runs of zeros between them.
template <typename T>
constexpr T run_mask(int run) {
    T m = 0;
    for (int i = 0; i < (int)(8 * sizeof(T)); ++i)
        if ((i / run) % 3 == 0) m |= (T)1 << i;
    return m;
}

// Moves bit i of v to bit 3i by doubling: each step pushes the upper half of every run two run-lengths up.
template <typename T, int RUN>
__host__ __device__ __forceinline__ T spread_step(T v) {
    constexpr T m = run_mask<T>(RUN);
    v = (v | (v << (2 * RUN))) & m;
    if constexpr (RUN > 1) v = spread_step<T, RUN / 2>(v);
    return v;
}

template <typename T>
__host__ __device__ __forceinline__ T spread3(T v) {
    return spread_step<T, (int)(2 * sizeof(T))>(v);      // first run length: 8 for 32-bit codes, 16 for 64-bit ones
}

// Inverse: collects bits 0, 3, 6, ... of v into the low bits.
template <typename T, int RUN>
__host__ __device__ __forceinline__ T gather_step(T v) {
    constexpr T m = run_mask<T>(2 * RUN > (int)(8 * sizeof(T)) ? (int)(8 * sizeof(T)) : 2 * RUN);
    v = (v | (v >> (2 * RUN))) & m;
    if constexpr (4 * RUN <= (int)(4 * sizeof(T))) v = gather_step<T, 2 * RUN>(v);
    return v;
}

template <typename T>
__host__ __device__ __forceinline__ T gather3(T v) {
    return gather_step<T, 1>(v & run_mask<T>(1));
}

// Skilling's transform as a state machine over the octants of a point, from the top bit down.  What the levels above have done to the
// lower bits is a signed permutation of the axes (exchanges and inversions act on all lower bits alike); what the Gray code's second half
// has added up so far is one parity.  A state is the two together.  In a state, the octant of a level gives the code's three bits of that
// level and the next state; both ways are tables of [state][octants of two levels], entry = the next state's row | the six bits.
// A level of zeros above the point's own changes the state only, so an odd number of levels starts in the state one zero octant before the
// first (`odd`).
struct Octant {
    uint8_t a[3];              // x, y, z
};

struct CurveState {
    uint8_t axis[3], flip[3];  // transformed bit i = bit axis[i] of the point ^ flip[i]
    uint8_t parity;
    constexpr bool operator==(const CurveState& o) const {
        for (int i = 0; i < 3; ++i)
            if (axis[i] != o.axis[i] || flip[i] != o.flip[i]) return false;
        return parity == o.parity;
    }
    // The code's octant for the point's octant p (x at bit 2, z at bit 0), and the state below.
    constexpr int step(int p, CurveState* below) const {
        const int point[3] = {(p >> 2) & 1, (p >> 1) & 1, p & 1};
        int t[3] = {};
        for (int i = 0; i < 3; ++i) t[i] = point[axis[i]] ^ flip[i];
        CurveState next = *this;
        for (int i = 0; i < 3; ++i) {          // axis i against axis 0: its bit set inverts axis 0 below, clear exchanges the two
            if (t[i]) {
                next.flip[0] ^= 1;
            } else if (i != 0) {
                const uint8_t ax = next.axis[0], fl = next.flip[0];
                next.axis[0] = next.axis[i], next.flip[0] = next.flip[i];
                next.axis[i] = ax, next.flip[i] = fl;
            }
        }
        const int g0 = t[0], g1 = g0 ^ t[1], g2 = g1 ^ t[2];
        next.parity = (uint8_t)(parity ^ g2);
        *below = next;
        return (g0 ^ parity) << 2 | (g1 ^ parity) << 1 | (g2 ^ parity);
    }
};

constexpr int kMaxStates = 96, kPairOctants = 64;      // (48 signed permutations, two parities)

struct CurveStates {
    CurveState s[kMaxStates] = {};
    int count = 0, odd = -1;
    constexpr int find(const CurveState& x) const {
        for (int i = 0; i < count; ++i)
            if (s[i] == x) return i;
        return -1;
    }
    constexpr CurveStates() {
        s[count++] = CurveState{{0, 1, 2}, {0, 0, 0}, 0};      // the top level's own
        for (int i = 0; i < count; ++i)
            for (int p = 0; p < 8; ++p) {
                CurveState below{};
                (void)s[i].step(p, &below);
                if (find(below) < 0) s[count++] = below;
            }
        for (int i = 0; i < count; ++i) {
            CurveState below{};
            if (s[i].step(0, &below) == 0 && below == s[0]) odd = i;
        }
    }
};
constexpr CurveStates kStates{};
constexpr int kStateCount = kStates.count, kOddStart = kStates.odd;
static_assert(kOddStart >= 0, "a zero octant leads to the first state from somewhere");

struct CurveTable {
    uint16_t entry[kStateCount * kPairOctants] = {};
    explicit constexpr CurveTable(bool decode) {
        for (int i = 0; i < kStateCount; ++i)
            for (int hi = 0; hi < 8; ++hi) {
                CurveState mid{}, end{};
                const int code_hi = kStates.s[i].step(hi, &mid);
                for (int lo = 0; lo < 8; ++lo) {
                    const int code = code_hi << 3 | mid.step(lo, &end), point = hi << 3 | lo;
                    entry[i * kPairOctants + (decode ? code : point)] =
                        (uint16_t)(kStates.find(end) * kPairOctants | (decode ? point : code));
                }
            }
    }
};
constexpr size_t kTableBytes = sizeof(CurveTable);
static_assert(kStateCount * kPairOctants <= 65536 && kTableBytes % 16 == 0, "table");
__device__ __attribute__((aligned(16))) const CurveTable g_encode_table(false), g_decode_table(true);

// The code's spatial bits for Morton codes of `bits` levels, or back, through the table in LDS: U of them side by side.
template <typename T, int U>
__device__ __forceinline__ void walk_curve(const uint16_t* table, T (&v)[U], int bits) {
    uint32_t row[U];
    T out[U];
#pragma unroll
    for (int u = 0; u < U; ++u) row[u] = bits & 1 ? kOddStart * kPairOctants : 0, out[u] = 0;
    for (int at = 3 * (bits + (bits & 1)) - 6; at >= 0; at -= 6) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const uint32_t e = table[row[u] | ((uint32_t)(v[u] >> at) & (kPairOctants - 1))];
            row[u] = e & ~(uint32_t)(kPairOctants - 1);
            out[u] = (T)(out[u] << 6) | (e & (kPairOctants - 1));
        }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = out[u];
}

template <typename T>
__host__ __device__ __forceinline__ T spatial_mask(int bits) {
    return bits == 0 ? (T)0 : (T)(~(T)0) >> (8 * sizeof(T) - 3 * bits);
}

template <typename T>
__device__ __forceinline__ T morton_of(int4 c, int bits) {
    const uint32_t keep = bits >= 32 ? 0xFFFFFFFFu : ((1u << bits) - 1u);
    const uint32_t x = (uint32_t)c.y & keep, y = (uint32_t)c.z & keep, z = (uint32_t)c.w & keep;
    return (spread3<T>((T)x) << 2) | (spread3<T>((T)y) << 1) | spread3<T>((T)z);
}

template <typename T>
__device__ __forceinline__ T with_batch(T spatial, int4 c, int bits) {
    const int shift = 3 * bits;
    const T batch = shift >= (int)(8 * sizeof(T)) ? (T)0 : (T)(uint32_t)c.x << shift;
    return (spatial & spatial_mask<T>(bits)) | batch;
}

template <typename T>
__device__ __forceinline__ int4 coords_of(T spatial, T code, int bits) {
    const uint32_t x = (uint32_t)gather3<T>(spatial >> 2), y = (uint32_t)gather3<T>(spatial >> 1), z = (uint32_t)gather3<T>(spatial);
    const int shift = 3 * bits;
    const uint32_t b = shift >= (int)(8 * sizeof(T)) ? 0u : (uint32_t)(code >> shift);
    return make_int4((int)b, (int)x, (int)y, (int)z);
}

// A thread per voxel of the z-order codes.  The Hilbert ones want their table in LDS (6 KB, read once per workgroup): no more
// workgroups than the chip holds go over the voxels.
__device__ __forceinline__ void load_table(uint16_t* table, const CurveTable& from) {
    for (int i = threadIdx.x; i < (int)(kTableBytes / 16); i += kBlock) ((uint4*)table)[i] = ((const uint4*)from.entry)[i];
    __syncthreads();
}
// Eight workgroups of four wavefronts fill a CU.  From a full chip on, three voxels a thread: three chains of dependent LDS reads side by
// side.  5.3 M voxels in random order, 32-bit codes, us encode / decode: 27.6 / 25.9 bit by bit, 18.4 / 19.9 one voxel a thread, 18.0 / 18.2
// three (5.9 TB/s), 18.4 / 18.0 four; 64-bit codes 30.0 / 28.9, 23.7 / 24.1, 21.6 / 21.6, 21.8 / 21.1; 100 000 voxels 3.0 / 2.8 and 2.5 / 2.6.
constexpr unsigned kCurveGroups = 256 * 8;
constexpr int kCurveVoxels = 3;

template <typename T, int MODE, int U>
__global__ void __launch_bounds__(kBlock) encode_kernel(const int32_t* __restrict__ coords, size_t n, int bits,
                                                        T* __restrict__ codes) {
    if constexpr (MODE == kZOrder) {
        const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
        if (i >= n) return;
        const int4 c = reinterpret_cast<const int4*>(coords)[i];
        codes[i] = with_batch<T>(morton_of<T>(c, bits), c, bits);
        return;
    }
    __shared__ __attribute__((aligned(16))) uint16_t table[kStateCount * kPairOctants];
    load_table(table, g_encode_table);
    for (size_t base = (size_t)blockIdx.x * (kBlock * U); base < n; base += (size_t)gridDim.x * (kBlock * U)) {
        int4 c[U];
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t i = base + u * kBlock + threadIdx.x;
            c[u] = reinterpret_cast<const int4*>(coords)[i < n ? i : n - 1];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = morton_of<T>(c[u], bits);
        walk_curve<T, U>(table, v, bits);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t i = base + u * kBlock + threadIdx.x;
            if (i < n) codes[i] = with_batch<T>(v[u], c[u], bits);
        }
    }
}

template <typename T, int MODE, int U>
__global__ void __launch_bounds__(kBlock) decode_kernel(const T* __restrict__ codes, size_t n, int bits,
                                                        int32_t* __restrict__ coords) {
    if constexpr (MODE == kZOrder) {
        const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
        if (i >= n) return;
        const T code = codes[i];
        reinterpret_cast<int4*>(coords)[i] = coords_of<T>(code & spatial_mask<T>(bits), code, bits);
        return;
    }
    __shared__ __attribute__((aligned(16))) uint16_t table[kStateCount * kPairOctants];
    load_table(table, g_decode_table);
    for (size_t base = (size_t)blockIdx.x * (kBlock * U); base < n; base += (size_t)gridDim.x * (kBlock * U)) {
        T code[U], v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t i = base + u * kBlock + threadIdx.x;
            code[u] = codes[i < n ? i : n - 1];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = code[u] & spatial_mask<T>(bits);
        walk_curve<T, U>(table, v, bits);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const size_t i = base + u * kBlock + threadIdx.x;
            if (i < n) reinterpret_cast<int4*>(coords)[i] = coords_of<T>(v[u], code[u], bits);
        }
    }
}

// Workgroups of U voxels a thread: all of them for the z-order codes, no more than fit the chip, and of even length, for the Hilbert ones.
unsigned groups_for(int mode, size_t n, int per_thread) {
    const unsigned all = cdiv(n, (size_t)kBlock * per_thread);
    return mode == kHilbert && all > kCurveGroups ? cdiv(all, cdiv(all, kCurveGroups)) : all;
}

template <typename T>
int launch_encode(int mode, const int32_t* coords, size_t n, int bits, T* codes, hipStream_t s) {
    if (mode == kZOrder)
        encode_kernel<T, kZOrder, 1><<<groups_for(mode, n, 1), kBlock, 0, s>>>(coords, n, bits, codes);
    else if (n < (size_t)kBlock * kCurveGroups)
        encode_kernel<T, kHilbert, 1><<<groups_for(mode, n, 1), kBlock, 0, s>>>(coords, n, bits, codes);
    else
        encode_kernel<T, kHilbert, kCurveVoxels><<<groups_for(mode, n, kCurveVoxels), kBlock, 0, s>>>(coords, n, bits, codes);
    FGX_CHECK_LAUNCH("fgx_serialize_encode");
    return FGX_OK;
}

template <typename T>
int launch_decode(int mode, const T* codes, size_t n, int bits, int32_t* coords, hipStream_t s) {
    if (mode == kZOrder)
        decode_kernel<T, kZOrder, 1><<<groups_for(mode, n, 1), kBlock, 0, s>>>(codes, n, bits, coords);
    else if (n < (size_t)kBlock * kCurveGroups)
        decode_kernel<T, kHilbert, 1><<<groups_for(mode, n, 1), kBlock, 0, s>>>(codes, n, bits, coords);
    else
        decode_kernel<T, kHilbert, kCurveVoxels><<<groups_for(mode, n, kCurveVoxels), kBlock, 0, s>>>(codes, n, bits, coords);
    FGX_CHECK_LAUNCH("fgx_serialize_decode");
    return FGX_OK;
}

int check_mode_bits(const char* who, int mode, int bit_length, int code_bits) {
    FGX_CHECK_ARG(mode == kZOrder || mode == kHilbert, "%s: mode must be 1 (z-order) or 2 (Hilbert), got %d", who, mode);
    FGX_CHECK_ARG(code_bits == 32 || code_bits == 64, "%s: code_bits must be 32 or 64, got %d", who, code_bits);
    FGX_CHECK_ARG(bit_length >= 0 && 3 * bit_length <= code_bits, "%s: bit_length %d does not fit %d-bit codes", who, bit_length,
                  code_bits);
    return FGX_OK;
}

struct ReorderLayout {
    size_t codes_a, codes_b, temp, temp_bytes, total;
};

template <typename T>
size_t sort_temp_bytes(size_t n) {
    size_t bytes = 0;
    (void)rocprim::radix_sort_keys(nullptr, bytes, (const T*)nullptr, (T*)nullptr, n ? n : 1, 0u, (unsigned)(8 * sizeof(T)),
                                   (hipStream_t)0);
    return bytes;
}

ReorderLayout reorder_layout(size_t n, int code_bits) {
    ReorderLayout L{};
    const size_t es = code_bits / 8, m = n ? n : 1;
    size_t off = 0;
    L.codes_a = off;
    off = align_up(off + m * es, 256);
    L.codes_b = off;
    off = align_up(off + m * es, 256);
    L.temp = off;
    L.temp_bytes = code_bits == 32 ? sort_temp_bytes<uint32_t>(n) : sort_temp_bytes<uint64_t>(n);
    L.total = off + align_up(L.temp_bytes, 256);
    return L;
}

template <typename T>
int reorder_impl(int mode, const int32_t* coords, size_t n, int bits, unsigned used_bits, char* ws, const ReorderLayout& L,
                 int32_t* out_coords, hipStream_t s) {
    T* a = (T*)(ws + L.codes_a);
    T* b = (T*)(ws + L.codes_b);
    int rc = launch_encode<T>(mode, coords, n, bits, a, s);
    if (rc != FGX_OK) return rc;
    size_t temp_bytes = L.temp_bytes;
    FGX_CHECK_HIP(rocprim::radix_sort_keys(ws + L.temp, temp_bytes, (const T*)a, b, n, 0u, used_bits, s));
    return launch_decode<T>(mode, b, n, bits, out_coords, s);
}

}  // namespace
}  // namespace fgx

using namespace fgx;

extern "C" {

int fgx_serialize_encode(int mode, const int32_t* coords, size_t n, int bit_length, int code_bits, void* codes,
                         fgx_stream_t stream) {
    int rc = check_mode_bits("fgx_serialize_encode", mode, bit_length, code_bits);
    if (rc != FGX_OK) return rc;
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(coords && codes, "fgx_serialize_encode: null buffer");
    FGX_CHECK_ARG(((uintptr_t)coords & 15) == 0, "fgx_serialize_encode: coords must be 16-byte aligned");
    FGX_CHECK_ARG(((uintptr_t)codes & (code_bits / 8 - 1)) == 0, "fgx_serialize_encode: codes are misaligned");
    hipStream_t s = (hipStream_t)stream;
    return code_bits == 32 ? launch_encode<uint32_t>(mode, coords, n, bit_length, (uint32_t*)codes, s)
                           : launch_encode<uint64_t>(mode, coords, n, bit_length, (uint64_t*)codes, s);
}

int fgx_serialize_decode(int mode, const void* codes, size_t n, int bit_length, int code_bits, int32_t* coords,
                         fgx_stream_t stream) {
    int rc = check_mode_bits("fgx_serialize_decode", mode, bit_length, code_bits);
    if (rc != FGX_OK) return rc;
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(coords && codes, "fgx_serialize_decode: null buffer");
    FGX_CHECK_ARG(((uintptr_t)coords & 15) == 0, "fgx_serialize_decode: coords must be 16-byte aligned");
    FGX_CHECK_ARG(((uintptr_t)codes & (code_bits / 8 - 1)) == 0, "fgx_serialize_decode: codes are misaligned");
    hipStream_t s = (hipStream_t)stream;
    return code_bits == 32 ? launch_decode<uint32_t>(mode, (const uint32_t*)codes, n, bit_length, coords, s)
                           : launch_decode<uint64_t>(mode, (const uint64_t*)codes, n, bit_length, coords, s);
}

size_t fgx_serialize_reorder_workspace_bytes(size_t n, int code_bits) {
    if (code_bits != 32 && code_bits != 64) return 0;
    return reorder_layout(n, code_bits).total;
}

int fgx_serialize_reorder_coords(int mode, const int32_t* coords, size_t n, int bit_length, int batch_bits, int code_bits,
                                 void* workspace, size_t workspace_bytes, int32_t* out_coords, fgx_stream_t stream) {
    int rc = check_mode_bits("fgx_serialize_reorder_coords", mode, bit_length, code_bits);
    if (rc != FGX_OK) return rc;
    FGX_CHECK_ARG(batch_bits >= 0 && batch_bits + 3 * bit_length <= code_bits,
                  "fgx_serialize_reorder_coords: %d batch bits + 3 * %d do not fit %d-bit codes", batch_bits, bit_length, code_bits);
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(coords && out_coords && workspace, "fgx_serialize_reorder_coords: null buffer");
    FGX_CHECK_ARG(coords != out_coords, "fgx_serialize_reorder_coords: in-place reordering is not supported");
    FGX_CHECK_ARG((((uintptr_t)coords | (uintptr_t)out_coords) & 15) == 0,
                  "fgx_serialize_reorder_coords: coordinate buffers must be 16-byte aligned");
    FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fgx_serialize_reorder_coords: workspace must be 256-byte aligned");
    const ReorderLayout L = reorder_layout(n, code_bits);
    FGX_CHECK_ARG(workspace_bytes >= L.total, "fgx_serialize_reorder_coords: workspace of %zu bytes, need %zu", workspace_bytes,
                  L.total);
    unsigned used = (unsigned)(batch_bits + 3 * bit_length);
    if (used == 0) used = 1;
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    return code_bits == 32 ? reorder_impl<uint32_t>(mode, coords, n, bit_length, used, ws, L, out_coords, s)
                           : reorder_impl<uint64_t>(mode, coords, n, bit_length, used, ws, L, out_coords, s);
}

}  // extern "C"
