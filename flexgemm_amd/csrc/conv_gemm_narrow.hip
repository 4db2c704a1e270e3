// Gather GEMM for narrow layers (16-bit types, source rows and output rows of at most 64 bytes: up to 32 channels on
// both sides) with the gathered rows RESIDENT in LDS.
//
// The streaming kernel gathers every source row once per (tile, offset): 10.5 row requests per voxel on a shell, each
// for a 64-byte row, and the memory system serves such requests at ~95 G/s whatever asks for them -- configuration 4
// (2.67 M voxels, 28.1 M pairs) cannot go below 0.29 ms that way.  Here the rows walk in chunks of 128 consecutive
// voxels of a Z-order curve; a chunk's output rows need ~220 distinct source rows (1.72 per voxel instead of 10.5), which
// a plan names once per neighbor cache.  Per chunk the loaders put those rows into LDS (direct-to-LDS loads), together
// with the chunk's table "which LDS slot holds the source of (row, offset)", and the multipliers run ALL offsets for
// all rows -- a missing neighbor is the slot of zeros -- because with K = 32 a product is two MFMAs and skipping would
// cost more instructions than it saves.  The weight (V x 2 KiB) stays in registers (3 x 3 x 3 kernels, narrow27_multiply) or LDS (others) for the
// whole launch.
//
// (the plan's layout: narrow_plan.h; the 3 x 3 x 3 kernels' walk: narrow_walk.h)
//
// Workgroup of the others: 4 multiplying wavefronts (32 chunk rows each, one 32 x 32 accumulator) + 4 loading wavefronts; two LDS
// buffers (the loads run one chunk ahead), one barrier per chunk.  Persistent: XCD x walks the x-th eighth of the chunks, its workgroups interleave, so
// that neighboring chunks -- which share their halo rows -- run on one L2 at one time.
#include "gemm_device.h"
#include "lane_swap.h"
#include "narrow_plan_build.h"
#include "narrow_walk.h"

namespace fgx {
namespace {

using rsrc_t = __amdgpu_buffer_rsrc_t;

__device__ __forceinline__ rsrc_t narrow_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

// ------------------------------------------------------------------------------------------------
// Plan builder: one workgroup per chunk (narrow_plan_build.h), from a neighbor map.
// ------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(64) narrow_plan_header_kernel(uint32_t* __restrict__ header) {
    header[threadIdx.x] = 0u;
}

// Bound by the latency of its LDS operations: with every insertion waiting for the one before it, a second walk through the table to
// find an entry again, sixteen barriers for the scan and divisions by a variable V, the plan of 2.67 M voxels took 0.271 ms; now 0.175
// (0.204 with the five wavefronts a SIMD that the compiler's own choice of registers leaves; reading the map and writing the plan take
// 0.085).  VC: V where it is 27, else 0.
template <typename Order, int VC>
__global__ void __launch_bounds__(256, VC ? 8 : 4) narrow_plan_kernel(const uint32_t* __restrict__ nmap, const Order* __restrict__ order,
                                                          uint32_t n, int v_any, int own_rows, unsigned char* __restrict__ plan) {
    const int V = VC ? VC : v_any;
    __shared__ NarrowPlanLds lds;
    const int tid = threadIdx.x;
    const uint32_t chunk = blockIdx.x;
    narrow_plan_clear<256>(lds, V);
    for (int r = tid; r < kNarrowRows; r += 256) {
        const uint32_t gr = chunk * kNarrowRows + (uint32_t)r;
        lds.grow_of[r] = gr < n ? (order ? (uint32_t)order[gr] : gr) : FGX_EMPTY32;
    }
    __syncthreads();
    narrow_plan_chunk<256, VC>(lds, V, own_rows != 0, plan, chunk, [&](int e) -> uint32_t {
        const uint32_t grow = lds.grow_of[e / V];
        if (grow == FGX_EMPTY32) return FGX_EMPTY32;
        return nmap[(size_t)grow * V + (e % V)];
    });
}

// ------------------------------------------------------------------------------------------------
// The GEMM.  LDS: weight [V][32 cols][64 B], two buffers of { rows [kNarrowSlots + 1][64 B], table, output rows },
// (a multiplier stages its output tile in its own rows of the table).  64-byte rows are kept with their four 16-byte pieces exchanged by
// (slot >> 2) & 3, so that the 32 lanes of a fragment read, which fall on arbitrary slots, spread over the banks.
// ------------------------------------------------------------------------------------------------
constexpr int kNarrowMult = 4, kNarrowLoad = 4, kNarrowThreads = 64 * (kNarrowMult + kNarrowLoad);
constexpr int kNarrowBuffers = 2;                              // chunks in LDS: one multiplied, one on its way (a third, two
                                                               // chunks ahead, measured the same)

__host__ __device__ constexpr int narrow_buffer_bytes(int V) { return kNarrowRowBufPad + kNarrowTableBytes + 1024; }
__host__ __device__ constexpr size_t narrow_lds_bytes(int V) {
    return (size_t)V * 2048 + (size_t)kNarrowBuffers * narrow_buffer_bytes(V);
}

// four fp32 values rounded (to nearest even) to four 16-bit ones
template <typename T> __device__ __forceinline__ uint64_t pack4(const float (&x)[4]);
template <> __device__ __forceinline__ uint64_t pack4<_Float16>(const float (&x)[4]) {
    using h4 = _Float16 __attribute__((ext_vector_type(4)));
    using f4 = float __attribute__((ext_vector_type(4)));
    const f4 v = {x[0], x[1], x[2], x[3]};
    return __builtin_bit_cast(uint64_t, __builtin_convertvector(v, h4));
}
template <> __device__ __forceinline__ uint64_t pack4<__bf16>(const float (&x)[4]) {
    using b4 = __bf16 __attribute__((ext_vector_type(4)));
    using f4 = float __attribute__((ext_vector_type(4)));
    const f4 v = {x[0], x[1], x[2], x[3]};
    return __builtin_bit_cast(uint64_t, __builtin_convertvector(v, b4));
}

// The order of the offsets, and the sums their products go to: with VT 27 the centre first, by halves of K, then the offsets below it to the first sum and
// those above it to the second; otherwise as they come, by halves of K.
template <int VT>
__device__ __forceinline__ constexpr int nth(int i) {
    return VT == 0 ? i : (i == 0 ? VT / 2 : (i <= VT / 2 ? i - 1 : i));
}
template <typename Tag, int VT>
__device__ __forceinline__ void add_products(int v, f32x16& acc, f32x16& acc1, const u32x4& w0, const u32x4& w1, const u32x4& a0, const u32x4& a1) {
    if (VT == 0 || v == VT / 2) {
        mma<Tag>(acc, w0, a0);
        mma<Tag>(acc1, w1, a1);
    } else if (v < VT / 2) {
        mma<Tag>(acc, w0, a0);
        mma<Tag>(acc, w1, a1);
    } else {
        mma<Tag>(acc1, w0, a0);
        mma<Tag>(acc1, w1, a1);
    }
}

// Any kernel volume, any plan: kernel volumes other than 27 (VT 0), and plans of 27 offsets that have chunks of more distinct sources than
// slots (VT 27: products in the order of narrow27_multiply, so that results do not depend on a plan's overflows).  By the first kNarrowThreads
// threads of the workgroup.
template <typename Tag, int VT>
__device__ __forceinline__ void narrow_gemm_any(const typename Tag::type* __restrict__ src, const typename Tag::type* __restrict__ panel,
                                                const typename Tag::type* __restrict__ bias, const uint32_t* __restrict__ nmap,
                                                const unsigned char* __restrict__ plan, uint32_t chunks, uint32_t plan_bytes, uint32_t src_bytes, int V,
                                                int K, int cols, int activation, typename Tag::type* __restrict__ out,
                                                uint8_t* __restrict__ relu_mask, unsigned char* lds) {
    using T = typename Tag::type;
    unsigned char* weight_lds = lds;                                            // [V][32][64 B], pieces exchanged by (col >> 2) & 3
    unsigned char* buffers = lds + (size_t)V * 2048;
    const int buffer_bytes = narrow_buffer_bytes(V);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool loader = wave >= kNarrowMult;
    const int row_bytes = K * 2, out_row_bytes = cols * 2;
    const int stride = kNarrowPlanStride, table_bytes = kNarrowTableBytes;

    // ---- chunks of this workgroup: XCD x owns the x-th eighth, its workgroups interleave ----
    const unsigned G = gridDim.x;
    const unsigned xcd = blockIdx.x % kXcds, slot_in_xcd = blockIdx.x / kXcds, per_round = G / kXcds;
    const unsigned per_xcd = (chunks + kXcds - 1) / kXcds;
    const unsigned range_lo = xcd * per_xcd, range_hi = (xcd + 1) * per_xcd < chunks ? (xcd + 1) * per_xcd : chunks;
    const unsigned first = range_lo + slot_in_xcd;

    // ---- once: the weight into LDS, zeros into the zero slot of both buffers ----
    for (int u = tid; u < V * 128; u += kNarrowThreads) {                        // 16-byte pieces: [v][col][piece]
        const int col = (u >> 2) & 31, piece = u & 3;
        const u32x4 w = *reinterpret_cast<const u32x4*>((const unsigned char*)panel + (size_t)u * 16);
        *reinterpret_cast<u32x4*>(weight_lds + (u >> 2) * 64 + ((piece ^ ((col >> 2) & 3)) << 4)) = w;
    }
    if (tid < 4 * kNarrowBuffers) {
        const u32x4 zero = {0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4*>(buffers + (size_t)(tid >> 2) * buffer_bytes + kNarrowSlots * 64 + (tid & 3) * 16) = zero;
    }
    if (first >= range_hi) return;                                              // whole workgroup

    const rsrc_t src_rs = narrow_rsrc(src, src_bytes);
    const rsrc_t plan_rs = narrow_rsrc(plan, plan_bytes);

    // Loaders: wavefront lw issues, per chunk, the row loads of the slot groups (j * 4 + lw) * 16 ... + 15 (j = 0 ... 5),
    // every fourth KiB of the table, and (lw == 3) the output rows.  The source rows of the chunk after next are fetched
    // into registers while the current loads fly.
    const int lw = loader ? wave - kNarrowMult : 0;
    constexpr int kGroups = kNarrowSlots / 16 / kNarrowLoad;                     // 6
    uint32_t ids[kGroups];
    auto fetch_ids = [&](unsigned chunk) {
#pragma unroll
        for (int j = 0; j < kGroups; ++j) {
            const uint32_t s = (uint32_t)((j * kNarrowLoad + lw) * 16 + (lane >> 2));
            ids[j] = __builtin_amdgcn_raw_buffer_load_b32(plan_rs, (uint32_t)kNarrowHeader + chunk * (uint32_t)stride + (uint32_t)table_bytes + s * 4u, 0, 0);
        }
    };
    auto enqueue = [&](unsigned chunk, int b) {
        unsigned char* buf = buffers + (size_t)b * buffer_bytes;
#pragma unroll
        for (int j = 0; j < kGroups; ++j) {
            const int group = j * kNarrowLoad + lw;
            const uint32_t s = (uint32_t)(group * 16 + (lane >> 2));
            const uint32_t piece = (uint32_t)(lane & 3) ^ ((s >> 2) & 3u);       // LDS position lane & 3 holds this piece
            const bool live = ids[j] != FGX_EMPTY32 && (int)(piece * 16) < row_bytes;
            const uint32_t vo = live ? ids[j] * (uint32_t)row_bytes + piece * 16u : kNarrowOob;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src_rs, FGX_LDS_PTR(buf + group * 1024), 16, vo, 0, 0, 0);
        }
        const int table_insts = kNarrowTableBytes / 1024;
        for (int j = lw; j < table_insts; j += kNarrowLoad)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(plan_rs, FGX_LDS_PTR(buf + kNarrowRowBufPad + j * 1024), 16,
                                                     (uint32_t)kNarrowHeader + chunk * (uint32_t)stride + (uint32_t)(j * 1024 + lane * 16), 0, 0, 0);
        if (lw == kNarrowLoad - 1) {
            const uint32_t vo = lane < kNarrowRows * 4 / 16
                                    ? (uint32_t)kNarrowHeader + chunk * (uint32_t)stride + (uint32_t)table_bytes + kNarrowSlots * 4u + (uint32_t)lane * 16u
                                    : kNarrowOob;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(plan_rs, FGX_LDS_PTR(buf + kNarrowRowBufPad + kNarrowTableBytes), 16, vo, 0, 0, 0);
        }
    };

    // Multipliers: wavefront mw owns chunk rows mw * 32 ... + 31.
    const int mw = loader ? 0 : wave;
    const int l32 = lane & 31, g = lane >> 5;
    float bias_e[16];                                                           // accumulator element e is column ...
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int col = (e >> 2) * 8 + g * 4 + (e & 3);
        bias_e[e] = (bias != nullptr && col < cols) ? to_float<T>(bias[col]) : 0.f;
    }

    // One chunk ahead: in the iteration that multiplies chunk i the loaders enqueue chunk i + 1 (its source rows are in
    // registers since the iteration before) and fetch the source rows of chunk i + 2; at the end of the iteration they
    // wait until chunk i + 1 has landed -- everything but the fetch, which was issued last (loads return in order).
    if (loader) {
        fetch_ids(first);
        enqueue(first, 0);
        if (first + per_round < range_hi) fetch_ids(first + per_round);
    }
    __builtin_amdgcn_s_waitcnt(0);                                              // the weight and zero stores, the first loads
    __syncthreads();

    int b = 0;
    for (unsigned chunk = first; chunk < range_hi; chunk += per_round, b ^= 1) {
        if (loader) {
            const unsigned next = chunk + per_round;
            const bool enqueues = next < range_hi, fetches = next + per_round < range_hi;
            if (enqueues) {
                enqueue(next, b ^ 1);
                if (fetches) fetch_ids(next + per_round);
            }
            if (fetches) wait_vmcnt<kGroups>();
            else wait_vmcnt<0>();
        } else {
            const unsigned char* buf = buffers + (size_t)b * buffer_bytes;
            const uint16_t* table = (const uint16_t*)(buf + kNarrowRowBufPad);
            const uint32_t* out_rows = (const uint32_t*)(buf + kNarrowRowBufPad + kNarrowTableBytes);
            const int r = mw * 32 + l32;
            // Products are taken as (weight fragment) x (row fragment): the accumulator then holds, per lane, ONE chunk row
            // (r) and sixteen output columns in four runs of four -- 8 bytes each, stored straight from the registers.
            // One accumulator per half of K (sums in a fixed order, like everything here).
            f32x16 acc, acc1;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = acc1[e] = 0.f;
            // this row's table entries: 32 x uint16 in four 16-byte reads; entry 31 says whether any of them is kNarrowOverflow
            u32x4 ent[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) ent[q] = *reinterpret_cast<const u32x4*>((const unsigned char*)table + r * (kNarrowTableStride * 2) + q * 16);
            auto entry = [&](int v) -> uint32_t {
                const uint32_t word = ent[v >> 3][(v >> 1) & 3];
                return (v & 1) ? word >> 16 : word & 0xFFFFu;
            };
            const uint32_t grow = out_rows[r];
            const uint32_t wkey = ((uint32_t)l32 >> 2) & 3u;
            const unsigned char* wrow0 = weight_lds + l32 * 64 + (((uint32_t)g ^ wkey) << 4);
            const unsigned char* wrow1 = weight_lds + l32 * 64 + (((uint32_t)(g + 2) ^ wkey) << 4);
            // (a table entry is the byte offset of a row's logical piece 0; piece q sits at entry ^ (q << 4))
            if (__builtin_expect(__any(entry(kNarrowTableStride - 1) != 0u), 0)) {
                // a chunk with more distinct sources than slots: lanes whose source is not resident read it from memory
                for (int i = 0; i < V; ++i) {
                    const int v = nth<VT>(i);
                    const uint32_t s = table[r * kNarrowTableStride + v];
                    const uint32_t off = s == kNarrowOverflow ? kNarrowZeroSlot * 64u : s;
                    u32x4 a0 = *reinterpret_cast<const u32x4*>(buf + (off ^ ((uint32_t)g << 4)));
                    u32x4 a1 = *reinterpret_cast<const u32x4*>(buf + (off ^ ((uint32_t)g << 4) ^ 32u));
                    if (s == kNarrowOverflow && grow != FGX_EMPTY32) {
                        const uint32_t id = nmap[(size_t)grow * V + v];
                        if (id != FGX_EMPTY32) {
                            const u32x4 zero = {0u, 0u, 0u, 0u};
                            const unsigned char* p = (const unsigned char*)src + (size_t)id * row_bytes;
                            a0 = g * 16 < row_bytes ? *reinterpret_cast<const u32x4*>(p + g * 16) : zero;
                            a1 = (g + 2) * 16 < row_bytes ? *reinterpret_cast<const u32x4*>(p + (g + 2) * 16) : zero;
                        }
                    }
                    add_products<Tag, VT>(v, acc, acc1, *reinterpret_cast<const u32x4*>(wrow0 + v * 2048), *reinterpret_cast<const u32x4*>(wrow1 + v * 2048), a0, a1);
                }
            } else if constexpr (VT > 0) {
                // The fragment reads run kFetched offsets ahead of the products (kFetched + 1 register sets): with one multiplying
                // wavefront per SIMD nothing else hides the LDS latency, and left to itself the compiler issues every
                // read right before its use.
                constexpr int kFetched = 2, kSets = kFetched + 1;    // (3, 4 and 6 ahead measure the same)
                u32x4 fa0[kSets], fa1[kSets], fb0[kSets], fb1[kSets];
                auto fetch = [&](int v, int set) __attribute__((always_inline)) {
                    const uint32_t at = entry(v) ^ ((uint32_t)g << 4);
                    fa0[set] = *reinterpret_cast<const u32x4*>(buf + at);
                    fa1[set] = *reinterpret_cast<const u32x4*>(buf + (at ^ 32u));
                    fb0[set] = *reinterpret_cast<const u32x4*>(wrow0 + v * 2048);
                    fb1[set] = *reinterpret_cast<const u32x4*>(wrow1 + v * 2048);
                };
#pragma unroll
                for (int i = 0; i < kFetched && i < VT; ++i) fetch(nth<VT>(i), i % kSets);
#pragma unroll
                for (int i = 0; i < VT; ++i) {
                    if (i + kFetched < VT) fetch(nth<VT>(i + kFetched), (i + kFetched) % kSets);
                    __builtin_amdgcn_sched_barrier(0);
                    add_products<Tag, VT>(nth<VT>(i), acc, acc1, fb0[i % kSets], fb1[i % kSets], fa0[i % kSets], fa1[i % kSets]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll 4
                for (int v = 0; v < V; ++v) {
                    const uint32_t at = (uint32_t)table[r * kNarrowTableStride + v] ^ ((uint32_t)g << 4);
                    const u32x4 a0 = *reinterpret_cast<const u32x4*>(buf + at);
                    const u32x4 a1 = *reinterpret_cast<const u32x4*>(buf + (at ^ 32u));
                    mma<Tag>(acc, *reinterpret_cast<const u32x4*>(wrow0 + v * 2048), a0);
                    mma<Tag>(acc1, *reinterpret_cast<const u32x4*>(wrow1 + v * 2048), a1);
                }
            }
            // epilogue: accumulator element e is column (e >> 2) * 8 + g * 4 + (e & 3) of chunk row r
            if (grow != FGX_EMPTY32) {
                unsigned char* orow = (unsigned char*)out + (size_t)grow * out_row_bytes;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int col0 = i * 8 + g * 4;
                    if (i * 8 < cols) {                                          // cols is a multiple of 8: whole pieces
                        float x[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j) x[j] = activate(acc[i * 4 + j] + acc1[i * 4 + j] + bias_e[i * 4 + j], activation);
                        const uint64_t packed = pack4<T>(x);
                        *reinterpret_cast<uint64_t*>(orow + col0 * 2) = packed;
                        if (relu_mask != nullptr) {
                            // the piece's other four columns are in lane ^ 32
                            uint32_t bits = 0;
#pragma unroll
                            for (int j = 0; j < 4; ++j) bits |= (x[j] > 0.f ? 1u : 0u) << j;
                            const uint32_t other = (uint32_t)__shfl_xor((int)bits, 32, 64);
                            if (g == 0) relu_mask[((size_t)grow * out_row_bytes >> 4) + i] = (uint8_t)(bits | (other << 4));
                        }
                    }
                }
            }
        }
        if (!loader) __builtin_amdgcn_s_waitcnt(0);          // the stage has been read, the output is on its way
        __syncthreads();
    }
}

template <typename Tag>
__global__ void __launch_bounds__(kNarrowThreads)
narrow_gemm_kernel(const typename Tag::type* __restrict__ src, const typename Tag::type* __restrict__ panel,
                   const typename Tag::type* __restrict__ bias, const uint32_t* __restrict__ nmap,
                   const unsigned char* __restrict__ plan, uint32_t chunks, uint32_t plan_bytes, uint32_t src_bytes, int V,
                   int K, int cols, int activation, typename Tag::type* __restrict__ out, uint8_t* __restrict__ relu_mask) {
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    narrow_gemm_any<Tag, 0>(src, panel, bias, nmap, plan, chunks, plan_bytes, src_bytes, V, K, cols, activation, out, relu_mask, lds);
}

// 3 x 3 x 3 kernels.  Eight multipliers: wavefront h * 4 + t has chunk rows t * 32 ... + 31 and the offsets below (h = 0) or above the
// centre, whose product the two share by halves of K: 27 matrix instructions each.  The weight of a wavefront's offsets stays in
// its registers for the launch.  The two sums of a row meet through LDS:
// a wavefront hands over the sums of one half of its rows and finishes the other's, at the start of the next iteration, when the barrier
// between the two has been met anyway; the 16 x 32 sums a wavefront finishes leave as one store of whole 64-byte rows.
// 2 667 120 voxels, 32 channels: 0.182 ms -> 0.152 in scan order, 0.191 -> 0.160 in random order; 166 977 voxels 17.9 -> 15.9 us; 667 763 voxels, 16
// channels 39.3 -> 35.9; 8 and 16 channels up to 90 000 rows, a chunk or two a workgroup, wait for the longer start, 10.2 -> 10.6.  Loads and stores alone take 0.117 ms (582 MB at 5 TB/s, 219 of them the plan); what is left are the two multipliers of a
// SIMD, which do not cover each other's waits altogether.  Leaving out the offsets that none of a tile's 32 rows has (7 of 27) costs in
// branches what it saves in products; registers for a second offset's fragments ahead change nothing.
constexpr int kAhead = 1;                                      // (offsets whose fragments are read ahead: registers for one)
constexpr int kN27Half = 13;                                   // offsets on either side of the centre
constexpr int kN27BufferBytes = kNarrowRowBufPad + kNarrowTableBytes;
constexpr int kN27SumBytes = 16 * 32 * 4;                      // what a wavefront hands over
constexpr size_t kN27LdsBytes = (size_t)kWalkBuffers * kN27BufferBytes + 2 * (size_t)kWalkMult * kN27SumBytes + (size_t)kWalkMetas * kWalkMetaBytes + 128 + 2048;
static_assert(kN27LdsBytes <= 160 * 1024 && narrow_lds_bytes(kNarrowCubeV) <= kN27LdsBytes, "LDS, also of narrow_gemm_any");

// The offsets below the centre (HALF 0) or above it.
template <typename Tag, int HALF>
__device__ __forceinline__ void narrow27_multiply(const NarrowWalk& walk, int t, int lane, const unsigned char* panel, const unsigned char* buffers,
                                                  unsigned char* handed, const unsigned char* meta, const float* bias_lds,
                                                  const unsigned char* centre_lds, int cols, int activation, unsigned char* out, uint8_t* relu_mask) {
    using T = typename Tag::type;
    constexpr int CENTRE = kNarrowCubeV / 2;
    const int out_row_bytes = cols * 2;
    const int l32 = lane & 31, g = lane >> 5, r = t * 32 + l32;
    const int piece = ((lane >> 4) & 1) * 2 + g;                               // of a finished row: columns 8 * piece ... + 7 of row lane % 16
    constexpr int FIRST = HALF == 0 ? 0 : CENTRE + 1;
    u32x4 wf[kN27Half][2];
    {
        const unsigned char* w = panel + l32 * 64 + g * 16;
#pragma unroll
        for (int i = 0; i < kN27Half; ++i) {
            wf[i][0] = *reinterpret_cast<const u32x4*>(w + (FIRST + i) * 2048);
            wf[i][1] = *reinterpret_cast<const u32x4*>(w + (FIRST + i) * 2048 + 32);
        }
    }
    const unsigned char* centre_at = centre_lds + l32 * 64 + (((g + 2 * HALF) ^ ((l32 >> 2) & 3)) << 4);
    unsigned char* mine_out = handed + (HALF * 4 + t) * kN27SumBytes + lane * 16;              // [2][64 lanes][16 bytes]
    const unsigned char* other_in = handed + ((HALF ^ 1) * 4 + t) * kN27SumBytes + lane * 16;
    float kept[8];
    uint32_t kept_row = FGX_EMPTY32;
    // the rows whose sums this wavefront finishes: 16 * HALF ... + 15 of its 32
    auto finish = [&](int parity) __attribute__((always_inline)) {
        const f32x4 o0 = *reinterpret_cast<const f32x4*>(other_in + parity * (kWalkMult * kN27SumBytes));
        const f32x4 o1 = *reinterpret_cast<const f32x4*>(other_in + parity * (kWalkMult * kN27SumBytes) + 1024);
        const f32x4 b0 = *reinterpret_cast<const f32x4*>(bias_lds + piece * 8), b1 = *reinterpret_cast<const f32x4*>(bias_lds + piece * 8 + 4);
        float x[2][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            // (offsets below the centre first, whoever adds)
            x[0][e] = activate((HALF == 0 ? kept[e] + o0[e] : o0[e] + kept[e]) + b0[e], activation);
            x[1][e] = activate((HALF == 0 ? kept[4 + e] + o1[e] : o1[e] + kept[4 + e]) + b1[e], activation);
        }
        if (kept_row == FGX_EMPTY32 || piece * 8 >= cols) return;
        const uint64_t p0 = pack4<T>(x[0]), p1 = pack4<T>(x[1]);
        const u32x4 out16 = {(uint32_t)p0, (uint32_t)(p0 >> 32), (uint32_t)p1, (uint32_t)(p1 >> 32)};
        *reinterpret_cast<u32x4*>(out + (size_t)kept_row * out_row_bytes + piece * 16) = out16;
        if (relu_mask != nullptr) {
            uint32_t bits = 0;
#pragma unroll
            for (int e = 0; e < 4; ++e) bits |= (x[0][e] > 0.f ? 1u : 0u) << e | (x[1][e] > 0.f ? 16u : 0u) << e;
            relu_mask[((size_t)kept_row * out_row_bytes >> 4) + piece] = (uint8_t)bits;
        }
    };

    walk_barrier();
    walk_barrier();
    for (unsigned i = 0; i < walk.count; ++i) {
        if (i > 0) finish((int)(i & 1) ^ 1);
        const unsigned char* buf = buffers + (i % kWalkBuffers) * kN27BufferBytes;
        const unsigned char* table = buf + kNarrowRowBufPad;
        const uint32_t* out_rows = (const uint32_t*)(meta + (i % kWalkMetas) * kWalkMetaBytes) + kNarrowSlots;
        // entries: pieces 0 and 1, or 1, 2 and 3
        u32x4 ent[2 + HALF];
#pragma unroll
        for (int q = 0; q < 2 + HALF; ++q) ent[q] = *reinterpret_cast<const u32x4*>(table + walk_table_at(r, HALF + q));
        kept_row = out_rows[t * 32 + HALF * 16 + (lane & 15)];
        auto entry = [&](int v) __attribute__((always_inline)) -> uint32_t {
            const uint32_t word = ent[(v >> 3) - HALF][(v >> 1) & 3];
            return (v & 1) ? word >> 16 : word & 0xFFFFu;
        };
        f32x16 acc;
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[e] = 0.f;
        // The fragments of kAhead offsets are read ahead of the products; the centre comes first.
        u32x4 a0[kAhead + 1], a1[kAhead + 1];
        auto fetch = [&](int j) __attribute__((always_inline)) {                 // 0: the centre (one half of K), j: the half's j-th offset
            const uint32_t at = entry(j == 0 ? CENTRE : FIRST + j - 1) ^ ((uint32_t)(j == 0 ? g + 2 * HALF : g) << 4);
            a0[j % (kAhead + 1)] = *reinterpret_cast<const u32x4*>(buf + at);
            if (j == 0) a1[0] = *reinterpret_cast<const u32x4*>(centre_at);
            else a1[j % (kAhead + 1)] = *reinterpret_cast<const u32x4*>(buf + (at ^ 32u));
        };
#pragma unroll
        for (int j = 0; j < kAhead; ++j) fetch(j);
#pragma unroll
        for (int j = 0; j <= kN27Half; ++j) {
            if (j + kAhead <= kN27Half) fetch(j + kAhead);
            __builtin_amdgcn_sched_barrier(0);
            if (j == 0) {
                mma<Tag>(acc, a1[0], a0[0]);
            } else {
                mma<Tag>(acc, wf[j - 1][0], a0[j % (kAhead + 1)]);
                mma<Tag>(acc, wf[j - 1][1], a1[j % (kAhead + 1)]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // element e of lane l: column 8 * (e / 4) + 4 * (l / 32) + e % 4 of row l % 32  ->  eight columns of row l % 16 and of row 16 + l % 16
        float x[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = acc[e];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            swap_halves(x[e], x[4 + e]);
            swap_halves(x[8 + e], x[12 + e]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) swap_rows(x[e], x[8 + e]);
        unsigned char* to = mine_out + (i & 1) * (kWalkMult * kN27SumBytes);
#pragma unroll
        for (int e = 0; e < 8; ++e) kept[e] = x[HALF * 8 + e];
        constexpr int GIVEN = 8 - HALF * 8;
        *reinterpret_cast<f32x4*>(to) = f32x4{x[GIVEN], x[GIVEN + 1], x[GIVEN + 2], x[GIVEN + 3]};
        *reinterpret_cast<f32x4*>(to + 1024) = f32x4{x[GIVEN + 4], x[GIVEN + 5], x[GIVEN + 6], x[GIVEN + 7]};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                 // handed over; the buffers have been read
        walk_barrier();
    }
    finish((int)(walk.count & 1) ^ 1);
}

template <typename Tag>
__global__ void __launch_bounds__(kWalkThreads)
narrow_gemm27_kernel(const typename Tag::type* __restrict__ src, const typename Tag::type* __restrict__ panel,
                     const typename Tag::type* __restrict__ bias, const uint32_t* __restrict__ nmap, const unsigned char* __restrict__ plan,
                     uint32_t chunks, uint32_t plan_bytes, uint32_t src_bytes, int K, int cols, int activation,
                     typename Tag::type* __restrict__ out, uint8_t* __restrict__ relu_mask) {
    using T = typename Tag::type;
    constexpr int V = kNarrowCubeV;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    unsigned char* buffers = lds;
    unsigned char* handed = lds + kWalkBuffers * kN27BufferBytes;              // [2][kWalkMult][kN27SumBytes]
    unsigned char* meta = handed + 2 * kWalkMult * kN27SumBytes;
    float* bias_lds = (float*)(meta + kWalkMetas * kWalkMetaBytes);            // [32]
    unsigned char* centre_lds = (unsigned char*)(bias_lds + 32);               // the centre's weight (registers for it as well are not left): [32][64 bytes]
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row_bytes = K * 2;
    // One chunk with sources that are not resident sends all of them to the four multipliers: reading such sources from memory wants registers that the
    // weight takes here.  32 channels, forward and weight gradient, a solid cube of 20 cells a side in the middle of the surface: 2.67 M voxels
    // 176 -> 209 us and 180 -> 367 (the weight gradient's kernel is another one then), 167 000 voxels 24 -> 40 and 27 -> 47.
    if (*reinterpret_cast<const uint32_t*>(plan) != 0u) {
        if (tid < kNarrowThreads)
            narrow_gemm_any<Tag, V>(src, panel, bias, nmap, plan, chunks, plan_bytes, src_bytes, V, K, cols, activation, out, relu_mask, lds);
        return;
    }
    const NarrowWalk walk(chunks, kXcds);
    if (walk.count == 0) return;                                               // whole workgroup
    if (tid < 4 * kWalkBuffers) {                                              // the rows of zeros
        const u32x4 zero = {0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4*>(buffers + (tid >> 2) * kN27BufferBytes + kNarrowSlots * 64 + (tid & 3) * 16) = zero;
    }
    if (tid >= 64 && tid < 96) bias_lds[tid - 64] = bias != nullptr && tid - 64 < cols ? to_float<T>(bias[tid - 64]) : 0.f;
    if (tid >= 128 && tid < 256) {
        const int col = (tid - 128) >> 2, piece = tid & 3;
        *reinterpret_cast<u32x4*>(centre_lds + col * 64 + ((piece ^ ((col >> 2) & 3)) << 4)) =
            *reinterpret_cast<const u32x4*>((const unsigned char*)panel + (V / 2) * 2048 + col * 64 + piece * 16);
    }
    const rsrc_t src_rs = narrow_rsrc(src, src_bytes), plan_rs = narrow_rsrc(plan, plan_bytes);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                         // (met by the barriers of the walk)

    if (wave >= kWalkMult) {
        narrow_load_walk<false, true>(walk, wave - kWalkMult, lane, src_rs, row_bytes, src_rs, 0, plan_rs, buffers, kN27BufferBytes, kNarrowRowBufPad, meta);
        return;
    }

    unsigned char* out_b = (unsigned char*)out;
    const unsigned char* panel_b = (const unsigned char*)panel;
    // (of two wavefronts on a SIMD the older one wins, and the younger would be late at every barrier: 2.67 M rows in random order 0.167 -> 0.160 ms)
    if (wave >= 4) __builtin_amdgcn_s_setprio(1);
    if (wave < 4) narrow27_multiply<Tag, 0>(walk, wave, lane, panel_b, buffers, handed, meta, bias_lds, centre_lds, cols, activation, out_b, relu_mask);
    else narrow27_multiply<Tag, 1>(walk, wave - 4, lane, panel_b, buffers, handed, meta, bias_lds, centre_lds, cols, activation, out_b, relu_mask);
}

template <typename Tag>
int launch_narrow(const void* src, const void* panel, const void* bias, const uint32_t* nmap, const void* plan, size_t n,
                  size_t n_src, int V, int K, int cols, int activation, void* out, uint8_t* relu_mask, hipStream_t s) {
    using T = typename Tag::type;
    const uint32_t chunks = (uint32_t)((n + kNarrowRows - 1) / kNarrowRows);
    int dev = 0, cus = 0;
    FGX_CHECK_HIP(hipGetDevice(&dev));
    FGX_CHECK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    unsigned groups = (unsigned)(cus > 0 ? cus : 256);
    groups = groups / kXcds * kXcds;
    if (groups < (unsigned)kXcds) groups = kXcds;
    static thread_local bool raised = false;
    if (!raised) {
        FGX_CHECK_HIP(hipFuncSetAttribute((const void*)narrow_gemm27_kernel<Tag>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        FGX_CHECK_HIP(hipFuncSetAttribute((const void*)narrow_gemm_kernel<Tag>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        raised = true;
    }
    if (V == kNarrowCubeV) {
        narrow_gemm27_kernel<Tag><<<groups, kWalkThreads, kN27LdsBytes, s>>>(
            (const T*)src, (const T*)panel, (const T*)bias, nmap, (const unsigned char*)plan, chunks,
            (uint32_t)(kNarrowHeader + (size_t)chunks * kNarrowPlanStride), (uint32_t)(n_src * (size_t)K * 2), K, cols, activation, (T*)out, relu_mask);
        FGX_CHECK_LAUNCH("fgx_conv_narrow_gemm");
        return FGX_OK;
    }
    const size_t lds = narrow_lds_bytes(V);
    narrow_gemm_kernel<Tag><<<groups, kNarrowThreads, lds, s>>>((const T*)src, (const T*)panel, (const T*)bias, nmap, (const unsigned char*)plan, chunks,
                                             (uint32_t)(kNarrowHeader + (size_t)chunks * kNarrowPlanStride), (uint32_t)(n_src * (size_t)K * 2), V, K,
                                             cols, activation, (T*)out, relu_mask);
    FGX_CHECK_LAUNCH("fgx_conv_narrow_gemm");
    return FGX_OK;
}

template <typename Order>
int make_narrow_plan(const uint32_t* map, const Order* order, size_t n, int V, int same_rows, void* plan, hipStream_t s) {
    FGX_CHECK_ARG(V >= 1 && V <= kNarrowMaxV, "fgx_narrow_plan: bad kernel volume %d", V);
    FGX_CHECK_ARG(n < 0xFFFFFFFFull, "fgx_narrow_plan: too many rows");
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(map && plan, "fgx_narrow_plan: null buffer");
    FGX_CHECK_ARG(((uintptr_t)plan & 15) == 0, "fgx_narrow_plan: plan must be 16-byte aligned");
    FGX_CHECK_ARG(fgx_narrow_plan_bytes(n, V) < 0xFF000000ull, "fgx_narrow_plan: plan of %zu rows passes the 32-bit offset range", n);
    const unsigned chunks = (unsigned)((n + kNarrowRows - 1) / kNarrowRows);
    narrow_plan_header_kernel<<<1, 64, 0, s>>>((uint32_t*)plan);
    FGX_CHECK_LAUNCH("fgx_narrow_plan(header)");
    auto kern = V == kNarrowCubeV ? narrow_plan_kernel<Order, kNarrowCubeV> : narrow_plan_kernel<Order, 0>;
    kern<<<chunks, 256, 0, s>>>(map, order, (uint32_t)n, V, same_rows ? 1 : 0, (unsigned char*)plan);
    FGX_CHECK_LAUNCH("fgx_narrow_plan");
    return FGX_OK;
}

}  // namespace
}  // namespace fgx

using namespace fgx;

extern "C" {

size_t fgx_narrow_plan_bytes(size_t n, int V) {
    if (V < 1 || V > kNarrowMaxV) return 0;
    return kNarrowHeader + ((n + kNarrowRows - 1) / kNarrowRows) * (size_t)kNarrowPlanStride;
}

int fgx_narrow_plan(const uint32_t* map, const int64_t* order, size_t n, int V, int same_rows, void* plan, fgx_stream_t stream) {
    return make_narrow_plan(map, order, n, V, same_rows, plan, (hipStream_t)stream);
}

int fgx_narrow_plan_walk(const uint32_t* map, const uint32_t* walk, size_t n, int V, void* plan, fgx_stream_t stream) {
    return make_narrow_plan(map, walk, n, V, 1, plan, (hipStream_t)stream);
}

int fgx_conv_narrow_gemm(int dtype, const void* src, const void* panel, const void* bias, const uint32_t* map, const void* plan,
                         size_t n, size_t n_src, int K, int cols, int V, int activation, void* out, uint8_t* relu_mask,
                         fgx_stream_t stream) {
    FGX_CHECK_ARG(dtype == FGX_F16 || dtype == FGX_BF16, "fgx_conv_narrow_gemm: 16-bit types only, got dtype %d", dtype);
    FGX_CHECK_ARG(V >= 1 && V <= kNarrowMaxV, "fgx_conv_narrow_gemm: bad kernel volume %d", V);
    FGX_CHECK_ARG(K >= 8 && K <= 32 && K % 8 == 0 && cols >= 8 && cols <= 32 && cols % 8 == 0,
                  "fgx_conv_narrow_gemm: K = %d and cols = %d must be 8, 16, 24 or 32", K, cols);
    FGX_CHECK_ARG(activation == FGX_ACT_NONE || activation == FGX_ACT_RELU, "fgx_conv_narrow_gemm: unknown activation %d", activation);
    FGX_CHECK_ARG(n < 0xFFFFFFFFull && (double)n_src * K * 2 < (double)0xFF000000u, "fgx_conv_narrow_gemm: operand too large for 32-bit offsets");
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(src && panel && map && plan && out, "fgx_conv_narrow_gemm: null buffer");
    FGX_CHECK_ARG((((uintptr_t)src | (uintptr_t)panel | (uintptr_t)out | (uintptr_t)plan) & 15) == 0, "fgx_conv_narrow_gemm: buffers must be 16-byte aligned");
    FGX_CHECK_ARG(fgx_narrow_plan_bytes(n, V) < 0xFF000000ull, "fgx_conv_narrow_gemm: plan passes the 32-bit offset range");
    FGX_CHECK_ARG(narrow_lds_bytes(V) <= 160 * 1024, "fgx_conv_narrow_gemm: kernel volume %d does not fit LDS", V);
    hipStream_t s = (hipStream_t)stream;
    if (dtype == FGX_F16) return launch_narrow<F16>(src, panel, bias, map, plan, n, n_src, V, K, cols, activation, out, relu_mask, s);
    return launch_narrow<BF16>(src, panel, bias, map, plan, n, n_src, V, K, cols, activation, out, relu_mask, s);
}

}  // extern "C"
