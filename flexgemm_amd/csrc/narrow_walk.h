// What the 3x3x3 kernels for narrow layers (conv_gemm_narrow.hip: forward and dgrad; wgrad_narrow.hip: weight gradient) share: the chunks
// of a workgroup and the loading wavefronts' walk over them.
//
// A workgroup has eight multiplying wavefronts (weight gradient: seven), two per SIMD, and four that only load.  With one multiplier per SIMD its
// products, its address arithmetic, its waits for LDS and its stores stood in a row (figures: narrow_gemm27_kernel, narrow_wgrad27_kernel).
//
// Two chunks are on their way while one is multiplied.  A chunk's source and output row numbers (its "meta": the plan's sources and rows)
// come two chunks earlier still, through a ring of their own in LDS: row numbers in registers would make the loads that need them wait for
// every load issued before.  Everything a loader issues, the chunk before last included, has landed when at most what it issued in the
// current iteration is still on its way.
//
//   iteration i (the multipliers have chunk i)          buffer of a chunk: chunk % kWalkBuffers
//     rows and table of chunk i + 2 go out              (the buffer of chunk i - 1)
//     meta of chunk i + 4 goes out                      (the slot of chunk i - 1, whose output rows the multipliers have read)
//     wait for what iteration i - 1 issued: rows and table of chunk i + 1, meta of chunk i + 3;  barrier
#pragma once
#include "narrow_plan.h"

namespace fgx {
namespace {

constexpr int kWalkMult = 8, kWalkLoad = 4, kWalkThreads = 64 * (kWalkMult + kWalkLoad);
constexpr int kWalkBuffers = 3, kWalkMetas = 5;
constexpr int kWalkMetaBytes = kNarrowSlots * 4 + kNarrowRows * 4;
constexpr int kWalkSrcGroups = kNarrowSlots / 16 / kWalkLoad;                    // wave-wide row loads per loader
constexpr int kWalkOutGroups = kNarrowRows / 16 / kWalkLoad;
constexpr int kWalkTableLoads = kNarrowTableBytes / 1024 / kWalkLoad;

// Chunks of a workgroup: XCD x owns the x-th eighth, its workgroups interleave, so that neighboring chunks -- which share their halo rows -- run on one L2 at
// one time.
struct NarrowWalk {
    unsigned first, step, count;
    __device__ __forceinline__ NarrowWalk(uint32_t chunks, unsigned xcds) {
        const unsigned xcd = blockIdx.x % xcds, slot_in_xcd = blockIdx.x / xcds, per_xcd = (chunks + xcds - 1) / xcds;
        const unsigned lo = xcd * per_xcd, hi = (xcd + 1) * per_xcd < chunks ? (xcd + 1) * per_xcd : chunks;
        step = gridDim.x / xcds;
        first = lo + slot_in_xcd;
        count = first < hi ? (hi - first + step - 1) / step : 0;
    }
    __device__ __forceinline__ uint32_t plan_at(unsigned i) const { return (uint32_t)kNarrowHeader + (first + i * step) * (uint32_t)kNarrowPlanStride; }
};

// (__syncthreads() would also wait for the loads in flight)
__device__ __forceinline__ void walk_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Where table piece q (16 bytes, eight entries) of chunk row r sits in LDS, if the walk exchanges the pieces (SWIZZLE): 16 rows' reads of one piece
// fall on distinct banks.
__device__ __forceinline__ uint32_t walk_table_at(int r, int q) { return (uint32_t)(r * (kNarrowTableStride * 2) + ((q ^ ((r >> 2) & 3)) << 4)); }

// The loaders' side of a pass: two barriers, then one per chunk.  buffers: [kWalkBuffers] of buffer_bytes (rows | grad_out rows with
// OUT_ROWS | table at table_off), meta: [kWalkMetas] of kWalkMetaBytes.
template <bool OUT_ROWS, bool SWIZZLE>
__device__ __forceinline__ void narrow_load_walk(const NarrowWalk& w, int lw, int lane, __amdgpu_buffer_rsrc_t src_rs, int src_row_bytes, __amdgpu_buffer_rsrc_t out_rs,
                                                 int out_row_bytes, __amdgpu_buffer_rsrc_t plan_rs, unsigned char* buffers, int buffer_bytes, int table_off,
                                                 unsigned char* meta) {
    auto issue_meta = [&](unsigned i) __attribute__((always_inline)) {
        unsigned char* slot = meta + (i % kWalkMetas) * kWalkMetaBytes;
        if (lw * 1024 + lane * 16 < kWalkMetaBytes)            // (the third KiB is a quarter; the fourth loader has nothing)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(plan_rs, FGX_LDS_PTR(slot + lw * 1024), 16,
                                                     w.plan_at(i) + (uint32_t)(kNarrowTableBytes + lw * 1024 + lane * 16), 0, 0, 0);
    };
    auto issue_chunk = [&](unsigned i) __attribute__((always_inline)) {
        unsigned char* buf = buffers + (i % kWalkBuffers) * buffer_bytes;
        const uint32_t* ids = (const uint32_t*)(meta + (i % kWalkMetas) * kWalkMetaBytes);
        uint32_t src[kWalkSrcGroups], dst[kWalkOutGroups];
#pragma unroll
        for (int j = 0; j < kWalkSrcGroups; ++j) src[j] = ids[(j * kWalkLoad + lw) * 16 + (lane >> 2)];
        if constexpr (OUT_ROWS) {
#pragma unroll
            for (int j = 0; j < kWalkOutGroups; ++j) dst[j] = ids[kNarrowSlots + (j * kWalkLoad + lw) * 16 + (lane >> 2)];
        }
#pragma unroll
        for (int j = 0; j < kWalkSrcGroups; ++j) {
            const int group = j * kWalkLoad + lw;
            const uint32_t piece = (uint32_t)(lane & 3) ^ narrow_piece_key((uint32_t)(group * 16 + (lane >> 2)));       // LDS position lane & 3 holds this piece
            const bool live = src[j] != FGX_EMPTY32 && (int)(piece * 16) < src_row_bytes;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src_rs, FGX_LDS_PTR(buf + group * 1024), 16,
                                                     live ? src[j] * (uint32_t)src_row_bytes + piece * 16u : kNarrowOob, 0, 0, 0);
        }
        if constexpr (OUT_ROWS) {
#pragma unroll
            for (int j = 0; j < kWalkOutGroups; ++j) {
                const int group = j * kWalkLoad + lw;
                const uint32_t piece = (uint32_t)(lane & 3) ^ narrow_piece_key((uint32_t)(group * 16 + (lane >> 2)));
                const bool live = dst[j] != FGX_EMPTY32 && (int)(piece * 16) < out_row_bytes;
                __builtin_amdgcn_raw_ptr_buffer_load_lds(out_rs, FGX_LDS_PTR(buf + kNarrowRowBufPad + group * 1024), 16,
                                                         live ? dst[j] * (uint32_t)out_row_bytes + piece * 16u : kNarrowOob, 0, 0, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < kWalkTableLoads; ++j) {
            const int inst = j * kWalkLoad + lw, row = inst * 16 + (lane >> 2), piece = SWIZZLE ? (lane & 3) ^ ((row >> 2) & 3) : lane & 3;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(plan_rs, FGX_LDS_PTR(buf + table_off + inst * 1024), 16,
                                                     w.plan_at(i) + (uint32_t)(row * (kNarrowTableStride * 2) + piece * 16), 0, 0, 0);
        }
    };
    constexpr int kChunkLoads = kWalkSrcGroups + (OUT_ROWS ? kWalkOutGroups : 0) + kWalkTableLoads;
    for (unsigned i = 0; i < 4 && i < w.count; ++i) issue_meta(i);
    wait_vmcnt<0>();
    walk_barrier();
    for (unsigned i = 0; i < 2 && i < w.count; ++i) issue_chunk(i);
    wait_vmcnt<0>();
    walk_barrier();
    for (unsigned i = 0; i < w.count; ++i) {
        const bool more = i + 2 < w.count, named = i + 4 < w.count;
        if (more) issue_chunk(i + 2);
        if (named) issue_meta(i + 4);
        if (!more) wait_vmcnt<0>();
        else if (named && lw * 1024 < kWalkMetaBytes) wait_vmcnt<kChunkLoads + 1>();
        else wait_vmcnt<kChunkLoads>();
        walk_barrier();
    }
}

}  // namespace
}  // namespace fgx
