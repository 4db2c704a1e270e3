// Building of a plan's chunk (narrow_plan.h) by one workgroup, from source rows that its caller names: the plan kernels
// (conv_gemm_narrow.hip) read them from a neighbor map, the map's own kernel (neighbor_grid.hip) has them in LDS.
// The distinct neighbors of the chunk's rows go through a hash table in LDS; slots are numbered in table order.
#pragma once
#include "fgx_common.h"
#include "narrow_plan.h"

namespace fgx {
namespace {

constexpr int kNarrowHash = 1024;                // hash table of the plan builder (a power of two)

struct NarrowPlanLds {
    uint32_t keys[kNarrowHash + 64];                                                // (a lane without an entry swaps a word of its own)
    __attribute__((aligned(4))) uint16_t slot_of[kNarrowHash];
    uint32_t scan[4];
    uint32_t row_flags[kNarrowRows / 32];
    uint32_t grow_of[kNarrowRows];                                                  // the chunk's rows (FGX_EMPTY32 beyond n): the caller's to write
    __attribute__((aligned(16))) uint16_t table[kNarrowRows * kNarrowTableStride];  // leaves as 16-byte stores
};

// before a barrier, which the caller has after it
template <int THREADS>
__device__ __forceinline__ void narrow_plan_clear(NarrowPlanLds& lds, int V) {
    const int tid = threadIdx.x;
    for (int i = tid; i < kNarrowHash + 64; i += THREADS) lds.keys[i] = FGX_EMPTY32;
    for (int i = tid; i < kNarrowHash / 2; i += THREADS) ((uint32_t*)lds.slot_of)[i] = (uint32_t)kNarrowOverflow << 16 | (uint32_t)kNarrowOverflow;
    if (tid < kNarrowRows / 32) lds.row_flags[tid] = 0u;
    // entries from V on: the row of zeros (entry 31, the row's overflow flag, is written at the end)
    for (int i = tid; i < kNarrowRows * (kNarrowTableStride - V); i += THREADS)
        lds.table[i / (kNarrowTableStride - V) * kNarrowTableStride + V + i % (kNarrowTableStride - V)] = (uint16_t)(kNarrowZeroSlot * 64u);
}

// source_of(e): the source row of entry e = chunk row * V + offset, FGX_EMPTY32 for none.  VC: V where it is 27, else 0.
template <int THREADS, int VC, typename Source>
__device__ __forceinline__ void narrow_plan_chunk(NarrowPlanLds& lds, int V, bool own_rows, unsigned char* __restrict__ plan, uint32_t chunk,
                                                  Source source_of) {
    static_assert(THREADS >= 256, "the scan is four positions of the table a thread");
    const int tid = threadIdx.x;
    unsigned char* mine = plan + kNarrowHeader + (size_t)chunk * kNarrowPlanStride;
    uint32_t* sources = (uint32_t*)(mine + kNarrowTableBytes);
    uint32_t* rows = sources + kNarrowSlots;
    const int entries = kNarrowRows * V;
    auto hash = [](uint32_t x) -> uint32_t { return (x * 2654435761u) >> 22; };      // 10 bits
    auto insert = [&](uint32_t idx, uint32_t h) -> int {                             // table position, -1 when the table is full
        for (int probe = 0; probe < kNarrowHash; ++probe) {
            const uint32_t old = atomicCAS(&lds.keys[h], FGX_EMPTY32, idx);
            if (old == FGX_EMPTY32 || old == idx) return (int)h;
            h = (h + 1) & (kNarrowHash - 1);
        }
        return -1;
    };
    // A chunk row that is also a source row (the same voxels on both sides: every row is its own centre neighbor) takes
    // the slot of its chunk row number: the 16 rows of a fragment read then fall on 16 different slots modulo 16 for
    // the centre offset and on nearly as many for the others -- the neighbors of consecutive rows are mostly
    // consecutive rows -- which is what keeps the reads of arbitrary slots off each other's banks.
    if (own_rows) {
        for (int r = tid; r < kNarrowRows; r += THREADS) {
            if (lds.grow_of[r] != FGX_EMPTY32) {
                const int pos = insert(lds.grow_of[r], hash(lds.grow_of[r]));
                if (pos >= 0) lds.slot_of[pos] = (uint16_t)r;
            }
        }
        __syncthreads();
    }
    // (a thread's entries stay in registers for the second pass: kNarrowRows * kNarrowMaxV / THREADS of them at most; all
    // of them are fetched before the first goes into the table, so that their latencies overlap)
    constexpr int kPerThread = (kNarrowRows * (VC ? VC : 32) + THREADS - 1) / THREADS;
    uint32_t mine_idx[kPerThread];
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int e = tid + j * THREADS;
        mine_idx[j] = e < entries ? source_of(e) : FGX_EMPTY32;
    }
    // first probes of all entries in flight together; the few that met another key go on from there.  An entry's place in the plan's table and its
    // position in the hash table share a register: rows and offsets kept, or worked out a second time, cost wavefronts or time (2.67 M voxels, from
    // the map: kept, with spills, 0.201 ms; a second time 0.167; so 0.164)
    int pos[kPerThread];
    uint32_t met[kPerThread];
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        pos[j] = mine_idx[j] != FGX_EMPTY32 ? (int)hash(mine_idx[j]) : kNarrowHash + (tid & 63);
        met[j] = atomicCAS(&lds.keys[pos[j]], FGX_EMPTY32, mine_idx[j]);
    }
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int e = tid + j * THREADS;
        if (met[j] != FGX_EMPTY32 && met[j] != mine_idx[j]) pos[j] = insert(mine_idx[j], (uint32_t)(pos[j] + 1) & (kNarrowHash - 1));
        pos[j] = ((e / V) * kNarrowTableStride + (e % V)) << 16 | (pos[j] & 0xFFFF);
        asm("" : "+v"(pos[j]));
    }
    __syncthreads();
    // the other sources: slots from `base` on in table order (exclusive scan of their positions, four per thread)
    const uint32_t base = own_rows ? (uint32_t)kNarrowRows : 0u;
    if (own_rows) {
        for (int r = tid; r < kNarrowRows; r += THREADS) sources[r] = lds.grow_of[r];
    }
    const bool counts = THREADS == 256 || tid < 256;            // (whole wavefronts)
    uint32_t own = 0;
    if (counts)
        for (int j = 0; j < 4; ++j) own += (lds.keys[tid * 4 + j] != FGX_EMPTY32 && lds.slot_of[tid * 4 + j] == kNarrowOverflow) ? 1u : 0u;
    uint32_t upto = own;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)upto, d, 64);
        upto += (tid & 63) >= d ? o : 0u;
    }
    if (counts && (tid & 63) == 63) lds.scan[tid >> 6] = upto;
    __syncthreads();
    uint32_t next = base + upto - own, total = base;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        next += w < (tid >> 6) ? lds.scan[w] : 0u;
        total += lds.scan[w];
    }
    for (int j = 0; j < 4 && counts; ++j) {
        const int pos = tid * 4 + j;
        if (lds.keys[pos] != FGX_EMPTY32 && lds.slot_of[pos] == kNarrowOverflow) {
            if (next < (uint32_t)kNarrowSlots) {
                lds.slot_of[pos] = (uint16_t)next;
                sources[next] = lds.keys[pos];
            }
            ++next;
        }
    }
    for (uint32_t s = total + tid; s < (uint32_t)kNarrowSlots; s += THREADS) sources[s] = FGX_EMPTY32;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPerThread; ++j) {
        const int e = tid + j * THREADS;
        if (e >= entries) break;
        uint16_t out = (uint16_t)kNarrowZeroSlot;
        const int in_hash = (int)(int16_t)pos[j], in_table = pos[j] >> 16;
        if (in_hash < kNarrowHash) out = in_hash >= 0 ? lds.slot_of[in_hash] : (uint16_t)kNarrowOverflow;
        // what the multipliers read: the byte offset of the row's logical piece 0 in the row buffer
        if (out != (uint16_t)kNarrowOverflow) out = (uint16_t)(out * 64u + (((uint32_t)out >> 2) & 3u) * 16u);
        lds.table[in_table] = out;
        if (out == (uint16_t)kNarrowOverflow) atomicOr(&lds.row_flags[in_table / kNarrowTableStride >> 5], 1u << (in_table / kNarrowTableStride & 31));
    }
    __syncthreads();
    for (int r = tid; r < kNarrowRows; r += THREADS)
        lds.table[r * kNarrowTableStride + kNarrowTableStride - 1] = (uint16_t)((lds.row_flags[r >> 5] >> (r & 31)) & 1u);
    if (tid == 0 && (lds.row_flags[0] | lds.row_flags[1] | lds.row_flags[2] | lds.row_flags[3]) != 0u) atomicAdd((uint32_t*)plan, 1u);
    for (int r = tid; r < kNarrowRows; r += THREADS) rows[r] = lds.grow_of[r];
    __syncthreads();
    {
        const uint4* from = (const uint4*)lds.table;
        uint4* to = (uint4*)mine;                       // (the plan and its chunks are 16-byte aligned)
        for (int i = tid; i < kNarrowTableBytes / 16; i += THREADS) to[i] = from[i];
    }
}

}  // namespace
}  // namespace fgx
