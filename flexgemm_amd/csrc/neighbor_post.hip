// Post-processing of the neighbor map for the masked implicit GEMM on gfx950:
// mask-sorted voxel order, (v, n)-ordered pair lists for wgrad, per-tile offset masks.
//
// Departures from the reference's data flow (flex_gemm/kernels/cuda/spconv/migemm_neighmap_pp.cu):
//   * pair lists are built from the 4-byte validity masks with a per-block count, one device scan
//     over [V, blocks] and a rank-and-write pass, instead of materialising a transposed map, a
//     transposed 0/1 mask and their N*V-long prefix sum (:85-154, :224-225);
//   * the sort is a stable LSD radix sort restricted to the V mask bits;
//   * tile masks are OR-reduced one wavefront per tile with cross-lane shuffles and accept any
//     tile size, not only powers of two.
#include <cstring>
#include <string.h>

#include <rocprim/rocprim.hpp>

#include "cache_parts.h"
#include "fgx_common.h"
#include "radix_sort.h"

namespace fgx {
namespace {

constexpr int kBlock = 256;
constexpr int kPairThreads = 256;    // a block of the pair-list passes is walked in chunks of this many voxels (larger blocks were not faster)

__global__ void __launch_bounds__(kBlock) iota_u32_kernel(uint32_t* out, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = (uint32_t)i;
}

__global__ void __launch_bounds__(kBlock) widen_u32_i64_kernel(const uint32_t* in, int64_t* out, size_t n) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i < n) out[i] = (int64_t)in[i];
}

// 16 bits of x, y, z interleaved (x highest), batch index on top: voxels close in space get close keys
__device__ __forceinline__ uint64_t spread16(uint32_t x) {
    uint64_t v = x & 0xFFFFu;
    v = (v | (v << 16)) & 0x0000FF0000FFull;
    v = (v | (v << 8)) & 0x00F00F00F00Full;
    v = (v | (v << 4)) & 0x0C30C30C30C3ull;
    v = (v | (v << 2)) & 0x249249249249ull;
    return v;
}

// Z-order key: the batch index right above the 3 * bits interleaved coordinate bits (Key: 32 bits when they all fit)
template <typename Key>
__global__ void __launch_bounds__(kBlock) morton_key_packed_kernel(const int32_t* __restrict__ coords, size_t n, int bits,
                                                                   Key* __restrict__ keys, uint32_t* __restrict__ vals) {
    size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    int4 c = reinterpret_cast<const int4*>(coords)[i];
    const uint64_t m = (spread16((uint32_t)c.y) << 2) | (spread16((uint32_t)c.z) << 1) | spread16((uint32_t)c.w);
    keys[i] = (Key)(((uint64_t)(uint32_t)c.x << (3 * bits)) | (m & ((1ull << (3 * bits)) - 1ull)));
    vals[i] = (uint32_t)i;
}

// position p of the spatial order -> (chunk of p, mask code of its voxel)
__global__ void __launch_bounds__(kBlock) chunk_code_key_kernel(const uint32_t* __restrict__ perm,
                                                                const int32_t* __restrict__ binary, size_t n,
                                                                uint32_t chunk_rows, int code_bits, uint64_t* __restrict__ keys) {
    size_t p = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    keys[p] = ((uint64_t)(p / chunk_rows) << code_bits) | (uint32_t)binary[perm[p]];
}

struct LocalityLayout {
    size_t keys_a, keys_b, vals_a, vals_b, temp, temp_bytes, radix, total;
};

LocalityLayout locality_layout(size_t n) {
    LocalityLayout L{};
    size_t nn = n ? n : 1;
    size_t temp_bytes = 0;
    (void)rocprim::radix_sort_pairs(nullptr, temp_bytes, (const uint64_t*)nullptr, (uint64_t*)nullptr,
                                    (const uint32_t*)nullptr, (uint32_t*)nullptr, nn, 0u, 64u, (hipStream_t)0);
    size_t off = 0;
    L.keys_a = off; off = align_up(off + nn * 8, 256);
    L.keys_b = off; off = align_up(off + nn * 8, 256);
    L.vals_a = off; off = align_up(off + nn * 4, 256);
    L.vals_b = off; off = align_up(off + nn * 4, 256);
    L.temp = off;   off = align_up(off + temp_bytes, 256);
    L.temp_bytes = temp_bytes;
    L.radix = off;
    if (n <= kRsMaxItems) off += radix_layout(n).total;
    L.total = off;
    return L;
}

int bits_for(size_t x) {   // smallest b with 2^b > x
    int b = 0;
    while (b < 63 && ((size_t)1 << b) <= x) ++b;
    return b;
}


// Mask sort of up to this many rows: every row counts the rows that come before it (rank_sort_kernel) -- one launch of n^2
// compares against nine of the radix sort (8 192 rows 0.017 ms against 0.037, 16 384 rows 0.030 against 0.039; the crossing lies
// near 20 000).
constexpr size_t kRankSortMax = 16384;
constexpr int kRankSlices = 16;      // wavefronts of a workgroup, each counting over a sixteenth of the keys for the same 64 rows

// order[rank of row i] = i, rows by (key, row).  A wavefront takes its keys 64 at a time, one per lane, and compares its 64
// rows with each of them in turn (read from the lane that holds it).  Chunks are aligned to the workgroup's own 64 rows, so
// whether equal keys come before or after is the same for a whole chunk, but for the one that is the rows themselves.
template <typename Before>
__device__ __forceinline__ uint32_t count_before(uint32_t held, uint32_t len, Before before) {
    uint32_t count = 0u;
    if (len == 64u) {
#pragma unroll
        for (int k = 0; k < 64; ++k) count += before((uint32_t)__builtin_amdgcn_readlane((int)held, k), (uint32_t)k) ? 1u : 0u;
    } else {
        for (uint32_t k = 0; k < len; ++k) count += before((uint32_t)__builtin_amdgcn_readlane((int)held, (int)k), k) ? 1u : 0u;
    }
    return count;
}

__global__ void __launch_bounds__(64 * kRankSlices) rank_sort_kernel(const uint32_t* __restrict__ keys, uint32_t n, uint32_t flip,
                                                                     int64_t* __restrict__ order) {
    __shared__ uint32_t part[kRankSlices][64];
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t i0 = blockIdx.x * 64u, i = i0 + lane;
    const uint32_t mine = i < n ? keys[i] ^ flip : 0u;
    uint32_t before = 0u;
    uint32_t j = wave * 64u;                                        // the wavefronts take the chunks in turn
    uint32_t next = j + lane < n ? keys[j + lane] ^ flip : 0u;
    while (j < n) {
        const uint32_t held = next, len = n - j < 64u ? n - j : 64u, at = j;
        j += kRankSlices * 64u;
        next = j + lane < n ? keys[j + lane] ^ flip : 0u;           // the next chunk is on its way
        if (at < i0) before += count_before(held, len, [&](uint32_t other, uint32_t) { return other <= mine; });
        else if (at > i0) before += count_before(held, len, [&](uint32_t other, uint32_t) { return other < mine; });
        else before += count_before(held, len, [&](uint32_t other, uint32_t k) { return other < mine || (other == mine && k < lane); });
    }
    part[wave][lane] = before;
    __syncthreads();
    if (wave == 0u && i < n) {
        uint32_t rank = 0u;
#pragma unroll
        for (int w = 0; w < kRankSlices; ++w) rank += part[w][lane];
        order[rank] = (int64_t)i;
    }
}

struct SortLayout {
    size_t keys_out, vals_in, vals_out, temp, temp_bytes, total;
};

// the library sort, for more rows than the radix sort of radix_sort.h takes
SortLayout sort_layout(size_t n) {
    SortLayout L{};
    size_t nn = n ? n : 1;
    size_t temp_bytes = 0;
    // size query only: no work is enqueued
    (void)rocprim::radix_sort_pairs(nullptr, temp_bytes, (const int32_t*)nullptr, (int32_t*)nullptr,
                                    (const uint32_t*)nullptr, (uint32_t*)nullptr, nn, 0u, 32u, (hipStream_t)0);
    size_t off = 0;
    L.keys_out = off; off = align_up(off + nn * 4, 256);
    L.vals_in = off;  off = align_up(off + nn * 4, 256);
    L.vals_out = off; off = align_up(off + nn * 4, 256);
    L.temp = off;     off = align_up(off + temp_bytes, 256);
    L.temp_bytes = temp_bytes;
    L.total = off;
    return L;
}

// counts[v * nblk + blk] = number of voxels of block blk whose mask has bit v set.  A block is kPairRows voxels, walked
// by kPairThreads threads in kPairRows / kPairThreads chunks.
__global__ void __launch_bounds__(kPairThreads) pair_count_kernel(const int32_t* __restrict__ gray, size_t n, int V,
                                                                  unsigned nblk, uint32_t* __restrict__ counts) {
    __shared__ uint32_t wave_cnt[kPairThreads / 64][32];
    constexpr int kChunks = kPairRows / kPairThreads;
    uint32_t g[kChunks];
#pragma unroll
    for (int c = 0; c < kChunks; ++c) {
        const size_t row = (size_t)blockIdx.x * kPairRows + c * kPairThreads + threadIdx.x;
        g[c] = row < n ? (uint32_t)gray[row] : 0u;
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int v = 0; v < V; ++v) {
        uint32_t cnt = 0;
#pragma unroll
        for (int c = 0; c < kChunks; ++c) cnt += (uint32_t)__popcll(__ballot((g[c] >> v) & 1u));
        if (lane == 0) wave_cnt[wave][v] = cnt;
    }
    __syncthreads();
    if (threadIdx.x < V) {
        uint32_t c = 0;
        for (int w = 0; w < kPairThreads / 64; ++w) c += wave_cnt[w][threadIdx.x];
        counts[(size_t)threadIdx.x * nblk + blockIdx.x] = c;
    }
}

// offsets[v * nblk + blk] = pairs of offset v in the blocks before blk, totals[v] = all of them: one workgroup per offset, four
// blocks per thread and turn.  A block's count is the sum of GROUP consecutive entries of counts[v][m].
template <int GROUP>
__global__ void __launch_bounds__(256) pair_scan_kernel(const uint32_t* __restrict__ counts, size_t m, unsigned nblk,
                                                        uint32_t* __restrict__ offsets, uint32_t* __restrict__ totals) {
    __shared__ uint32_t part[4];
    const uint32_t* row = counts + (size_t)blockIdx.x * m;
    uint32_t* out = offsets + (size_t)blockIdx.x * nblk;
    uint32_t carry = 0u;
    for (unsigned t0 = 0; t0 < nblk; t0 += 1024) {               // (uniform)
        const unsigned t = t0 + threadIdx.x * 4;
        uint32_t v[4], sum = 0u, all;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = 0u;
#pragma unroll
            for (int q = 0; q < GROUP; ++q) {
                const size_t i = (size_t)(t + k) * GROUP + q;
                v[k] += i < m ? row[i] : 0u;
            }
            sum += v[k];
        }
        uint32_t run = carry + block_exclusive_sum<4>(sum, part, &all);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (t + k < nblk) out[t + k] = run;
            run += v[k];
        }
        carry += all;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// first pair of offset `v` = pairs of the offsets before it, for lane v of a wavefront (lane V: all pairs)
__device__ __forceinline__ uint32_t pair_segment(const uint32_t* __restrict__ totals, int V, int lane) {
    const uint32_t mine = lane < V ? totals[lane] : 0u;
    uint32_t incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
        if (lane >= d) incl += o;
    }
    return incl - mine;
}

// seg[0 .. V] of an empty (totals == nullptr) or a counted cache
__global__ void pair_seg_kernel(const uint32_t* __restrict__ totals, int V, uint32_t* __restrict__ seg) {
    const int v = threadIdx.x;
    const uint32_t first = totals != nullptr ? pair_segment(totals, V, v) : 0u;
    if (v <= V) seg[v] = first;
}

// A block takes kPairRows voxels in chunks of kPairThreads: the chunk's map rows are staged in LDS with coalesced loads,
// then for every offset the present voxels are ranked (wave ballot + prefix of the wave totals) and (n, map[n, v]) goes
// to first[v] + rank, where first[v] starts at offsets[v, blk] and moves on by the chunk's count.  The pairs a block
// adds to one offset's list are therefore one run of up to kPairRows entries written by one workgroup within a few
// microseconds: the partial cache lines at the seams of the chunks' pieces meet in L2.
// KV: V as a constant (0: any), so that a thread's map words and LDS reads are all in flight together; small inputs wait for
// little else (3 716 voxels 13.9 -> 7.1 us, 424 000 30.7 -> 20.2).
template <int KV>
__global__ void __launch_bounds__(kPairThreads) pair_fill_kernel(const uint32_t* __restrict__ map,
                                                                 const int32_t* __restrict__ gray, size_t n, int v_count,
                                                                 unsigned nblk, const uint32_t* __restrict__ offsets,
                                                                 const uint32_t* __restrict__ totals, uint32_t* __restrict__ seg,
                                                                 uint32_t* __restrict__ seg_host, uint32_t* __restrict__ sig_i, uint32_t* __restrict__ sig_o) {
    extern __shared__ uint32_t lds[];
    constexpr int kWaves = kPairThreads / 64;
    constexpr int kFlight = KV ? KV : 8;                     // loads in flight per thread
    const int V = KV ? KV : v_count;
    uint32_t* rows = lds;                                    // [kPairThreads * V]
    uint32_t* wave_cnt2 = lds + (size_t)kPairThreads * V;    // [2][kWaves][32], by chunk parity
    uint32_t* first = wave_cnt2 + 2 * kWaves * 32;           // [32] where the next pairs of each offset go
    // fetched once, up front: a load inside the offset loop below would put a memory round trip into each of its turns
    if (threadIdx.x < 64) {
        const uint32_t start = pair_segment(totals, V, (int)threadIdx.x);
        if (threadIdx.x < V) first[threadIdx.x] = start + offsets[(size_t)threadIdx.x * nblk + blockIdx.x];
        if (seg != nullptr && blockIdx.x == 0 && threadIdx.x <= V) {
            seg[threadIdx.x] = start;
            if (seg_host != nullptr) seg_host[threadIdx.x] = start;
        }
    }
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const unsigned long long below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    for (int c = 0; c < kPairRows / kPairThreads; ++c) {
        const size_t base = (size_t)blockIdx.x * kPairRows + (size_t)c * kPairThreads;
        if (base >= n) break;                                // uniform
        // two count tables: the first wavefront may still be adding up the previous chunk's counts (below) while the
        // others write this chunk's
        uint32_t* wave_cnt = wave_cnt2 + (c & 1) * kWaves * 32;
        const size_t len = (n - base < (size_t)kPairThreads ? n - base : (size_t)kPairThreads) * V;
        // several loads in flight per thread: a plain copy loop waits for each load before it issues the next
        for (size_t i0 = 0; i0 < len; i0 += kFlight * kPairThreads) {
            uint32_t t8[kFlight];
#pragma unroll
            for (int q = 0; q < kFlight; ++q) {
                const size_t i = i0 + (size_t)q * kPairThreads + threadIdx.x;
                t8[q] = i < len ? map[base * V + i] : 0u;
            }
#pragma unroll
            for (int q = 0; q < kFlight; ++q) {
                const size_t i = i0 + (size_t)q * kPairThreads + threadIdx.x;
                if (i < len) rows[i] = t8[q];
            }
        }
        const size_t row = base + threadIdx.x;
        const uint32_t g = row < n ? (uint32_t)gray[row] : 0u;
        for (int v = 0; v < V; ++v) {
            unsigned long long b = __ballot((g >> v) & 1u);
            if (lane == 0) wave_cnt[wave * 32 + v] = (uint32_t)__popcll(b);
        }
        __syncthreads();
        // where this wavefront's pairs of offset v go: in lane v
        uint32_t at = 0u;
        if (lane < V) {
            at = first[lane];
            for (int w = 0; w < wave; ++w) at += wave_cnt[w * 32 + lane];
        }
        auto put = [&](int v, uint32_t source) {
            const unsigned long long b = __ballot((g >> v) & 1u);
            const uint32_t to = (uint32_t)__builtin_amdgcn_readlane((int)at, v) + (uint32_t)__popcll(b & below);
            if ((g >> v) & 1u) {
                sig_o[to] = (uint32_t)row;
                sig_i[to] = source;
            }
        };
        if constexpr (KV != 0) {
            uint32_t source[KV];
#pragma unroll
            for (int v = 0; v < KV; ++v) source[v] = rows[(size_t)threadIdx.x * KV + v];
#pragma unroll
            for (int v = 0; v < KV; ++v) put(v, source[v]);
        } else {
            for (int v = 0; v < V; ++v) put(v, rows[(size_t)threadIdx.x * V + v]);
        }
        __syncthreads();                                     // rows and first[] have been read by everyone
        if (threadIdx.x < V) {
            uint32_t add = 0;
            for (int w = 0; w < kWaves; ++w) add += wave_cnt[w * 32 + threadIdx.x];
            first[threadIdx.x] += add;
        }
        // the next chunk's first barrier orders these updates before they are read
    }
}

// One wavefront per tile and turn: OR of gray[sorted_idx[r]] over the tile's rows.
__global__ void __launch_bounds__(kBlock) tile_or_kernel(const int32_t* __restrict__ gray,
                                                         const int64_t* __restrict__ sorted_idx, size_t n, int block,
                                                         size_t num_tiles, int32_t* __restrict__ tile_code) {
    const int lane = threadIdx.x & 63;
    for (size_t tile = ((size_t)blockIdx.x * kBlock + threadIdx.x) >> 6; tile < num_tiles; tile += (size_t)gridDim.x * (kBlock / 64)) {
        const size_t lo = tile * (size_t)block;
        const size_t hi = lo + (size_t)block < n ? lo + (size_t)block : n;
        uint32_t code = 0;
        for (size_t r = lo + lane; r < hi; r += 64) code |= (uint32_t)gray[sorted_idx[r]];
        for (int off = 32; off > 0; off >>= 1) code |= (uint32_t)__shfl_xor((int)code, off, 64);
        if (lane == 0) tile_code[tile] = (int32_t)code;
    }
}

__global__ void set_i32_kernel(int32_t* dst, int32_t value) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *dst = value;
}

__global__ void __launch_bounds__(kBlock) tile_fill_kernel(const int32_t* __restrict__ tile_code,
                                                           const int32_t* __restrict__ seg, size_t num_tiles,
                                                           int32_t* __restrict__ valid_kernel) {
    size_t t = (size_t)blockIdx.x * kBlock + threadIdx.x;
    if (t >= num_tiles) return;
    uint32_t code = (uint32_t)tile_code[t];
    int32_t* dst = valid_kernel + seg[t];
    while (code) {
        *dst++ = __ffs((int)code) - 1;
        code &= code - 1;
    }
}

// ---------------------------------------------------------------------------------------------------------------
// The tables over all row tiles, by one workgroup: where each tile's public offset list and its gather-plan rows start, and
// the item order of the streaming GEMM.
// ---------------------------------------------------------------------------------------------------------------
// Items (row tile * col_tiles + column tile) cost about max(popcount(tile_code), 1) offsets each.  Workgroup slot q of
// `groups` works through the positions q, q + groups, ... of the sequence written here.  Step 1 sorts the items by
// cost, most expensive first (stable counting sort over the 33 possible popcounts: a wavefront counts, then places, a
// contiguous piece 64 items at a time, equal costs found by ballots).  Step 2 deals them round by round: the incomplete
// last round takes the cheapest items, every full round gives its most expensive item to the least loaded slot (rank of
// each slot's load by counting, or by a sort of the loads).  Everything is deterministic.  One workgroup, so what bounds it is the length of its
// dependent chains: the counting sort by one thread per piece with serial prefixes over 256 of them, and the ranks one
// load at a time, took 0.040 ms for 1 306 items and 256 slots; this form, the scans of 1 306 tiles included, 0.017.
constexpr int kOrderThreads = 1024;     // also the largest number of slots
constexpr int kOrderWaves = kOrderThreads / 64;
constexpr unsigned kOrderInLds = 8192;  // items whose sorted list stays in LDS

__device__ __forceinline__ unsigned tile_cost_bin(uint32_t code) { return 32u - (unsigned)__popc(code); }   // 0 = most expensive

// A sorted item carries its cost above 26 bits of its number; WIDE: more items than that, whose cost is looked up again.
constexpr unsigned kItemBits = 26;
template <bool WIDE, int THREADS>
__device__ void order_items(const int32_t* __restrict__ tile_code, unsigned num_tiles, unsigned col_tiles, unsigned slabs, unsigned groups,
                            uint32_t* __restrict__ sorted, uint32_t* __restrict__ item_at) {
    constexpr int WAVES = THREADS / 64;
    __shared__ uint32_t count[WAVES][64];
    __shared__ __attribute__((aligned(16))) uint32_t load[THREADS];
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const unsigned total = num_tiles * col_tiles;
    const unsigned long long below = (1ull << lane) - 1ull;
    const unsigned piece = ((total + WAVES - 1) / WAVES + 63u) & ~63u;
    const unsigned lo = wave * piece < total ? wave * piece : total, hi = lo + piece < total ? lo + piece : total;
    auto bin_of = [&](unsigned item) -> unsigned { return tile_cost_bin((uint32_t)tile_code[col_tiles == 1 ? item : item / col_tiles]); };
    // ---- step 1: stable counting sort, cost descending ----
    count[wave][lane] = 0u;
    for (unsigned i0 = lo; i0 < hi; i0 += 64) {                   // (one wavefront: its LDS accesses stay in order)
        const bool live = i0 + lane < hi;
        const unsigned bin = live ? bin_of(i0 + lane) : 0u;
        const unsigned long long peers = radix_peers(bin, 6, live);
        if (live && lane == (unsigned)(__ffsll((long long)peers) - 1)) count[wave][bin] += (uint32_t)__popcll(peers);
    }
    __syncthreads();
    if (wave == 0) {                                              // lane = bin
        uint32_t mine = 0u, before[WAVES];
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            before[w] = mine;
            mine += count[w][lane];
        }
        uint32_t incl = mine;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
            if ((int)lane >= d) incl += o;
        }
#pragma unroll
        for (int w = 0; w < WAVES; ++w) count[w][lane] = incl - mine + before[w];
    }
    __syncthreads();
    for (unsigned i0 = lo; i0 < hi; i0 += 64) {
        const bool live = i0 + lane < hi;
        const unsigned bin = live ? bin_of(i0 + lane) : 0u;
        const unsigned long long peers = radix_peers(bin, 6, live);
        const int leader = live ? __ffsll((long long)peers) - 1 : 0;
        uint32_t first = 0u;
        if (live && (int)lane == leader) {
            first = count[wave][bin];
            count[wave][bin] = first + (uint32_t)__popcll(peers);
        }
        first = (uint32_t)__shfl((int)first, leader, 64);
        if (live) sorted[first + (uint32_t)__popcll(peers & below)] = WIDE ? i0 + lane : bin << kItemBits | (i0 + lane);
    }
    __threadfence_block();
    __syncthreads();
    // ---- step 2: deal the rounds ----
    // A slot's standing is its load above its number, so that one compare orders two slots; loads are kept within 21 bits.
    const unsigned rounds = total / groups, rem = total % groups;
    unsigned scale = 0;
    while ((((unsigned long long)(rounds + 1) * (32u * slabs + 3u)) >> scale) >= (1ull << 21)) ++scale;
    auto item_of = [](uint32_t entry) -> uint32_t { return WIDE ? entry : entry & ((1u << kItemBits) - 1u); };
    auto cost_of = [&](uint32_t entry) -> uint32_t {
        const unsigned pc = 32u - (WIDE ? bin_of(entry) : entry >> kItemBits);
        return ((pc ? pc : 1u) * slabs + 3u) >> scale;
    };
    if (groups > 256u) {
        // Ranks by counting read every load once per slot (512 slots: 7 us a round); with this many the standings are sorted instead (2.5 us), and a thread
        // goes on with the slot whose standing it was given.  2 611 items in 512 slots beside the plan of as many tiles 41 -> 19 us, 3 817 items 57 -> 27.
        uint32_t key = tid < groups ? tid : 0xFFFFFFFFu;
        if (tid < rem) {
            const uint32_t entry = sorted[total - rem + tid];
            item_at[rounds * groups + tid] = item_of(entry);
            key += cost_of(entry) << 10;
        }
        for (unsigned r = 0; r < rounds; ++r) {
#pragma unroll
            for (unsigned k = 2; k <= (unsigned)THREADS; k *= 2)
#pragma unroll
                for (unsigned j = k / 2; j > 0; j /= 2) {
                    uint32_t other;
                    if (j < 64) {
                        other = (uint32_t)__shfl_xor((int)key, (int)j, 64);
                    } else {
                        load[tid] = key;
                        __syncthreads();
                        other = load[tid ^ j];
                        __syncthreads();
                    }
                    key = ((tid & j) == 0) == ((tid & k) == 0) ? (key < other ? key : other) : (key < other ? other : key);
                }
            if (tid < groups) {
                const uint32_t entry = sorted[r * groups + tid];      // the least loaded slot <- most expensive item
                item_at[r * groups + (key & 1023u)] = item_of(entry);
                key += cost_of(entry) << 10;
            }
        }
        return;
    }
    // P threads per slot share the counting
    const unsigned P = groups <= THREADS / 4 ? 4u : (groups <= THREADS / 2 ? 2u : 1u);
    const unsigned slot = tid / P, part = tid % P;
    uint32_t mine = slot;
    if (slot < rem) {                                             // cheapest items: the positions of the last round
        const uint32_t entry = sorted[total - rem + slot];
        if (part == 0) item_at[rounds * groups + slot] = item_of(entry);
        mine += cost_of(entry) << 10;
    }
    const unsigned quads = (groups + 3u) / 4u;
    for (unsigned r = 0; r < rounds; ++r) {
        if (part == 0) load[slot] = slot < groups ? mine : 0xFFFFFFFFu;
        __syncthreads();
        unsigned rank = 0;
        const uint4* load4 = reinterpret_cast<const uint4*>(load);
#pragma unroll 4
        for (unsigned q = part; q < quads; q += P) {
            const uint4 o = load4[q];
            rank += (o.x < mine ? 1u : 0u) + (o.y < mine ? 1u : 0u) + (o.z < mine ? 1u : 0u) + (o.w < mine ? 1u : 0u);
        }
        if (P >= 2) rank += (unsigned)__shfl_xor((int)rank, 1, 64);
        if (P >= 4) rank += (unsigned)__shfl_xor((int)rank, 2, 64);
        if (slot < groups) {
            const uint32_t entry = sorted[r * groups + rank];     // rank 0 = least loaded slot <- most expensive item
            if (part == 0) item_at[r * groups + slot] = item_of(entry);
            mine += cost_of(entry) << 10;
        }
        __syncthreads();
    }
}

struct TilePrefix {
    uint32_t at, plan_at;           // offsets, gather-plan rows
};
// sums of `mine` over the threads before this one, and (*all) over the workgroup's
__device__ __forceinline__ TilePrefix tile_prefix(const TilePrefix& mine, uint32_t (*part)[kOrderWaves], TilePrefix* all) {
    TilePrefix before;
    before.at = block_exclusive_sum<kOrderWaves>(mine.at, part[0], &all->at);
    before.plan_at = block_exclusive_sum<kOrderWaves>(mine.plan_at, part[1], &all->plan_at);
    return before;
}

// (a tile without any offset has one plan row, all rows missing: every tile owns at least one step of the GEMM)
__device__ __forceinline__ TilePrefix tile_counts(const int32_t* __restrict__ tile_code, unsigned t, unsigned num_tiles) {
    const uint32_t c = t < num_tiles ? (uint32_t)__popc((uint32_t)tile_code[t]) : 0u;
    return TilePrefix{c, t < num_tiles && c == 0u ? 1u : c};
}

// seg (optional): exclusive offsets of the tiles' public offset lists, plan_seg (optional): of their gather-plan rows, both with
// the total at [num_tiles]; item_at (optional): the item order, `sorted` its workspace.
__global__ void __launch_bounds__(kOrderThreads) tile_tables_kernel(const int32_t* __restrict__ tile_code, unsigned num_tiles,
                                                                    int32_t* __restrict__ seg, int32_t* __restrict__ plan_seg,
                                                                    unsigned col_tiles, unsigned slabs, unsigned groups,
                                                                    uint32_t* __restrict__ sorted, uint32_t* __restrict__ item_at) {
    __shared__ uint32_t part[2][kOrderWaves];
    __shared__ uint32_t sorted_lds[kOrderInLds];
    if (seg != nullptr || plan_seg != nullptr) {
        TilePrefix run{0u, 0u}, all;
        for (unsigned t0 = 0; t0 < num_tiles; t0 += kOrderThreads) {         // (uniform)
            const unsigned t = t0 + threadIdx.x;
            const TilePrefix before = tile_prefix(tile_counts(tile_code, t, num_tiles), part, &all);
            if (t < num_tiles) {
                if (seg != nullptr) seg[t] = (int32_t)(run.at + before.at);
                if (plan_seg != nullptr) plan_seg[t] = (int32_t)(run.plan_at + before.plan_at);
            }
            run.at += all.at;
            run.plan_at += all.plan_at;
        }
        if (threadIdx.x == 0) {
            if (seg != nullptr) seg[num_tiles] = (int32_t)run.at;
            if (plan_seg != nullptr) plan_seg[num_tiles] = (int32_t)run.plan_at;
        }
    }
    if (item_at == nullptr) return;
    if ((unsigned long long)num_tiles * col_tiles < (1ull << kItemBits))
        order_items<false, kOrderThreads>(tile_code, num_tiles, col_tiles, slabs, groups, num_tiles * col_tiles <= kOrderInLds ? sorted_lds : sorted, item_at);
    else
        order_items<true, kOrderThreads>(tile_code, num_tiles, col_tiles, slabs, groups, sorted, item_at);
}

// The segment tables of many tiles, in chunks: a chunk's sums are left in its last entries of the tables, one workgroup adds them up
// there, and every chunk then writes its own entries from what it finds there.  One workgroup for all tiles takes
// 1.45 us per 1024 of them (8 192 tiles 13.1 us, 10 419 17.6, 83 350 120, 2 667 120 4 079); the chunks' three launches take 13.3 us for
// 10 419, 14.7 for 83 350, 32 for 2 667 120.
constexpr unsigned kOneScanTiles = 8192, kScanChunk = 4096;

__global__ void __launch_bounds__(kOrderThreads) tile_sums_kernel(const int32_t* __restrict__ tile_code, unsigned num_tiles, int32_t* seg,
                                                                  int32_t* plan_seg) {
    __shared__ uint32_t part[2][kOrderWaves];
    const unsigned t0 = blockIdx.x * kScanChunk, last = (num_tiles - t0 < kScanChunk ? num_tiles : t0 + kScanChunk) - 1u;
    TilePrefix mine{0u, 0u}, all;
#pragma unroll
    for (unsigned r = 0; r < kScanChunk; r += kOrderThreads) {
        const TilePrefix c = tile_counts(tile_code, t0 + r + threadIdx.x, num_tiles);
        mine.at += c.at;
        mine.plan_at += c.plan_at;
    }
    tile_prefix(mine, part, &all);
    if (threadIdx.x == 0) {
        if (seg != nullptr) seg[last] = (int32_t)all.at;
        if (plan_seg != nullptr) plan_seg[last] = (int32_t)all.plan_at;
    }
}

__global__ void __launch_bounds__(kOrderThreads) chunk_scan_kernel(unsigned num_tiles, unsigned chunks, int32_t* seg,
                                                                   int32_t* plan_seg) {
    __shared__ uint32_t part[2][kOrderWaves];
    TilePrefix run{0u, 0u};
    for (unsigned b0 = 0; b0 < chunks; b0 += kOrderThreads) {                // (uniform)
        const unsigned b = b0 + threadIdx.x;
        const unsigned last = b + 1 < chunks ? (b + 1) * kScanChunk - 1u : num_tiles - 1u;
        TilePrefix mine{0u, 0u}, all;
        if (b < chunks && seg != nullptr) mine.at = (uint32_t)seg[last];
        if (b < chunks && plan_seg != nullptr) mine.plan_at = (uint32_t)plan_seg[last];
        const TilePrefix before = tile_prefix(mine, part, &all);
        if (b < chunks && seg != nullptr) seg[last] = (int32_t)(run.at + before.at);
        if (b < chunks && plan_seg != nullptr) plan_seg[last] = (int32_t)(run.plan_at + before.plan_at);
        run.at += all.at;
        run.plan_at += all.plan_at;
    }
    if (threadIdx.x == 0) {
        if (seg != nullptr) seg[num_tiles] = (int32_t)run.at;
        if (plan_seg != nullptr) plan_seg[num_tiles] = (int32_t)run.plan_at;
    }
}

__global__ void __launch_bounds__(kOrderThreads) chunk_tables_kernel(const int32_t* __restrict__ tile_code, unsigned num_tiles, int32_t* seg,
                                                                     int32_t* plan_seg) {
    __shared__ uint32_t part[2][kOrderWaves];
    const unsigned t0 = blockIdx.x * kScanChunk, last = (num_tiles - t0 < kScanChunk ? num_tiles : t0 + kScanChunk) - 1u;
    TilePrefix run{seg != nullptr ? (uint32_t)seg[last] : 0u, plan_seg != nullptr ? (uint32_t)plan_seg[last] : 0u};
#pragma unroll
    for (unsigned r = 0; r < kScanChunk; r += kOrderThreads) {
        const unsigned t = t0 + r + threadIdx.x;
        const TilePrefix c = tile_counts(tile_code, t, num_tiles);
        TilePrefix all;
        const TilePrefix before = tile_prefix(c, part, &all);               // (its barriers: the chunk's sum has been read)
        if (t < num_tiles) {
            if (seg != nullptr) seg[t] = (int32_t)(run.at + before.at);
            if (plan_seg != nullptr) plan_seg[t] = (int32_t)(run.plan_at + before.plan_at);
        }
        run.at += all.at;
        run.plan_at += all.plan_at;
    }
}

// ---------------------------------------------------------------------------------------------------------------
// A workgroup per tile, or per two or four short ones (fill_together): plan_idx[plan_seg[t] + k][r] = map[order[t * tile_rows + r]][k-th offset present in the tile]
// (EMPTY for rows past the end); plan_band[plan_seg[t] + k] (optional) has bit b set when rows [32 b, 32 b + 32) of the
// tile hold at least one present neighbor for that offset.
//
// The tile's rows sit wherever the mask order put them: a half-wave fetches one whole row (V consecutive words: one or two cache
// lines per request) into LDS, and kFillThreads / R threads share a row's offsets.  Bound by latency: with 256 threads a tile, each
// of them walking all offsets of its row, 1 306 tiles of 128 rows took 18.4 us.  512 threads and no more LDS than the rows need
// put four tiles on a CU at a time (1024 threads, two tiles: 29 us with the tables below).
//
// TABLES: a workgroup adds up the counts of the tiles before its own itself (and leaves them in seg and plan_seg), and the first one
// (item_at) deals the item order beside them.  One workgroup that scanned and dealt before the others could start took 15.7 us for
// 1 306 tiles: tables and fill 34.1 -> 17.8 us, 12.5 with two tiles a workgroup (and for the two maps of a 2 x 2 x 2 stride over a 256^3 shell 34.0 -> 18.3).  Up to
// kFillScanTiles tiles: the additions are quadratic.
// ---------------------------------------------------------------------------------------------------------------
constexpr int kFillThreads = 512, kFillRows = 256, kFillTogether = 4;
constexpr unsigned kFillScanTiles = 4096;

template <bool TABLES>
__global__ void __launch_bounds__(kFillThreads) plan_fill_kernel(const uint32_t* __restrict__ map, const int64_t* __restrict__ order,
                                                                 const int32_t* __restrict__ tile_code, size_t num_tiles, size_t n, int V,
                                                                 int tile_rows, int R, int32_t* __restrict__ seg, int32_t* __restrict__ plan_seg,
                                                                 uint32_t* __restrict__ plan_idx, uint32_t* __restrict__ plan_band,
                                                                 unsigned col_tiles, unsigned slabs, unsigned groups, uint32_t* __restrict__ sorted,
                                                                 uint32_t* __restrict__ item_at, int together) {
    extern __shared__ uint32_t stage[];              // R map rows of V words; the item order's sorted list in the workgroup that makes it
    __shared__ int64_t src_row[kFillRows];           // which map row each of them is (-1: past the end)
    __shared__ uint32_t bands[kFillTogether][32], offsets[kFillTogether][32];
    const int tid = threadIdx.x, lane = tid & 63;
    size_t t = blockIdx.x;
    if constexpr (TABLES) {
        if (item_at != nullptr) {
            if (t == 0) {
                order_items<false, kFillThreads>(tile_code, (unsigned)num_tiles, col_tiles, slabs, groups,
                                                 num_tiles * col_tiles <= kOrderInLds ? stage : sorted, item_at);
                return;
            }
            --t;
        }
    }
    t *= (size_t)together;                           // the first of this workgroup's tiles
    const int all_rows = together * tile_rows;
    auto fetch_order = [&](int r0) {
        if (tid < R) {
            const size_t row = t * (size_t)tile_rows + r0 + tid;
            src_row[tid] = (r0 + tid < all_rows && row < n) ? order[row] : (int64_t)-1;
        }
    };
    fetch_order(0);
    const int sub = together > 1 ? tid % R / tile_rows : 0;                 // this thread's tile (whole wavefronts share one)
    const size_t own_tile = t + sub;
    size_t slot;
    if constexpr (TABLES) {
        __shared__ uint64_t part[kFillThreads / 64];
        uint64_t mine = 0;                           // offsets of the tiles before this one | their plan rows (at most 32 each)
        for (unsigned q = tid; q < (unsigned)t; q += kFillThreads) {
            const TilePrefix c = tile_counts(tile_code, q, (unsigned)num_tiles);
            mine += (uint64_t)c.at << 32 | c.plan_at;
        }
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) mine += (uint64_t)__shfl_xor((unsigned long long)mine, d, 64);
        if (lane == 0) part[tid >> 6] = mine;
        __syncthreads();
        uint64_t before = 0;
#pragma unroll
        for (int w = 0; w < kFillThreads / 64; ++w) before += part[w];
        TilePrefix upto;
        upto.at = (uint32_t)(before >> 32);
        upto.plan_at = (uint32_t)before;
        slot = upto.plan_at;
        for (int i = 0; i < together && t + i < num_tiles; ++i) {
            if (tid == 0) {
                if (seg != nullptr) seg[t + i] = (int32_t)upto.at;
                plan_seg[t + i] = (int32_t)upto.plan_at;
            }
            const TilePrefix own = tile_counts(tile_code, (unsigned)(t + i), (unsigned)num_tiles);
            upto.at += own.at;
            upto.plan_at += own.plan_at;
            slot += i < sub ? own.plan_at : 0u;
            if (tid == 0 && t + i + 1 == num_tiles) {
                if (seg != nullptr) seg[num_tiles] = (int32_t)upto.at;
                plan_seg[num_tiles] = (int32_t)upto.plan_at;
            }
        }
    } else {
        slot = own_tile < num_tiles ? (size_t)plan_seg[own_tile] : 0;
    }
    // (a tile without an offset owns one row of missing neighbors: any offset's)
    const uint32_t given = own_tile < num_tiles ? (uint32_t)tile_code[own_tile] : 0u;
    const uint32_t code = own_tile < num_tiles && given == 0u ? 1u : given;
    const int ways = kFillThreads / R, way = tid / R, mine_r = tid % R;        // (whole wavefronts share a way)
    const int cnt = __popc(code), in_tile = together > 1 ? mine_r % tile_rows : mine_r;
    if (tid < R && in_tile < 32) {
        bands[sub][in_tile] = 0u;
        if (code >> in_tile & 1u) offsets[sub][__popc(code & ((1u << in_tile) - 1u))] = (uint32_t)in_tile;
    }
    for (int r0 = 0; r0 < all_rows; r0 += R) {
        if (r0 > 0) {
            __syncthreads();                     // the previous chunk's rows have been consumed
            fetch_order(r0);
        }
        __syncthreads();
        for (int i0 = 0; i0 < R * 32; i0 += 8 * kFillThreads) {      // eight loads in flight per thread
            uint32_t word[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int i = i0 + q * kFillThreads + tid;
                const int64_t src = i < R * 32 ? src_row[i >> 5] : -1;
                word[q] = ((i & 31) < V && src >= 0) ? map[(size_t)src * V + (i & 31)] : FGX_EMPTY32;
            }
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                const int i = i0 + q * kFillThreads + tid;
                if (i < R * 32 && (i & 31) < V) stage[(i >> 5) * V + (i & 31)] = word[q];
            }
        }
        __syncthreads();
        const int r = r0 + in_tile;
        for (int k = way; k < cnt; k += ways) {
            const uint32_t m = stage[mine_r * V + offsets[sub][k]];  // (a row past the end is EMPTY throughout)
            if (r < tile_rows) plan_idx[(slot + k) * tile_rows + r] = m;
            if (plan_band != nullptr) {
                const unsigned long long live = __ballot(m != FGX_EMPTY32);    // all 64 lanes take part
                if (lane == 0) {
                    const int b0 = (r0 + (in_tile & ~63)) >> 5;                // band of this wavefront's lanes 0-31
                    uint32_t bits = ((live & 0xFFFFFFFFull) ? 1u : 0u) << (b0 & 31);
                    bits |= ((live >> 32) ? 1u : 0u) << ((b0 + 1) & 31);
                    if (bits) atomicOr(&bands[sub][k], bits);
                }
            }
        }
    }
    if (plan_band != nullptr) {
        __syncthreads();
        if (tid < R && in_tile < cnt) plan_band[slot + in_tile] = bands[sub][in_tile];
    }
}

// Tiles of 64 or 128 rows that a workgroup fills together, as many rows at a time as of a longer one, once the workgroups left are as many as CUs: a workgroup
// takes 6 us whatever its rows, and 1 024 of them fit the chip (64 rows, 1 149 tiles 18.9 -> 9.4 us; 128 rows, 1 306 tiles 20.6 -> 12.5; 322 tiles
// of 64 rows, one each, 6.1, as many of 256 8.4).
inline int fill_together(int tile_rows, size_t num_tiles) {
    int t = 1;
    while (tile_rows % 64 == 0 && 2 * t * tile_rows <= kFillRows && num_tiles >= (size_t)512 * t) t *= 2;
    return t;
}
inline int fill_rows(int tile_rows) { return tile_rows <= 64 ? 64 : tile_rows <= 128 ? 128 : kFillRows; }
inline size_t fill_lds(int tile_rows, int V) { return (size_t)fill_rows(tile_rows) * V * 4; }

struct PairLayout {
    unsigned nblk;
    size_t counts, offsets, totals, total;
};

PairLayout pair_layout(size_t n, int V) {
    PairLayout L{};
    L.nblk = cdiv(n, kPairRows);
    size_t cnt = (size_t)L.nblk * V;
    size_t off = 0;
    L.counts = off;  off = align_up(off + (cnt ? cnt : 1) * 4, 256);
    L.offsets = off; off = align_up(off + (cnt ? cnt : 1) * 4, 256);
    L.totals = off;  off += 256;
    L.total = off;
    return L;
}

int pair_fill_launch(const uint32_t* map, const int32_t* gray, size_t n, int V, const uint32_t* offsets, const uint32_t* totals, uint32_t* seg,
                     uint32_t* seg_host, uint32_t* sig_i, uint32_t* sig_o, hipStream_t s) {
    const size_t lds = ((size_t)kPairThreads * V + 2 * (kPairThreads / 64) * 32 + 32) * sizeof(uint32_t);
    const unsigned nblk = cdiv(n, kPairRows);
    if (V == 27) pair_fill_kernel<27><<<nblk, kPairThreads, lds, s>>>(map, gray, n, V, nblk, offsets, totals, seg, seg_host, sig_i, sig_o);
    else if (V == 8) pair_fill_kernel<8><<<nblk, kPairThreads, lds, s>>>(map, gray, n, V, nblk, offsets, totals, seg, seg_host, sig_i, sig_o);
    else pair_fill_kernel<0><<<nblk, kPairThreads, lds, s>>>(map, gray, n, V, nblk, offsets, totals, seg, seg_host, sig_i, sig_o);
    FGX_CHECK_LAUNCH("fgx_pair_fill");
    return FGX_OK;
}

// Rows ranked along the Z-order curve (batch index above 3 * bits interleaved coordinate bits): a radix sort over the key
// bits a coordinate of the grid can differ in, on 32-bit keys when they fit.  The ranking goes to wide[] (64-bit) or, when
// that is null, to *ranked (a buffer of the workspace).
int zorder_rank(const int32_t* coords, size_t n, int bits_per_axis, int batch_bits, const LocalityLayout& L, char* ws,
                const uint32_t** ranked, int64_t* wide, hipStream_t s, const char* what) {
    const unsigned grid = cdiv(n, kBlock);
    const unsigned end_bit = (unsigned)(3 * bits_per_axis + batch_bits);
    uint32_t* vals_a = (uint32_t*)(ws + L.vals_a);
    uint32_t* vals_b = (uint32_t*)(ws + L.vals_b);
    size_t temp_bytes = L.temp_bytes;
    if (end_bit <= 32) {
        uint32_t* keys_a = (uint32_t*)(ws + L.keys_a);
        uint32_t* keys_b = (uint32_t*)(ws + L.keys_b);
        morton_key_packed_kernel<uint32_t><<<grid, kBlock, 0, s>>>(coords, n, bits_per_axis, keys_a, vals_a);
        FGX_CHECK_LAUNCH(what);
        if (n <= kRsMaxItems)
            return radix_sort_pairs_u32(keys_a, nullptr, n, end_bit, false, ws + L.radix, radix_layout(n), nullptr, ranked, wide, s, what);
        FGX_CHECK_HIP(rocprim::radix_sort_pairs(ws + L.temp, temp_bytes, keys_a, keys_b, vals_a, vals_b, n, 0u, end_bit, s));
    } else {
        uint64_t* keys_a = (uint64_t*)(ws + L.keys_a);
        uint64_t* keys_b = (uint64_t*)(ws + L.keys_b);
        morton_key_packed_kernel<uint64_t><<<grid, kBlock, 0, s>>>(coords, n, bits_per_axis, keys_a, vals_a);
        FGX_CHECK_LAUNCH(what);
        FGX_CHECK_HIP(rocprim::radix_sort_pairs(ws + L.temp, temp_bytes, keys_a, keys_b, vals_a, vals_b, n, 0u, end_bit, s));
    }
    *ranked = vals_b;
    if (wide != nullptr) {
        widen_u32_i64_kernel<<<grid, kBlock, 0, s>>>(vals_b, wide, n);
        FGX_CHECK_LAUNCH(what);
    }
    return FGX_OK;
}

}  // namespace

int pair_counts(const int32_t* gray, size_t n, int V, uint32_t* counts, hipStream_t s) {
    const unsigned nblk = cdiv(n, kPairRows);
    phase_mark("pair count", s);
    pair_count_kernel<<<nblk, kPairThreads, 0, s>>>(gray, n, V, nblk, counts);
    FGX_CHECK_LAUNCH("fgx_pair_count(count)");
    return FGX_OK;
}

int pair_lists_from_counts(const uint32_t* map, const int32_t* gray, size_t n, int V, const uint32_t* counts, size_t m, bool sub,
                           uint32_t* offsets, uint32_t* totals, uint32_t* seg, uint32_t* seg_host, uint32_t* sig_i, uint32_t* sig_o,
                           hipStream_t s) {
    const unsigned nblk = cdiv(n, kPairRows);
    phase_mark("pair fill", s);
    if (sub) pair_scan_kernel<kPairRows / kPairSubRows><<<V, 256, 0, s>>>(counts, m, nblk, offsets, totals);
    else pair_scan_kernel<1><<<V, 256, 0, s>>>(counts, m, nblk, offsets, totals);
    FGX_CHECK_LAUNCH("fgx_pair_count(scan)");
    return pair_fill_launch(map, gray, n, V, offsets, totals, seg, seg_host, sig_i, sig_o, s);
}

}  // namespace fgx

using namespace fgx;

extern "C" {

size_t fgx_sort_workspace_bytes(size_t n) {
    if (n <= kRankSortMax) return 256;
    return n <= kRsMaxItems ? radix_layout(n).total : sort_layout(n).total;
}

int fgx_sort_by_code(const int32_t* binary, size_t n, int V, int64_t* sorted_idx, void* workspace,
                     size_t workspace_bytes, fgx_stream_t stream) {
    FGX_CHECK_ARG(V >= 1 && V <= 32, "fgx_sort_by_code: kernel volume must be in [1, 32], got %d", V);
    FGX_CHECK_ARG(n < 0xFFFFFFFFull, "fgx_sort_by_code: too many rows");
    if (n == 0) return FGX_OK;
    const size_t need = fgx_sort_workspace_bytes(n);
    FGX_CHECK_ARG(binary && sorted_idx && workspace, "fgx_sort_by_code: null buffer");
    FGX_CHECK_ARG(workspace_bytes >= need, "fgx_sort_by_code: workspace of %zu bytes, need %zu", workspace_bytes, need);
    FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fgx_sort_by_code: workspace must be 256-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    PhaseEnd phases{s};
    phase_mark("mask sort", s);
    // With V < 32 every key is non-negative and only bits [0, V) can differ.
    const unsigned end_bit = V < 32 ? (unsigned)V : 32u;
    if (n <= kRankSortMax) {
        rank_sort_kernel<<<cdiv(n, 64), 64 * kRankSlices, 0, s>>>((const uint32_t*)binary, (uint32_t)n, V == 32 ? 0x80000000u : 0u, sorted_idx);
        FGX_CHECK_LAUNCH("fgx_sort_by_code(rank)");
        return FGX_OK;
    }
    if (n <= kRsMaxItems)       // the first pass numbers the rows itself and the last one writes the 64-bit indices
        return radix_sort_pairs_u32((const uint32_t*)binary, nullptr, n, end_bit, true, ws, radix_layout(n), nullptr, nullptr, sorted_idx,
                                    s, "fgx_sort_by_code");
    const SortLayout L = sort_layout(n);
    int32_t* keys_out = (int32_t*)(ws + L.keys_out);
    uint32_t* vals_in = (uint32_t*)(ws + L.vals_in);
    uint32_t* vals_out = (uint32_t*)(ws + L.vals_out);
    iota_u32_kernel<<<cdiv(n, kBlock), kBlock, 0, s>>>(vals_in, n);
    FGX_CHECK_LAUNCH("fgx_sort_by_code(iota)");
    size_t temp_bytes = L.temp_bytes;
    FGX_CHECK_HIP(rocprim::radix_sort_pairs(ws + L.temp, temp_bytes, binary, keys_out, vals_in, vals_out, n, 0u, end_bit, s));
    widen_u32_i64_kernel<<<cdiv(n, kBlock), kBlock, 0, s>>>(vals_out, sorted_idx, n);
    FGX_CHECK_LAUNCH("fgx_sort_by_code(widen)");
    return FGX_OK;
}

size_t fgx_locality_workspace_bytes(size_t n) { return locality_layout(n).total; }

int fgx_locality_order_grid(const int32_t* coords, const int32_t* binary, size_t n, int V, int chunk_rows, int bits_per_axis,
                            int batch_bits, int64_t* order, void* workspace, size_t workspace_bytes, fgx_stream_t stream) {
    FGX_CHECK_ARG(V >= 1 && V <= 32, "fgx_locality_order: kernel volume must be in [1, 32], got %d", V);
    FGX_CHECK_ARG(chunk_rows >= 1, "fgx_locality_order: chunk_rows must be positive, got %d", chunk_rows);
    FGX_CHECK_ARG(bits_per_axis >= 1 && bits_per_axis <= 16 && batch_bits >= 0 && 3 * bits_per_axis + batch_bits <= 64,
                  "fgx_locality_order: %d bits per axis and %d batch bits do not fit a 64-bit key", bits_per_axis, batch_bits);
    FGX_CHECK_ARG(n < 0xFFFFFFFFull, "fgx_locality_order: too many rows");
    if (n == 0) return FGX_OK;
    LocalityLayout L = locality_layout(n);
    FGX_CHECK_ARG(coords && binary && order && workspace, "fgx_locality_order: null buffer");
    FGX_CHECK_ARG(((uintptr_t)coords & 15) == 0, "fgx_locality_order: coords must be 16-byte aligned");
    FGX_CHECK_ARG(workspace_bytes >= L.total, "fgx_locality_order: workspace of %zu bytes, need %zu", workspace_bytes, L.total);
    FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fgx_locality_order: workspace must be 256-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    uint64_t* keys_a = (uint64_t*)(ws + L.keys_a);
    uint64_t* keys_b = (uint64_t*)(ws + L.keys_b);
    uint32_t* vals_a = (uint32_t*)(ws + L.vals_a);
    const unsigned grid = cdiv(n, kBlock);
    const uint32_t* ranked = nullptr;
    // (chunks of one rank: the curve's own order, nothing to sort inside them)
    int rc = zorder_rank(coords, n, bits_per_axis, batch_bits, L, ws, &ranked, chunk_rows == 1 ? order : nullptr, s, "fgx_locality_order(keys)");
    if (rc != FGX_OK || chunk_rows == 1) return rc;
    // (chunk, mask code) keys with the chunk right above the V code bits: the sort runs over the bits in use alone
    chunk_code_key_kernel<<<grid, kBlock, 0, s>>>(ranked, binary, n, (uint32_t)chunk_rows, V, keys_a);
    FGX_CHECK_LAUNCH("fgx_locality_order(chunk keys)");
    const unsigned end_bit = (unsigned)V + (unsigned)bits_for((n - 1) / (size_t)chunk_rows);
    size_t temp_bytes = L.temp_bytes;
    FGX_CHECK_HIP(rocprim::radix_sort_pairs(ws + L.temp, temp_bytes, keys_a, keys_b, ranked, vals_a, n, 0u, end_bit, s));
    widen_u32_i64_kernel<<<grid, kBlock, 0, s>>>(vals_a, order, n);
    FGX_CHECK_LAUNCH("fgx_locality_order(widen)");
    return FGX_OK;
}

int fgx_locality_order(const int32_t* coords, const int32_t* binary, size_t n, int V, int chunk_rows, int64_t* order,
                       void* workspace, size_t workspace_bytes, fgx_stream_t stream) {
    // coordinates of any grid: 16 bits per axis and 16 bits of batch index
    return fgx_locality_order_grid(coords, binary, n, V, chunk_rows, 16, 16, order, workspace, workspace_bytes, stream);
}

int fgx_zorder_rows(const int32_t* coords, size_t n, int bits_per_axis, int batch_bits, int64_t* order, void* workspace,
                    size_t workspace_bytes, fgx_stream_t stream) {
    FGX_CHECK_ARG(bits_per_axis >= 1 && bits_per_axis <= 16 && batch_bits >= 0 && 3 * bits_per_axis + batch_bits <= 64,
                  "fgx_zorder_rows: %d bits per axis and %d batch bits do not fit a 64-bit key", bits_per_axis, batch_bits);
    FGX_CHECK_ARG(n < 0xFFFFFFFFull, "fgx_zorder_rows: too many rows");
    if (n == 0) return FGX_OK;
    LocalityLayout L = locality_layout(n);
    FGX_CHECK_ARG(coords && order && workspace, "fgx_zorder_rows: null buffer");
    FGX_CHECK_ARG(((uintptr_t)coords & 15) == 0, "fgx_zorder_rows: coords must be 16-byte aligned");
    FGX_CHECK_ARG(workspace_bytes >= L.total, "fgx_zorder_rows: workspace of %zu bytes, need %zu", workspace_bytes, L.total);
    FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fgx_zorder_rows: workspace must be 256-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    const uint32_t* ranked = nullptr;
    return zorder_rank(coords, n, bits_per_axis, batch_bits, L, ws, &ranked, order, s, "fgx_zorder_rows(keys)");
}

size_t fgx_pair_workspace_bytes(size_t n, int V) { return pair_layout(n, V > 0 ? V : 1).total; }

int fgx_pair_count(const int32_t* gray, size_t n, int V, uint32_t* seg, void* workspace, size_t workspace_bytes,
                   fgx_stream_t stream) {
    FGX_CHECK_ARG(V >= 1 && V <= 32, "fgx_pair_count: kernel volume must be in [1, 32], got %d", V);
    FGX_CHECK_ARG(seg != nullptr, "fgx_pair_count: null segment table");
    FGX_CHECK_ARG(n * (size_t)V < 0xFFFFFFFFull, "fgx_pair_count: pair offsets must fit in 32 bits");
    hipStream_t s = (hipStream_t)stream;
    PairLayout L = pair_layout(n, V);
    if (n > 0) {
        FGX_CHECK_ARG(gray && workspace, "fgx_pair_count: null buffer");
        FGX_CHECK_ARG(workspace_bytes >= L.total, "fgx_pair_count: workspace of %zu bytes, need %zu", workspace_bytes, L.total);
        FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fgx_pair_count: workspace must be 256-byte aligned");
    }
    char* ws = (char*)workspace;
    PhaseEnd phases{s};
    phase_mark("pair count", s);
    uint32_t* totals = n ? (uint32_t*)(ws + L.totals) : nullptr;
    if (n > 0) {
        uint32_t* counts = (uint32_t*)(ws + L.counts);
        const int rc = pair_counts(gray, n, V, counts, s);
        if (rc != FGX_OK) return rc;
        pair_scan_kernel<1><<<V, 256, 0, s>>>(counts, L.nblk, L.nblk, (uint32_t*)(ws + L.offsets), totals);
        FGX_CHECK_LAUNCH("fgx_pair_count(scan)");
    }
    pair_seg_kernel<<<1, 64, 0, s>>>(totals, V, seg);
    FGX_CHECK_LAUNCH("fgx_pair_count(seg)");
    return FGX_OK;
}

int fgx_pair_fill(const uint32_t* map, const int32_t* gray, size_t n, int V, const void* workspace, uint32_t* sig_i,
                  uint32_t* sig_o, fgx_stream_t stream) {
    FGX_CHECK_ARG(V >= 1 && V <= 32, "fgx_pair_fill: kernel volume must be in [1, 32], got %d", V);
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(map && gray && workspace && sig_i && sig_o, "fgx_pair_fill: null buffer");
    const PairLayout L = pair_layout(n, V);
    const char* ws = (const char*)workspace;
    PhaseEnd phases{(hipStream_t)stream};
    phase_mark("pair fill", (hipStream_t)stream);
    return pair_fill_launch(map, gray, n, V, (const uint32_t*)(ws + L.offsets), (const uint32_t*)(ws + L.totals), nullptr, nullptr, sig_i, sig_o,
                            (hipStream_t)stream);
}

size_t fgx_tile_workspace_bytes(size_t n, int block) {
    (void)n;
    (void)block;
    return 256;         // (the scans need none any more)
}

int fgx_tile_codes(const int32_t* gray, const int64_t* sorted_idx, size_t n, int block, int32_t* tile_code,
                   int32_t* seg, void* workspace, size_t workspace_bytes, fgx_stream_t stream) {
    (void)workspace;
    (void)workspace_bytes;
    FGX_CHECK_ARG(block >= 1, "fgx_tile_codes: tile size must be >= 1, got %d", block);
    FGX_CHECK_ARG(seg != nullptr, "fgx_tile_codes: null segment table");
    return fgx_tile_plan(gray, sorted_idx, nullptr, n, 1, block, 0, tile_code, seg, nullptr, nullptr, nullptr, 1, 1, 1, nullptr, nullptr, stream);
}

int fgx_tile_plan(const int32_t* gray, const int64_t* order, const uint32_t* map, size_t n, int V, int tile_rows, int have_codes,
                  int32_t* tile_code, int32_t* seg, int32_t* plan_seg, uint32_t* plan_idx, uint32_t* plan_band, int col_tiles, int slabs,
                  int groups, uint32_t* item_ws, uint32_t* item_at, fgx_stream_t stream) {
    FGX_CHECK_ARG(tile_rows >= 1 && V >= 1 && V <= 32, "fgx_tile_plan: bad shape tile_rows=%d V=%d", tile_rows, V);
    hipStream_t s = (hipStream_t)stream;
    const size_t num_tiles = (n + tile_rows - 1) / tile_rows;
    FGX_CHECK_ARG(num_tiles <= 0x7FFFFFFFu, "fgx_tile_plan: too many tiles");
    PhaseEnd phases{s};
    phase_mark("tile tables", s);
    if (n == 0) {
        for (int32_t* table : {seg, plan_seg})
            if (table != nullptr) set_i32_kernel<<<1, 64, 0, s>>>(table, 0);
        FGX_CHECK_LAUNCH("fgx_tile_plan(empty)");
        return FGX_OK;
    }
    FGX_CHECK_ARG(tile_code && (have_codes || (gray && order)), "fgx_tile_plan: null buffer");
    FGX_CHECK_ARG(plan_idx == nullptr || (map && order && plan_seg), "fgx_tile_plan: a gather plan needs the map, the order and its segment table");
    FGX_CHECK_ARG(plan_band == nullptr || (plan_idx != nullptr && tile_rows <= 1024), "fgx_tile_plan: band masks need a plan and tile_rows <= 1024");
    if (item_at != nullptr) {
        FGX_CHECK_ARG(col_tiles >= 1 && slabs >= 1 && groups >= 1 && groups <= kOrderThreads && item_ws != nullptr,
                      "fgx_tile_plan: bad item order col_tiles=%d slabs=%d groups=%d", col_tiles, slabs, groups);
        FGX_CHECK_ARG(num_tiles * (size_t)col_tiles < 0x7FFFFFFFull, "fgx_tile_plan: too many items");
    }
    if (!have_codes) {
        const size_t groups_or = cdiv(num_tiles, (size_t)(kBlock / 64)), most = (size_t)0xFFFFFFFFu / kBlock;       // (of one launch)
        tile_or_kernel<<<(unsigned)(groups_or < most ? groups_or : most), kBlock, 0, s>>>(gray, order, n, tile_rows, num_tiles, tile_code);
        FGX_CHECK_LAUNCH("fgx_tile_plan(or)");
    }
    bool scans = seg != nullptr || plan_seg != nullptr;
    if (scans && num_tiles > kOneScanTiles) {
        const unsigned chunks = cdiv(num_tiles, kScanChunk);
        tile_sums_kernel<<<chunks, kOrderThreads, 0, s>>>(tile_code, (unsigned)num_tiles, seg, plan_seg);
        chunk_scan_kernel<<<1, kOrderThreads, 0, s>>>((unsigned)num_tiles, chunks, seg, plan_seg);
        chunk_tables_kernel<<<chunks, kOrderThreads, 0, s>>>(tile_code, (unsigned)num_tiles, seg, plan_seg);
        FGX_CHECK_LAUNCH("fgx_tile_plan(chunks)");
        scans = false;
    }
    const size_t items = item_at != nullptr ? num_tiles * (size_t)col_tiles : 0;
    const int together = fill_together(tile_rows, num_tiles);
    const unsigned fills = (unsigned)cdiv(num_tiles, (size_t)together);
    if (plan_idx != nullptr && num_tiles <= kFillScanTiles && items < ((size_t)1 << kItemBits) && (item_at == nullptr || groups <= kFillThreads)) {
        const size_t lds = fill_lds(together * tile_rows, V), list = items <= kOrderInLds ? items * 4 : 0;
        phase_mark("gather plan fill", s);
        plan_fill_kernel<true><<<fills + (item_at != nullptr ? 1u : 0u), kFillThreads, lds > list ? lds : list, s>>>(
            map, order, tile_code, num_tiles, n, V, tile_rows, fill_rows(together * tile_rows), seg, plan_seg, plan_idx, plan_band, (unsigned)col_tiles,
            (unsigned)slabs, (unsigned)groups, item_ws, item_at, together);
        FGX_CHECK_LAUNCH("fgx_tile_plan(tables and plan)");
        return FGX_OK;
    }
    if (scans || item_at != nullptr) {
        tile_tables_kernel<<<1, kOrderThreads, 0, s>>>(tile_code, (unsigned)num_tiles, scans ? seg : nullptr, scans ? plan_seg : nullptr,
                                                       (unsigned)col_tiles, (unsigned)slabs, (unsigned)groups, item_ws, item_at);
        FGX_CHECK_LAUNCH("fgx_tile_plan(tables)");
    }
    if (plan_idx != nullptr) {
        phase_mark("gather plan fill", s);
        plan_fill_kernel<false><<<fills, kFillThreads, fill_lds(together * tile_rows, V), s>>>(map, order, tile_code, num_tiles, n, V, tile_rows, fill_rows(together * tile_rows),
                                                                              nullptr, plan_seg, plan_idx, plan_band, 1, 1, 1, nullptr, nullptr, together);
        FGX_CHECK_LAUNCH("fgx_tile_plan(plan)");
    }
    return FGX_OK;
}

int fgx_tile_fill(const int32_t* tile_code, const int32_t* seg, size_t num_tiles, int32_t* valid_kernel,
                  fgx_stream_t stream) {
    if (num_tiles == 0) return FGX_OK;
    FGX_CHECK_ARG(tile_code && seg && valid_kernel, "fgx_tile_fill: null buffer");
    tile_fill_kernel<<<cdiv(num_tiles, kBlock), kBlock, 0, (hipStream_t)stream>>>(tile_code, seg, num_tiles, valid_kernel);
    FGX_CHECK_LAUNCH("fgx_tile_fill");
    return FGX_OK;
}

int fgx_gather_plan_count(const int32_t* tile_code, size_t num_tiles, int32_t* plan_seg, void* workspace,
                          size_t workspace_bytes, fgx_stream_t stream) {
    (void)workspace;
    (void)workspace_bytes;
    FGX_CHECK_ARG(plan_seg != nullptr, "fgx_gather_plan_count: null segment table");
    // (tiles of one row: as many tiles as rows)
    return fgx_tile_plan(nullptr, nullptr, nullptr, num_tiles, 1, 1, 1, const_cast<int32_t*>(tile_code), nullptr, plan_seg, nullptr, nullptr, 1,
                         1, 1, nullptr, nullptr, stream);
}

int fgx_gather_plan_fill(const uint32_t* map, const int64_t* order, const int32_t* tile_code, const int32_t* plan_seg,
                         size_t n, int V, int tile_rows, uint32_t* plan_idx, uint32_t* plan_band, fgx_stream_t stream) {
    FGX_CHECK_ARG(tile_rows >= 1 && V >= 1 && V <= 32, "fgx_gather_plan_fill: bad shape tile_rows=%d V=%d", tile_rows, V);
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(map && order && tile_code && plan_seg && plan_idx, "fgx_gather_plan_fill: null buffer");
    const size_t num_tiles = (n + tile_rows - 1) / tile_rows;
    FGX_CHECK_ARG(num_tiles <= 0x7FFFFFFFu, "fgx_gather_plan_fill: too many tiles");
    FGX_CHECK_ARG(plan_band == nullptr || tile_rows <= 1024, "fgx_gather_plan_fill: band masks need tile_rows <= 1024");
    PhaseEnd phases{(hipStream_t)stream};
    phase_mark("gather plan fill", (hipStream_t)stream);
    const int together = fill_together(tile_rows, num_tiles);
    plan_fill_kernel<false><<<(unsigned)cdiv(num_tiles, (size_t)together), kFillThreads, fill_lds(together * tile_rows, V), (hipStream_t)stream>>>(
        map, order, tile_code, num_tiles, n, V, tile_rows, fill_rows(together * tile_rows), nullptr, const_cast<int32_t*>(plan_seg), plan_idx, plan_band, 1,
        1, 1, nullptr, nullptr, together);
    FGX_CHECK_LAUNCH("fgx_gather_plan_fill");
    return FGX_OK;
}

size_t fgx_gather_item_order_workspace_bytes(size_t num_tiles, int col_tiles) {
    if (col_tiles < 1) return 0;
    return align_up((num_tiles * (size_t)col_tiles + 1) * sizeof(uint32_t), 256);
}

int fgx_gather_item_order(const int32_t* tile_code, size_t num_tiles, int col_tiles, int slabs, int groups, void* workspace,
                          size_t workspace_bytes, uint32_t* item_at, fgx_stream_t stream) {
    FGX_CHECK_ARG(col_tiles >= 1 && slabs >= 1, "fgx_gather_item_order: bad shape col_tiles=%d slabs=%d", col_tiles, slabs);
    FGX_CHECK_ARG(groups >= 1 && groups <= kOrderThreads, "fgx_gather_item_order: groups must be in [1, %d], got %d", kOrderThreads,
                  groups);
    const size_t total = num_tiles * (size_t)col_tiles;
    if (total == 0) return FGX_OK;
    FGX_CHECK_ARG(total < 0x7FFFFFFFull, "fgx_gather_item_order: too many items");
    FGX_CHECK_ARG(tile_code && workspace && item_at, "fgx_gather_item_order: null buffer");
    FGX_CHECK_ARG(workspace_bytes >= fgx_gather_item_order_workspace_bytes(num_tiles, col_tiles),
                  "fgx_gather_item_order: workspace of %zu bytes is too small", workspace_bytes);
    FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fgx_gather_item_order: workspace must be 256-byte aligned");
    tile_tables_kernel<<<1, kOrderThreads, 0, (hipStream_t)stream>>>(tile_code, (unsigned)num_tiles, nullptr, nullptr, (unsigned)col_tiles,
                                                                     (unsigned)slabs, (unsigned)groups, (uint32_t*)workspace, item_at);
    FGX_CHECK_LAUNCH("fgx_gather_item_order");
    return FGX_OK;
}

}  // extern "C"
