// Stable LSD radix sort of (32-bit key, row index) pairs for gfx950, for the sorts of the neighbor-cache build:
// some ten thousand to some million items whose keys have 20 ... 32 significant bits.
//
// Every pass is three launches over digits of up to 9 bits (27-bit mask keys: three passes): a histogram per tile, an
// exclusive scan over the [digit][tile] table (one workgroup per digit scans its row of tiles and leaves the row's total),
// and a scatter.  The scatter's wavefronts walk contiguous pieces of the tile 64 items at a time -- the lanes holding the
// same digit find each other with one ballot per digit bit -- and count in LDS, so equal digits keep their order; the
// tile is then put in digit order in LDS and leaves as runs of consecutive words.  What bounds it is launches for few
// rows and the 16 bytes per row and pass for many.  Measured for the mask sort (27-bit keys, three passes): 2 667 120 rows
// 0.113 ms (library onesweep 0.172), 669 288 rows 0.067 (0.089 with every item written from where it was read), 166 232
// rows 0.041 (library block sort and merges 0.063).
// The first pass can take the row index from the item's position, the last pass can write 64-bit indices and drop the keys.
#pragma once
#include "fgx_common.h"

namespace fgx {
namespace {

constexpr int kRsThreads = 512;
constexpr int kRsWaves = kRsThreads / 64;
constexpr int kRsMaxBits = 9;             // digit width limit: 512 counters of LDS per wavefront
constexpr int kRsBins = 1 << kRsMaxBits;
constexpr size_t kRsMaxItems = (size_t)1 << 30;

// tiles of 1024 items keep every CU busy on a few hundred thousand items, tiles of 4096 write longer runs
constexpr size_t kRsLongTilesFrom = 786432;

inline int radix_items_per_thread(size_t n) { return n >= kRsLongTilesFrom ? 8 : 2; }

struct RadixLayout {
    unsigned tiles;
    int items;          // per thread
    size_t keys_a, keys_b, vals_a, vals_b, hist, offs, totals, total;
};

inline RadixLayout radix_layout(size_t n) {
    RadixLayout L{};
    const size_t nn = n ? n : 1;
    L.items = radix_items_per_thread(nn);
    L.tiles = cdiv(nn, (size_t)kRsThreads * L.items);
    size_t off = 0;
    L.keys_a = off;
    off = align_up(off + nn * 4, 256);
    L.keys_b = off;
    off = align_up(off + nn * 4, 256);
    L.vals_a = off;
    off = align_up(off + nn * 4, 256);
    L.vals_b = off;
    off = align_up(off + nn * 4, 256);
    L.hist = off;
    const size_t entries = (size_t)kRsBins * L.tiles;
    off = align_up(off + entries * 4, 256);
    L.offs = off;
    off = align_up(off + entries * 4, 256);
    L.totals = off;
    off = align_up(off + (size_t)kRsBins * 4, 256);
    L.total = off;
    return L;
}

// lanes of the wavefront (of those with `live`) whose digit equals this lane's: one ballot per digit bit
__device__ __forceinline__ unsigned long long radix_peers(uint32_t digit, unsigned bits, bool live) {
    unsigned long long peers = __ballot(live);
    for (unsigned b = 0; b < bits; ++b) {
        const bool bit = (digit >> b) & 1u;
        const unsigned long long have = __ballot(bit);
        peers &= bit ? have : ~have;
    }
    return peers;
}

// hist[digit * tiles + tile] = items of the tile with that digit.  run_if != nullptr: the whole sort is conditional on that
// word, which an earlier kernel of the stream has written -- every wavefront returns at once when it is zero.
template <int ITEMS>
__global__ void __launch_bounds__(kRsThreads) radix_hist_kernel(const uint32_t* __restrict__ keys, size_t n, unsigned shift,
                                                                unsigned bits, uint32_t flip, unsigned tiles,
                                                                uint32_t* __restrict__ hist, const uint32_t* __restrict__ run_if) {
    if (run_if != nullptr && *run_if == 0u) return;
    __shared__ uint32_t count[kRsBins];
    const unsigned bins = 1u << bits, mask = bins - 1u;
    for (unsigned b = threadIdx.x; b < bins; b += kRsThreads) count[b] = 0u;
    const size_t base = (size_t)blockIdx.x * (kRsThreads * ITEMS) + threadIdx.x;
    uint32_t key[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {               // all loads of the tile in flight together
        const size_t i = base + (size_t)r * kRsThreads;
        key[r] = i < n ? keys[i] ^ flip : 0u;
    }
    __syncthreads();
    // neighboring rows often share their digit: equal ones are counted by one lane (64 lanes adding to one counter take turns)
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool live = base + (size_t)r * kRsThreads < n;
        const uint32_t digit = (key[r] >> shift) & mask;
        const unsigned long long peers = radix_peers(digit, bits, live);
        if (live && (threadIdx.x & 63u) == (unsigned)(__ffsll((long long)peers) - 1)) atomicAdd(&count[digit], (uint32_t)__popcll(peers));
    }
    __syncthreads();
    for (unsigned b = threadIdx.x; b < bins; b += kRsThreads) hist[(size_t)b * tiles + blockIdx.x] = count[b];
}

// exclusive sum of `v` over the workgroup's threads; *total: the sum of all.  `part`: one word per wavefront.
template <int WAVES>
__device__ __forceinline__ uint32_t block_exclusive_sum(uint32_t v, uint32_t* part, uint32_t* total) {
    const unsigned lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    uint32_t incl = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
        if ((int)lane >= d) incl += o;
    }
    __syncthreads();                                // an earlier use of `part` is over
    if (lane == 63u) part[wave] = incl;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        const uint32_t p = part[w];
        before += w < (int)wave ? p : 0u;
        all += p;
    }
    *total = all;
    return before + incl - v;
}

// offs[digit][tile] = items with that digit in the tiles before this one; totals[digit] = items with that digit.  One
// workgroup per digit, 4 consecutive tiles per thread and turn.
__global__ void __launch_bounds__(256) radix_row_scan_kernel(const uint32_t* __restrict__ hist, unsigned tiles,
                                                             uint32_t* __restrict__ offs, uint32_t* __restrict__ totals,
                                                             const uint32_t* __restrict__ run_if) {
    if (run_if != nullptr && *run_if == 0u) return;
    __shared__ uint32_t part[4];
    const uint32_t* row = hist + (size_t)blockIdx.x * tiles;
    uint32_t* out = offs + (size_t)blockIdx.x * tiles;
    uint32_t carry = 0u;
    for (unsigned t0 = 0; t0 < tiles; t0 += 1024) {             // (uniform)
        const unsigned t = t0 + threadIdx.x * 4;
        uint32_t v[4], sum = 0u, all;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            v[k] = t + k < tiles ? row[t + k] : 0u;
            sum += v[k];
        }
        uint32_t run = carry + block_exclusive_sum<4>(sum, part, &all);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if (t + k < tiles) out[t + k] = run;
            run += v[k];
        }
        carry += all;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// Item i of the tile goes to (items with a lower digit) + offs[digit][tile] + (items of the tile with the same
// digit before it).  vals_in == nullptr: the value is the item's position.  out64 != nullptr: last pass, the values are
// written there as 64-bit integers and neither keys nor 32-bit values are written.
template <int ITEMS>
__global__ void __launch_bounds__(kRsThreads) radix_scatter_kernel(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals_in,
                                                                   size_t n, unsigned shift, unsigned bits, uint32_t flip, unsigned tiles,
                                                                   const uint32_t* __restrict__ offs, const uint32_t* __restrict__ totals,
                                                                   uint32_t* __restrict__ keys_out, uint32_t* __restrict__ vals_out,
                                                                   int64_t* __restrict__ out64, const uint32_t* __restrict__ run_if) {
    if (run_if != nullptr && *run_if == 0u) return;
    constexpr int kTile = kRsThreads * ITEMS;
    __shared__ uint32_t count[kRsWaves][kRsBins];       // items per wavefront and digit, then the digit's first place per wavefront
    __shared__ uint32_t to_global[kRsBins];             // add to a place in the tile's digit order: the place in the output
    __shared__ uint32_t part[kRsWaves];
    __shared__ uint32_t skey[kTile], sval[kTile];
    const unsigned bins = 1u << bits, mask = bins - 1u;
    const unsigned tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const size_t base = (size_t)blockIdx.x * kTile;
    const unsigned len = n - base < (size_t)kTile ? (unsigned)(n - base) : (unsigned)kTile;
    static_assert(kRsBins <= kRsThreads, "a digit per thread");
    const uint32_t dig_total = tid < bins ? totals[tid] : 0u;
    const uint32_t dig_offs = tid < bins ? offs[(size_t)tid * tiles + blockIdx.x] : 0u;
    uint32_t key_r[ITEMS], val_r[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {                   // a wavefront's piece is contiguous
        const size_t i = base + (size_t)wave * (64 * ITEMS) + r * 64 + lane;
        key_r[r] = i < n ? keys[i] ^ flip : 0u;
        val_r[r] = i < n ? (vals_in ? vals_in[i] : (uint32_t)i) : 0u;
    }
    for (unsigned b = tid; b < kRsWaves * kRsBins; b += kRsThreads) (&count[0][0])[b] = 0u;
    __syncthreads();
    const unsigned long long below = (1ull << lane) - 1ull;
    uint32_t rank_r[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool live = wave * (64 * ITEMS) + r * 64 + lane < len;
        const uint32_t digit = (key_r[r] >> shift) & mask;
        const unsigned long long peers = radix_peers(digit, bits, live);
        // the lowest lane of a run of equal digits takes the run's places; one wavefront, so LDS accesses stay in order
        const int leader = live ? __ffsll((long long)peers) - 1 : 0;
        uint32_t first = 0u;
        if (live && (int)lane == leader) {
            first = count[wave][digit];
            count[wave][digit] = first + (uint32_t)__popcll(peers);
        }
        first = (uint32_t)__shfl((int)first, leader, 64);
        rank_r[r] = first + (uint32_t)__popcll(peers & below);
    }
    __syncthreads();
    // the digits' places in the tile and in the output
    uint32_t in_tile = 0u;
    if (tid < bins)
#pragma unroll
        for (int w = 0; w < kRsWaves; ++w) {
            const uint32_t c = count[w][tid];
            count[w][tid] = in_tile;
            in_tile += c;
        }
    uint32_t all;
    const uint32_t tile_first = block_exclusive_sum<kRsWaves>(in_tile, part, &all);
    const uint32_t out_first = block_exclusive_sum<kRsWaves>(dig_total, part, &all);
    if (tid < bins) {
        to_global[tid] = out_first + dig_offs - tile_first;
#pragma unroll
        for (int w = 0; w < kRsWaves; ++w) count[w][tid] += tile_first;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r)
        if (wave * (64 * ITEMS) + r * 64 + lane < len) {
            const uint32_t at = count[wave][(key_r[r] >> shift) & mask] + rank_r[r];
            skey[at] = key_r[r];
            sval[at] = val_r[r];
        }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const unsigned at = r * kRsThreads + tid;
        if (at < len) {
            const uint32_t key = skey[at];
            const size_t pos = (size_t)(to_global[(key >> shift) & mask] + at);
            if (out64) {
                out64[pos] = (int64_t)sval[at];
            } else {
                keys_out[pos] = key ^ flip;
                vals_out[pos] = sval[at];
            }
        }
    }
}

// Sorts (keys[i], vals[i] or i) by the low `end_bit` bits of the keys, stable (all 32 bits with is_signed: as signed
// numbers).  `ws`: radix_layout(n).total bytes, 256-byte aligned.  The result ends in (*keys_sorted, *vals_sorted), which
// point into the workspace, or, with out64, in out64 alone.
// run_if (a device word, or nullptr): when it reads zero every kernel of the sort returns at once and the buffers the result
// would have ended in are left as they were.
inline int radix_sort_pairs_u32(const uint32_t* keys, const uint32_t* vals, size_t n, unsigned end_bit, bool is_signed, char* ws,
                                const RadixLayout& L, const uint32_t** keys_sorted, const uint32_t** vals_sorted, int64_t* out64,
                                hipStream_t s, const char* what, const uint32_t* run_if = nullptr) {
    if (end_bit < 1) end_bit = 1;
    if (end_bit > 32) end_bit = 32;
    const unsigned passes = (end_bit + kRsMaxBits - 1) / kRsMaxBits;
    const unsigned bits = (end_bit + passes - 1) / passes;
    const uint32_t flip = is_signed && end_bit == 32 ? 0x80000000u : 0u;
    uint32_t* kbuf[2] = {(uint32_t*)(ws + L.keys_a), (uint32_t*)(ws + L.keys_b)};
    uint32_t* vbuf[2] = {(uint32_t*)(ws + L.vals_a), (uint32_t*)(ws + L.vals_b)};
    uint32_t* hist = (uint32_t*)(ws + L.hist);
    uint32_t* offs = (uint32_t*)(ws + L.offs);
    uint32_t* totals = (uint32_t*)(ws + L.totals);
    if (n > kRsMaxItems) {
        set_error("%s: %zu items are more than the radix sort takes", what, n);
        return FGX_ERR_UNSUPPORTED;
    }
    const uint32_t* kin = keys;
    const uint32_t* vin = vals;
    for (unsigned p = 0; p < passes; ++p) {
        const unsigned shift = p * bits;
        int64_t* const wide = p + 1 == passes ? out64 : nullptr;
        if (L.items == 8) radix_hist_kernel<8><<<L.tiles, kRsThreads, 0, s>>>(kin, n, shift, bits, flip, L.tiles, hist, run_if);
        else radix_hist_kernel<2><<<L.tiles, kRsThreads, 0, s>>>(kin, n, shift, bits, flip, L.tiles, hist, run_if);
        FGX_CHECK_LAUNCH(what);
        radix_row_scan_kernel<<<1u << bits, 256, 0, s>>>(hist, L.tiles, offs, totals, run_if);
        FGX_CHECK_LAUNCH(what);
        if (L.items == 8)
            radix_scatter_kernel<8><<<L.tiles, kRsThreads, 0, s>>>(kin, vin, n, shift, bits, flip, L.tiles, offs, totals, kbuf[p & 1],
                                                                    vbuf[p & 1], wide, run_if);
        else
            radix_scatter_kernel<2><<<L.tiles, kRsThreads, 0, s>>>(kin, vin, n, shift, bits, flip, L.tiles, offs, totals, kbuf[p & 1],
                                                                   vbuf[p & 1], wide, run_if);
        FGX_CHECK_LAUNCH(what);
        kin = kbuf[p & 1];
        vin = vbuf[p & 1];
    }
    if (keys_sorted) *keys_sorted = kin;
    if (vals_sorted) *vals_sorted = vin;
    return FGX_OK;
}

}  // namespace
}  // namespace fgx
