// Neighbor maps and output coordinates through an index over the grid's cells (grid_index.h), for gfx950.
//
// What bounds it: a question is one or two loads from lines its neighbors in the walk ask for as well, so the map kernel
// runs at the rate its 4 * V bytes per row leave, and the small kernels before it at launch cost.
//
// Output coordinates of the generic convolution are the set bits of a bit map over the output grid: every (voxel, kernel
// position) candidate sets its bit, one counting pass gives their number and places, and the bits leave as coordinates in
// cell order -- the order of the sorted, unique keys the expanding builder (sparse_neighbor.hip) ends with, without
// writing, sorting and uniquing V keys per voxel.
#include "cache_parts.h"
#include "grid_index.h"
#include "narrow_plan_build.h"

namespace fgx {
namespace {

constexpr int kRowsPerGroup = 64;           // rows whose neighbors one workgroup finds: a wavefront of questions per kernel column
constexpr int kMaxStageV = 128;             // their map rows are staged in LDS: kernel volumes up to this
constexpr unsigned kLookbackValue = (1u << 30) - 1u, kLookbackSum = 1u << 30, kLookbackTotal = 2u << 30;
// The counting pass: 128-bit blocks per thread.  A large bit map takes tiles of 256 KiB of bits, so that its workgroups do not queue at the ticket
// (128 MiB: 0.063 -> 0.048 ms); one of up to 4 MiB waits for the scans one after the other of a thread's blocks, so it has two of them (tiles
// of 16 KiB against 64: 0.4 MiB 7.4 -> 5.2 us, 2 MiB 8.6 -> 6.6, 3.4 MiB 8.7 -> 8.6).
constexpr int kCountThreads = 512, kCountRowsFew = 2, kCountRowsShort = 8, kCountRowsLong = 32;
constexpr size_t kCountFewUpTo = (size_t)1 << 18, kCountLongFrom = (size_t)1 << 20;                 // blocks (4 and 16 MiB of bits)
constexpr int count_rows(size_t blocks) { return blocks > kCountLongFrom ? kCountRowsLong : (blocks > kCountFewUpTo ? kCountRowsShort : kCountRowsFew); }

static_assert(kRowsPerGroup == kPairSubRows, "the map kernel counts pairs by its own rows");

// [zero, zero + zero_pieces) := 0, 16 bytes at a time, and the words of fill := all ones
__global__ void __launch_bounds__(256) clear_kernel(uint4* __restrict__ zero, size_t zero_pieces, uint4* __restrict__ fill, size_t fill_words) {
    const size_t stride = (size_t)gridDim.x * 256;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < zero_pieces; i += stride) zero[i] = make_uint4(0u, 0u, 0u, 0u);
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < fill_words / 4; i += stride)
        fill[i] = make_uint4(FGX_EMPTY32, FGX_EMPTY32, FGX_EMPTY32, FGX_EMPTY32);
    if (blockIdx.x == 0 && threadIdx.x < (fill_words & 3)) ((uint32_t*)(fill + fill_words / 4))[threadIdx.x] = FGX_EMPTY32;
}

__device__ __forceinline__ bool in_grid(const GridIndex& g, int b, int x, int y, int z) {
    return (unsigned)b < (unsigned)g.B && (unsigned)x < (unsigned)g.W && (unsigned)y < (unsigned)g.H && (unsigned)z < (unsigned)g.D;
}

__global__ void __launch_bounds__(256) insert_cells_kernel(const int32_t* __restrict__ coords, size_t n, GridIndex g, uint32_t* __restrict__ cells) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int4 c = reinterpret_cast<const int4*>(coords)[i];
    if (in_grid(g, c.x, c.y, c.z, c.w)) atomicMin(&cells[grid_cell(g, c.x, c.y, c.z, c.w)], (uint32_t)i);
}

// words[word] |= set for every lane (set == 0: nothing).  Lanes next to each other that name the same word -- voxels in scan order
// do, dozens at a time -- are merged first: atomics on one word are served one after the other.
__device__ __forceinline__ void or_word(uint32_t* __restrict__ words, size_t word, uint32_t set) {
    const int lane = threadIdx.x & 63;
    const uint32_t w = set ? (uint32_t)word : 0xFFFFFFFFu;         // (bit maps end below 2^32 words)
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t other = (uint32_t)__shfl_down((int)set, d, 64);
        const uint32_t ow = (uint32_t)__shfl_down((int)w, d, 64);
        if (lane + d < 64 && ow == w) set |= other;
    }
    const uint32_t before = (uint32_t)__shfl_up((int)w, 1, 64);
    if (set && (lane == 0 || before != w)) atomicOr(&words[word], set);
}

// steps_back (a word): how many of the sampled rows come before the row in front of them (every `every`-th workgroup looks)
__global__ void __launch_bounds__(256) set_bits_kernel(const int32_t* __restrict__ coords, size_t n, GridIndex g, uint32_t* __restrict__ words,
                                                       unsigned every, uint32_t* __restrict__ steps_back) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int4 c = i < n ? reinterpret_cast<const int4*>(coords)[i] : make_int4(-1, 0, 0, 0);
    const bool in = in_grid(g, c.x, c.y, c.z, c.w);
    const GridPlace<false> p = grid_place<false>(g, c.x, c.y, c.z, c.w);
    or_word(words, (size_t)p.brick * 4 + (p.at >> 5), in ? 1u << (p.at & 31u) : 0u);
    if (blockIdx.x % every == 0u) {
        const int lane = threadIdx.x & 63;
        const size_t cell = in ? grid_cell(g, c.x, c.y, c.z, c.w) : 0;
        const uint32_t lo = (uint32_t)__shfl_up((int)(uint32_t)cell, 1, 64), hi = (uint32_t)__shfl_up((int)(uint32_t)(cell >> 32), 1, 64);
        const unsigned long long back = __ballot(in && lane > 0 && cell < (((size_t)hi << 32) | lo));
        if (back != 0ull && lane == 0) atomicAdd(steps_back, (uint32_t)__popcll(back));
    }
}

__device__ __forceinline__ uint32_t state_load(const uint32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void state_store(uint32_t* p, uint32_t v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// Single-pass prefix sums with decoupled look-back (Merrill and Garland, 2016): sum of the tiles before `tile`, by one whole wavefront; the tile's own sum is made known to the tiles after it first, the
// running total last.  A word says what it holds (kLookbackSum / kLookbackTotal) in the bits above its value, so one relaxed
// load is enough.  Tiles are numbered in the order their workgroups started (a ticket), so every tile waited for is running.
__device__ __forceinline__ uint32_t lookback(uint32_t* state, unsigned tile, uint32_t sum) {
    const int lane = threadIdx.x & 63;
    if (tile == 0) {
        if (lane == 0) state_store(&state[0], kLookbackTotal | sum);
        return 0u;
    }
    if (lane == 0) state_store(&state[tile], kLookbackSum | sum);
    uint32_t before = 0u;
    int last = (int)tile - 1;                                       // 64 tiles at a time, nearest in lane 0
    while (true) {
        const int t = last - lane;
        uint32_t w = t >= 0 ? state_load(&state[t]) : kLookbackTotal;
        unsigned long long totals = __ballot((w & kLookbackTotal) != 0u);
        unsigned long long unknown = __ballot(w == 0u);
        const unsigned long long need = totals ? (totals & (~totals + 1ull)) * 2ull - 1ull : ~0ull;    // lanes up to the first total
        if (unknown & need) continue;                               // one of them is still counting
        uint32_t v = ((need >> lane) & 1ull) ? (w & kLookbackValue) : 0u;
#pragma unroll
        for (int d = 32; d > 0; d >>= 1) v += (uint32_t)__shfl_xor((int)v, d, 64);
        before += v;
        if (totals) break;
        last -= 64;
    }
    if (lane == 0) state_store(&state[tile], kLookbackTotal | (before + sum));
    return before;
}

// counts[block] = set bits before the block, in one pass over the bits.  state[tiles] is the ticket; total (optional): all
// set bits.  A wavefront counts 64 * ROWS consecutive blocks.
template <int ROWS, typename Total>
__global__ void __launch_bounds__(kCountThreads) count_bits_kernel(const ulonglong2* __restrict__ bits, size_t blocks, unsigned tiles,
                                                                   uint32_t* __restrict__ state, uint32_t* __restrict__ counts,
                                                                   Total* __restrict__ total) {
    constexpr int kWaves = kCountThreads / 64;
    __shared__ uint32_t wave_sum[kWaves];
    __shared__ uint32_t tile_lds, before_lds;
    if (threadIdx.x == 0) tile_lds = atomicAdd(&state[tiles], 1u);
    __syncthreads();
    const unsigned tile = tile_lds;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t base = (size_t)tile * (kCountThreads * ROWS) + (size_t)wave * (64 * ROWS) + lane;
    uint32_t c[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const size_t i = base + (size_t)r * 64;
        const ulonglong2 w = i < blocks ? bits[i] : make_ulonglong2(0ull, 0ull);
        c[r] = (uint32_t)(__popcll(w.x) + __popcll(w.y));
    }
    uint32_t run = 0u;
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        uint32_t incl = c[r];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = (uint32_t)__shfl_up((int)incl, d, 64);
            if (lane >= d) incl += o;
        }
        const uint32_t all = (uint32_t)__shfl((int)incl, 63, 64);
        c[r] = run + incl - c[r];
        run += all;
    }
    if (lane == 0) wave_sum[wave] = run;
    __syncthreads();
    if (wave == 0) {
        uint32_t sum = 0u;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) sum += wave_sum[w];
        const uint32_t before = lookback(state, tile, sum);
        if (lane == 0) {
            before_lds = before;
            if (tile == tiles - 1 && total != nullptr) *total = (Total)(before + sum);
        }
    }
    __syncthreads();
    uint32_t first = before_lds;
    for (int w = 0; w < wave; ++w) first += wave_sum[w];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) {
        const size_t i = base + (size_t)r * 64;
        if (i < blocks) counts[i] = first + c[r];
    }
}

// rows[rank of the voxel's cell] = the smallest row of that cell.  losers (optional): the rows that lose (and those outside the grid)
// from the end, in no fixed order
__global__ void __launch_bounds__(256) place_rows_kernel(const int32_t* __restrict__ coords, size_t n, GridIndex g, uint32_t* __restrict__ rows,
                                                         uint32_t* __restrict__ losers) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int4 c = reinterpret_cast<const int4*>(coords)[i];
    uint32_t loser = (uint32_t)i;
    if (in_grid(g, c.x, c.y, c.z, c.w)) {
        const GridPlace<false> p = grid_place<false>(g, c.x, c.y, c.z, c.w);
        const uint32_t rank = g.counts[p.brick] + bits_before(g.bits[p.brick], p.at);
        if ((size_t)g.order[0] == n) {           // as many cells as rows: nobody loses
            rows[rank] = (uint32_t)i;
            return;
        }
        const uint32_t had = atomicMin(&rows[rank], (uint32_t)i);
        loser = had == FGX_EMPTY32 ? FGX_EMPTY32 : (had > (uint32_t)i ? had : (uint32_t)i);
    }
    // every row but the cell's smallest loses exactly once, so these places and the ranks together are the n rows
    if (losers != nullptr && loser != FGX_EMPTY32) rows[n - 1 - atomicAdd(losers, 1u)] = loser;
}

// The rows that lost their cell (and those outside the grid) behind the others in row order: a walk that outlives the build is the
// chunks and the summation order of the narrow layers, and has to be a function of the coordinates.  One pass, tiles of rows by
// decoupled look-back; nobody loses in most builds, and then it is a launch that returns at once.
constexpr int kLoserThreads = 512, kLoserRows = 8;                  // rows per thread
__global__ void __launch_bounds__(kLoserThreads) list_losers_kernel(const int32_t* __restrict__ coords, size_t n, GridIndex g, uint32_t* __restrict__ state,
                                                                    uint32_t* rows, uint32_t* __restrict__ plan_header) {
    if (plan_header != nullptr && blockIdx.x == 0 && threadIdx.x < kNarrowHeader / 4) plan_header[threadIdx.x] = 0u;
    if ((size_t)g.order[0] == n) return;
    __shared__ uint32_t wave_sum[kLoserThreads / 64];
    __shared__ uint32_t tile_lds, before_lds;
    if (threadIdx.x == 0) tile_lds = atomicAdd(&state[gridDim.x], 1u);
    __syncthreads();
    const unsigned tile = tile_lds;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const size_t base = ((size_t)tile * (kLoserThreads / 64) + wave) * (64 * kLoserRows) + lane;       // a wavefront's rows are consecutive
    unsigned long long loses[kLoserRows];
    uint32_t mine = 0u;
#pragma unroll
    for (int r = 0; r < kLoserRows; ++r) {
        const size_t i = base + (size_t)r * 64;
        const int4 c = i < n ? reinterpret_cast<const int4*>(coords)[i] : make_int4(-1, 0, 0, 0);
        const bool in = in_grid(g, c.x, c.y, c.z, c.w);
        const bool kept = in && grid_find<false>(g, grid_place<false>(g, c.x, c.y, c.z, c.w)) == (uint32_t)i;
        loses[r] = __ballot(i < n && !kept);
        mine += (uint32_t)__popcll(loses[r]);
    }
    if (lane == 0) wave_sum[wave] = mine;
    __syncthreads();
    if (wave == 0) {
        uint32_t sum = 0u;
#pragma unroll
        for (int w = 0; w < kLoserThreads / 64; ++w) sum += wave_sum[w];
        const uint32_t before = lookback(state, tile, sum);
        if (lane == 0) before_lds = before;
    }
    __syncthreads();
    size_t at = (size_t)g.order[0] + before_lds;
    for (int w = 0; w < wave; ++w) at += wave_sum[w];
#pragma unroll
    for (int r = 0; r < kLoserRows; ++r) {
        if ((loses[r] >> lane) & 1ull) rows[at + (size_t)__popcll(loses[r] & ((1ull << lane) - 1ull))] = (uint32_t)(base + (size_t)r * 64);
        at += (size_t)__popcll(loses[r]);
    }
}

enum { kSubm = 0, kConvFwd = 1, kConvBwd = 2 };

struct QueryGeom {
    int Kw, Kh, Kd, V;
    int Sw, Sh, Sd;
    int Pw, Ph, Pd;
    int Dw, Dh, Dd;
};

__device__ __forceinline__ uint32_t gray_decode(uint32_t g) {
    g ^= g >> 16;
    g ^= g >> 8;
    g ^= g >> 4;
    g ^= g >> 2;
    g ^= g >> 1;
    return g;
}

// coordinate along one axis of the cell that kernel position k of a query at c asks for; false: there is none
template <int MODE>
__device__ __forceinline__ bool target(int c, int k, int K, int S, int P, int Dil, int extent, int* out) {
    int t;
    bool ok = true;
    if constexpr (MODE == kSubm) {
        t = c + (k - K / 2) * Dil;
    } else if constexpr (MODE == kConvFwd) {
        t = c * S - P + k * Dil;
    } else {                                    // the output whose position k reads the input at c
        const int num = c + P - k * Dil;
        if (S == 1) {                           // (uniform: no division where there is none to make)
            t = num;
        } else if (S == 2) {
            t = num >> 1;
            ok = (num & 1) == 0;
        } else {
            t = num / S;
            ok = num == t * S;
        }
    }
    *out = t;
    return ok && (unsigned)t < (unsigned)extent;
}

// map[row][v] for kRowsPerGroup rows (`walk`: an index of the queries whose row order makes neighbors ask for neighboring cells;
// without rows, or where the voxels come in scan order anyway and their map rows then lie side by side: as they come).  A wavefront asks the questions of one kernel column (kx, ky) for all of them, KD along z (0: g.Kd).  `own` (kConvBwd):
// the index of the queries themselves -- a row that is not the one its cell is known by gets an empty map row.  counts
// (rows as they come only): set mask bits per offset of every group, [V][gridDim.x].
template <bool DENSE, int MODE, int KD>
__global__ void map_kernel(const int32_t* __restrict__ coords, GridIndex walk, size_t n, GridIndex index, GridIndex own,
                           int own_dense, QueryGeom g, uint32_t* __restrict__ out_map, int32_t* __restrict__ gray, int32_t* __restrict__ binary,
                           uint32_t* __restrict__ counts) {
    extern __shared__ uint32_t lds[];
    const int V = g.V;
    const int pitch = V | 1;                                        // odd: the lanes of a wavefront write one column without conflicts
    int4* c_lds = (int4*)lds;                                       // [64]
    uint32_t* id_lds = lds + 4 * kRowsPerGroup;                     // [64] row number, EMPTY past the end
    uint32_t* mask_lds = id_lds + kRowsPerGroup;                    // [64]
    uint32_t* stage = mask_lds + kRowsPerGroup;                     // [64][pitch]
    const size_t p0 = (size_t)blockIdx.x * kRowsPerGroup;
    const int cnt = (int)(n - p0 < (size_t)kRowsPerGroup ? n - p0 : (size_t)kRowsPerGroup);
    const int tid = threadIdx.x, nt = blockDim.x;
    if (tid < kRowsPerGroup) {
        uint32_t id = FGX_EMPTY32;
        int4 c = make_int4(-1, 0, 0, 0);
        if (tid < cnt) {
            id = walk.rows != nullptr && !grid_in_scan_order(walk, n) ? walk.rows[p0 + tid] : (uint32_t)(p0 + tid);
            c = reinterpret_cast<const int4*>(coords)[id];
            if constexpr (MODE == kConvBwd) {
                bool known = in_grid(own, c.x, c.y, c.z, c.w);
                if (known)
                    known = (own_dense ? grid_find<true>(own, grid_place<true>(own, c.x, c.y, c.z, c.w))
                                       : grid_find<false>(own, grid_place<false>(own, c.x, c.y, c.z, c.w))) == id;
                if (!known) c.x = -1;
            }
        }
        id_lds[tid] = id;
        c_lds[tid] = c;
        mask_lds[tid] = 0u;
    }
    __syncthreads();
    const int R = g.Kw * g.Kh, kd = KD ? KD : g.Kd;
    const int lane = tid & 63, waves = nt >> 6;
    const int4 c = c_lds[lane];
    const uint32_t id = id_lds[lane];
    const bool batch_ok = (unsigned)c.x < (unsigned)index.B;
    for (int r = __builtin_amdgcn_readfirstlane(tid >> 6); r < R; r += waves) {
        const int kx = r / g.Kh, ky = r - kx * g.Kh;
        int x, y;
        const bool x_ok = target<MODE>(c.y, kx, g.Kw, g.Sw, g.Pw, g.Dw, index.W, &x);
        const bool y_ok = target<MODE>(c.z, ky, g.Kh, g.Sh, g.Ph, g.Dh, index.H, &y);
        const bool column = batch_ok && x_ok && y_ok;
        const GridPlace<DENSE> at = place_bx<DENSE>(index, c.x, x) + place_y<DENSE>(index, y);
        uint32_t found = 0u;
        auto ask = [&](int kz) {
            int z;
            uint32_t value = FGX_EMPTY32;
            if (target<MODE>(c.w, kz, g.Kd, g.Sd, g.Pd, g.Dd, index.D, &z) && column) value = grid_find<DENSE>(index, at + place_z<DENSE>(index, z));
            if (MODE == kSubm && r * kd + kz == V / 2) value = id;       // the middle entry is the voxel itself, found or not
            return value;
        };
        if constexpr (KD != 0) {
            uint32_t value[KD];
#pragma unroll
            for (int kz = 0; kz < KD; ++kz) value[kz] = ask(kz);           // all loads of the column in flight together
#pragma unroll
            for (int kz = 0; kz < KD; ++kz) {
                stage[lane * pitch + r * KD + kz] = value[kz];
                if (value[kz] != FGX_EMPTY32) found |= 1u << kz;
            }
        } else {
            for (int kz = 0; kz < kd; ++kz) {
                const uint32_t value = ask(kz);
                stage[lane * pitch + r * kd + kz] = value;
                if (value != FGX_EMPTY32 && kz < 32) found |= 1u << kz;
            }
        }
        if (gray != nullptr && found) atomicOr(&mask_lds[lane], found << (r * kd));      // (codes are asked for V <= 32 alone)
    }
    __syncthreads();
    for (int i = tid; i < cnt * V; i += nt) {
        const int row = i / V, v = i - row * V;
        out_map[(size_t)id_lds[row] * V + v] = stage[row * pitch + v];
    }
    if (gray == nullptr) return;
    if (tid < cnt) {
        const uint32_t m = mask_lds[tid];
        gray[id_lds[tid]] = (int32_t)m;
        binary[id_lds[tid]] = (int32_t)gray_decode(m);
    }
    if (counts != nullptr) {
        const uint32_t m = lane < cnt ? mask_lds[lane] : 0u;
        for (int v = tid >> 6; v < V; v += waves) {
            const unsigned long long have = __ballot((m >> v) & 1u);
            if (lane == 0) counts[(size_t)v * gridDim.x + blockIdx.x] = (uint32_t)__popcll(have);
        }
    }
}

// Answers of K columns of K cells (`bits` form; zp ascends by at most 32 cells, z_first and z_last the bricks of the first and the last one inside the grid).
template <int K>
__device__ __forceinline__ void brick_columns(const GridIndex& index, const GridPlace<false>& xp, bool x_ok, const bool (&y_ok)[K], const GridPlace<false> (&yp)[K],
                                              const bool (&z_ok)[K], const GridPlace<false> (&zp)[K], uint32_t z_first, uint32_t z_last, uint32_t (&value)[K][K]) {
    // the column's cells ascend along z and span at most 32: they lie in the brick of the first one inside the grid or in
    // that of the last one
    ulonglong2 wa[K], wb[K];
    uint32_t na[K], nb[K];
#pragma unroll
    for (int ky = 0; ky < K; ++ky) {
        const bool column = x_ok && y_ok[ky];
        const uint32_t brick_a = column ? xp.brick + yp[ky].brick + z_first : 0u;
        wa[ky] = index.bits[brick_a];
        na[ky] = index.counts[brick_a];
        wb[ky] = make_ulonglong2(0ull, 0ull);
        nb[ky] = 0u;
        if (column && z_last != z_first) {
            wb[ky] = index.bits[xp.brick + yp[ky].brick + z_last];
            nb[ky] = index.counts[xp.brick + yp[ky].brick + z_last];
        }
    }
#pragma unroll
    for (int ky = 0; ky < K; ++ky) {
        uint32_t rank[K];
        bool have[K];
#pragma unroll
        for (int kz = 0; kz < K; ++kz) {
            const bool in_a = zp[kz].brick == z_first;
            const ulonglong2 w = make_ulonglong2(in_a ? wa[ky].x : wb[ky].x, in_a ? wa[ky].y : wb[ky].y);
            const uint32_t at = (xp.at + yp[ky].at + zp[kz].at) & 127u;
            have[kz] = x_ok && y_ok[ky] && z_ok[kz] && (((at & 64u ? w.y : w.x) >> (at & 63u)) & 1ull);
            rank[kz] = (in_a ? na[ky] : nb[ky]) + bits_before(w, at);
        }
#pragma unroll
        for (int kz = 0; kz < K; ++kz) value[ky][kz] = have[kz] ? index.rows[rank[kz]] : FGX_EMPTY32;
    }
}

// The same for K x K x K kernels, K = 2 or 3: K wavefronts for 64 rows, a row per lane and a plane of the kernel per wavefront, which asks its K columns
// (K * K questions) before it needs the first answer.  What bounds it is the latency of three dependent reads (row, bits, row number)
// against what a CU holds in flight: one column per wavefront, as above, took 0.261 ms for 2 667 120 voxels of a surface in scan order (3x3x3, map
// and codes, 331 MB read and written), all planes in one wavefront 0.136 (sort and merge: 0.331).  So against that: 434 000 voxels 25.0 -> 21.7 us, of which
// the map and its codes leave at 2.3 TB/s; 67 000 outputs under a stride of 2 12.7 -> 10.0; 3 758 voxels 5.6 -> 4.3; 667 763 voxels in random order
// 64 -> 59; from 2 million voxels on level in either order, in random order because the scattered 108-byte rows bound it (2.54 and 2.67 M voxels 249 and
// 250 us; a plain scatter: 0.26 ms for 2 667 120).  In the `bits` form a column's cells have to lie in two bricks: columns longer than 32 cells go to the general kernel.
template <bool DENSE, int MODE, int K>
__global__ void __launch_bounds__(64 * K) cube_map_kernel(const int32_t* __restrict__ coords, GridIndex walk, size_t n,
                                                      GridIndex index, GridIndex own, int own_dense, QueryGeom g, uint32_t* __restrict__ out_map,
                                                      int32_t* __restrict__ gray, int32_t* __restrict__ binary, uint32_t* __restrict__ counts) {
    constexpr int V = K * K * K, PITCH = V | 1;
    __shared__ __attribute__((aligned(16))) uint32_t stage[kRowsPerGroup * PITCH];
    __shared__ uint32_t id_lds[kRowsPerGroup], masks[K][kRowsPerGroup];
    const size_t p0 = (size_t)blockIdx.x * kRowsPerGroup;
    const int cnt = (int)(n - p0 < (size_t)kRowsPerGroup ? n - p0 : (size_t)kRowsPerGroup);
    const int tid = threadIdx.x, lane = tid & 63, kx = __builtin_amdgcn_readfirstlane(tid >> 6);
    uint32_t id = FGX_EMPTY32;
    int4 c = make_int4(-1, 0, 0, 0);
    if (lane < cnt) {
        id = walk.rows != nullptr && !grid_in_scan_order(walk, n) ? walk.rows[p0 + lane] : (uint32_t)(p0 + lane);
        c = reinterpret_cast<const int4*>(coords)[id];
        if constexpr (MODE == kConvBwd) {
            bool known = in_grid(own, c.x, c.y, c.z, c.w);
            if (known)
                known = (own_dense ? grid_find<true>(own, grid_place<true>(own, c.x, c.y, c.z, c.w))
                                   : grid_find<false>(own, grid_place<false>(own, c.x, c.y, c.z, c.w))) == id;
            if (!known) c.x = -1;
        }
    }
    if (kx == 0) id_lds[lane] = id;
    const bool batch_ok = (unsigned)c.x < (unsigned)index.B;
    bool y_ok[K], z_ok[K];
    GridPlace<DENSE> yp[K], zp[K];
    uint32_t z_first = 0u, z_last = 0u;         // (`bits` form: bricks of the first and the last cell along z inside the grid)
#pragma unroll
    for (int k = 0; k < K; ++k) {
        int t;
        y_ok[k] = target<MODE>(c.z, k, K, g.Sh, g.Ph, g.Dh, index.H, &t);
        yp[k] = place_y<DENSE>(index, t);
        z_ok[k] = target<MODE>(c.w, k, K, g.Sd, g.Pd, g.Dd, index.D, &t);
        zp[k] = place_z<DENSE>(index, t);
        if constexpr (!DENSE) {
            if (z_ok[k]) z_last = zp[k].brick;
        }
    }
    if constexpr (!DENSE) {
        z_first = z_last;
#pragma unroll
        for (int k = K - 1; k >= 0; --k)
            if (z_ok[k]) z_first = zp[k].brick;
    }
    uint32_t mask = 0u;
    int xt;
    const bool x_ok = target<MODE>(c.y, kx, K, g.Sw, g.Pw, g.Dw, index.W, &xt) && batch_ok;
    uint32_t value[K][K];
    const GridPlace<DENSE> xp = place_bx<DENSE>(index, c.x, xt);
    if constexpr (DENSE || MODE == kConvBwd) {
#pragma unroll
        for (int ky = 0; ky < K; ++ky)
#pragma unroll
            for (int kz = 0; kz < K; ++kz)
                value[ky][kz] = x_ok && y_ok[ky] && z_ok[kz] ? grid_find<DENSE>(index, xp + yp[ky] + zp[kz]) : FGX_EMPTY32;
    } else {
        brick_columns<K>(index, xp, x_ok, y_ok, yp, z_ok, zp, z_first, z_last, value);
    }
#pragma unroll
    for (int ky = 0; ky < K; ++ky)
#pragma unroll
        for (int kz = 0; kz < K; ++kz) {
            const int v = (kx * K + ky) * K + kz;
            if (MODE == kSubm && v == V / 2) value[ky][kz] = id;       // the voxel itself, found or not
            stage[lane * PITCH + v] = value[ky][kz];
            if (value[ky][kz] != FGX_EMPTY32) mask |= 1u << (ky * K + kz);
        }
    masks[kx][lane] = mask;
    __syncthreads();
    const uint32_t id0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)id);
    if (PITCH == V && cnt == kRowsPerGroup && (id0 & 3u) == 0u && ((uintptr_t)out_map & 15) == 0 && __ballot(id != id0 + lane) == 0ull) {
        // the rows lie next to each other in the map as well: one run of 16-byte pieces
        uint4* dst = reinterpret_cast<uint4*>(out_map + (size_t)id0 * V);
        const uint4* src = reinterpret_cast<const uint4*>(stage);
        for (int i = tid; i < kRowsPerGroup * V / 4; i += 64 * K) dst[i] = src[i];
    } else {
        constexpr int kShare = (kRowsPerGroup + K - 1) / K;                // rows that a wavefront writes: a row leaves in one or two stores
        const int last = (kx + 1) * kShare < cnt ? (kx + 1) * kShare : cnt;
        for (int i = kx * kShare * V + lane; i < last * V; i += 64) {
            const int row = i / V, v = i - row * V;
            out_map[(size_t)id_lds[row] * V + v] = stage[row * PITCH + v];
        }
    }
    if (gray == nullptr) return;
    if (kx == 0 && lane < cnt) {
        uint32_t all = 0u;
#pragma unroll
        for (int k = 0; k < K; ++k) all |= masks[k][lane] << (k * K * K);
        gray[id] = (int32_t)all;
        binary[id] = (int32_t)gray_decode(all);
    }
    if (counts != nullptr) {
        uint32_t mine = 0u;
#pragma unroll
        for (int v = 0; v < K * K; ++v) {
            const uint32_t have = (uint32_t)__popcll(__ballot(lane < cnt && ((mask >> v) & 1u)));
            if (lane == v) mine = have;
        }
        if (lane < K * K) counts[(size_t)(kx * K * K + lane) * gridDim.x + blockIdx.x] = mine;
    }
}

// The map of a 3 x 3 x 3 submanifold convolution (`bits` form) and the plan of the narrow layers in one go: a workgroup finds the neighbors of 128 rows that
// follow each other in the walk -- a chunk of the plan --, three threads a row, and has them in LDS for both.  Reading the map's rows back in the
// walk's order is what the plan otherwise waits for.  Index, map and plan, one after the other -> so: 2 669 444 voxels in
// random order 765 -> 650 us (the two kernels 248 + 166 -> 330, bound by the scattered rows of the map), in scan order, which the cells' order scatters a little as
// well, 409 -> 398; 667 763 voxels 178 -> 138 and 108 -> 93; 166 977 voxels 52 -> 42.
constexpr int kPlanThreads = 3 * kNarrowRows;
__global__ void __launch_bounds__(kPlanThreads, 6) subm_map_plan_kernel(const int32_t* __restrict__ coords, GridIndex index, size_t n, QueryGeom g, uint32_t* __restrict__ out_map,
                                                                       int32_t* __restrict__ gray, int32_t* __restrict__ binary, unsigned char* __restrict__ plan) {
    constexpr int K = 3, V = 27;
    static_assert(V == kNarrowCubeV, "the plan's volume");
    __shared__ NarrowPlanLds lds;
    __shared__ uint32_t stage[kNarrowRows * V];
    __shared__ uint32_t masks[K][kNarrowRows];
    const int tid = threadIdx.x;
    const int kx = __builtin_amdgcn_readfirstlane(tid / kNarrowRows), row = tid % kNarrowRows;
    const size_t at = (size_t)blockIdx.x * kNarrowRows + row;
    const uint32_t id = at < n ? index.rows[at] : FGX_EMPTY32;
    const int4 c = at < n ? reinterpret_cast<const int4*>(coords)[id] : make_int4(-1, 0, 0, 0);
    if (kx == 0) lds.grow_of[row] = id;
    narrow_plan_clear<kPlanThreads>(lds, V);
    bool y_ok[K], z_ok[K];
    GridPlace<false> yp[K], zp[K];
    uint32_t z_first = 0u, z_last = 0u;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        int t;
        y_ok[k] = target<kSubm>(c.z, k, K, 1, 0, g.Dh, index.H, &t);
        yp[k] = place_y<false>(index, t);
        z_ok[k] = target<kSubm>(c.w, k, K, 1, 0, g.Dd, index.D, &t);
        zp[k] = place_z<false>(index, t);
        if (z_ok[k]) z_last = zp[k].brick;
    }
    z_first = z_last;
#pragma unroll
    for (int k = K - 1; k >= 0; --k)
        if (z_ok[k]) z_first = zp[k].brick;
    int xt;
    const bool x_ok = target<kSubm>(c.y, kx, K, 1, 0, g.Dw, index.W, &xt) && (unsigned)c.x < (unsigned)index.B;
    uint32_t value[K][K], mask = 0u;
    brick_columns<K>(index, place_bx<false>(index, c.x, xt), x_ok, y_ok, yp, z_ok, zp, z_first, z_last, value);
#pragma unroll
    for (int ky = 0; ky < K; ++ky)
#pragma unroll
        for (int kz = 0; kz < K; ++kz) {
            const int i = ky * K + kz;
            if (kx == 1 && i == 4) value[ky][kz] = id;               // the voxel itself, found or not
            stage[row * V + kx * (K * K) + i] = value[ky][kz];
            if (value[ky][kz] != FGX_EMPTY32) mask |= 1u << (kx * (K * K) + i);
        }
    masks[kx][row] = mask;
    __syncthreads();
    for (int i = tid; i < kNarrowRows * V; i += kPlanThreads) {
        const uint32_t to = lds.grow_of[i / V];
        if (to != FGX_EMPTY32) out_map[(size_t)to * V + i % V] = stage[i];
    }
    if (kx == 0 && id != FGX_EMPTY32) {
        const uint32_t all = masks[0][row] | masks[1][row] | masks[2][row];
        gray[id] = (int32_t)all;
        binary[id] = (int32_t)gray_decode(all);
    }
    narrow_plan_chunk<kPlanThreads, V>(lds, V, true, plan, blockIdx.x, [&](int e) -> uint32_t { return stage[e]; });
}

template <bool DENSE, int MODE>
int launch_map(const int32_t* coords, const GridIndex& walk, size_t n, const GridIndex& index, const GridIndex& own, bool own_dense,
               const QueryGeom& g, uint32_t* out_map, int32_t* gray, int32_t* binary, uint32_t* counts, hipStream_t s, const char* what) {
    const unsigned grid = cdiv(n, kRowsPerGroup);
    const int R = g.Kw * g.Kh;
    const bool cube = g.Kw == g.Kh && g.Kh == g.Kd && (DENSE || MODE == kConvBwd || g.Dd * (g.Kd - 1) <= 32);
    if (cube && g.Kd == 3) {
        cube_map_kernel<DENSE, MODE, 3><<<grid, 64 * 3, 0, s>>>(coords, walk, n, index, own, own_dense ? 1 : 0, g, out_map, gray, binary, counts);
    } else if (MODE != kSubm && cube && g.Kd == 2) {
        cube_map_kernel<DENSE, MODE, 2><<<grid, 64 * 2, 0, s>>>(coords, walk, n, index, own, own_dense ? 1 : 0, g, out_map, gray, binary, counts);
    } else {
        const int waves = R < 9 ? R : (R % 9 == 0 ? 9 : 8);         // a wavefront per kernel column
        const size_t lds = (size_t)kRowsPerGroup * (4 + 1 + 1 + (g.V | 1)) * 4;
        if (g.Kd == 3) map_kernel<DENSE, MODE, 3><<<grid, 64 * waves, lds, s>>>(coords, walk, n, index, own, own_dense ? 1 : 0, g, out_map, gray, binary, counts);
        else map_kernel<DENSE, MODE, 0><<<grid, 64 * waves, lds, s>>>(coords, walk, n, index, own, own_dense ? 1 : 0, g, out_map, gray, binary, counts);
    }
    FGX_CHECK_LAUNCH(what);
    return FGX_OK;
}

// ---- output coordinates ----
// K = 3: kernels of up to three cells along each axis.  A voxel's few outputs along an axis are listed first, so that a round of exchanging words takes a
// column of outputs from every lane -- under a stride of 2 one or two per axis where the kernel has two or three positions --, not one from the
// lanes of the right parity: 229 050 voxels, 3 x 3 x 3 13.9 -> 7.7 us; 255 000 voxels, 2 x 2 x 2 7.0 -> 4.9 (the divisions by the stride,
// five a column, were most of it).  K = 0: any kernel, position by position.
template <int K>
__global__ void __launch_bounds__(256) set_output_bits_kernel(const int32_t* __restrict__ coords, size_t n, int B, QueryGeom g, GridIndex out,
                                                              uint32_t* __restrict__ words) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int4 c = i < n ? reinterpret_cast<const int4*>(coords)[i] : make_int4(-1, 0, 0, 0);
    const bool batch_ok = (unsigned)c.x < (unsigned)B;
    if constexpr (K != 0) {
        int xs[K], ys[K], zs[K];
        auto list = [](int (&to)[K], int c, int taps, int S, int P, int Dil, int extent) {
            int many = 0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                int t;
                if (k >= taps || !target<kConvBwd>(c, k, taps, S, P, Dil, extent, &t)) continue;
#pragma unroll
                for (int i = 0; i < K; ++i) to[i] = many == i ? t : to[i];
                ++many;
            }
            return many;
        };
#pragma unroll
        for (int i = 0; i < K; ++i) xs[i] = ys[i] = zs[i] = 0;
        const int nx = batch_ok ? list(xs, c.y, g.Kw, g.Sw, g.Pw, g.Dw, out.W) : 0;
        const int ny = list(ys, c.z, g.Kh, g.Sh, g.Ph, g.Dh, out.H), nz = list(zs, c.w, g.Kd, g.Sd, g.Pd, g.Dd, out.D);
#pragma unroll
        for (int ix = 0; ix < K; ++ix)
#pragma unroll
            for (int iy = 0; iy < K; ++iy) {
                const bool column = ix < nx && iy < ny && nz > 0;
                if (__ballot(column) == 0ull) continue;             // (the whole wavefront: or_word exchanges words between lanes)
                const size_t cell0 = column ? grid_cell(out, c.x, xs[ix], ys[iy], 0) : 0;
                size_t word = 0;
                uint32_t set = 0u;
#pragma unroll
                for (int iz = 0; iz < K; ++iz) {
                    if (iz >= nz || !column) continue;
                    const size_t cell = cell0 + (size_t)zs[iz];
                    if (set != 0u && cell >> 5 != word) {           // the run along z leaves its first word
                        atomicOr(&words[word], set);
                        set = 0u;
                    }
                    word = cell >> 5;
                    set |= 1u << (cell & 31u);
                }
                or_word(words, word, set);
            }
        return;
    }
    for (int kx = 0; kx < g.Kw; ++kx)
        for (int ky = 0; ky < g.Kh; ++ky) {
            int x, y, z;
            const bool x_ok = target<kConvBwd>(c.y, kx, g.Kw, g.Sw, g.Pw, g.Dw, out.W, &x);
            const bool y_ok = target<kConvBwd>(c.z, ky, g.Kh, g.Sh, g.Ph, g.Dh, out.H, &y);
            const bool column = batch_ok && x_ok && y_ok;
            if (__ballot(column) == 0ull) continue;                 // (the whole wavefront: or_word exchanges words between lanes)
            const size_t cell0 = column ? grid_cell(out, c.x, x, y, 0) : 0;
            size_t word = 0;
            uint32_t set = 0u;
            for (int kz = 0; kz < g.Kd; ++kz) {
                if (!target<kConvBwd>(c.w, kz, g.Kd, g.Sd, g.Pd, g.Dd, out.D, &z) || !column) continue;
                const size_t cell = cell0 + (size_t)z;
                if (set != 0u && cell >> 5 != word) {               // the run along z leaves its first word
                    atomicOr(&words[word], set);
                    set = 0u;
                }
                word = cell >> 5;
                set |= 1u << (cell & 31u);
            }
            or_word(words, word, set);
        }
}

// Coordinates of the set bits at their ranks: 32 cells a thread, the coordinates by division for the first one and by counting on for the
// others.  Bound by its chain of reads, divisions (a bit map has 2^32 cells at most) and bits: with 128 cells a thread and 64-bit divisions
// 151 x 151 x 151 cells took 10.0 us, so 5.4; 128 x 128 x 128 6.7 and 4.5.
static_assert(kBitsMaxBytes * 8 <= (size_t)1 << 32, "a cell's number has 32 bits");
__global__ void __launch_bounds__(256) emit_coords_kernel(const uint4* __restrict__ bits, const uint32_t* __restrict__ counts, size_t blocks,
                                                          int W, int H, int D, size_t count, int32_t* __restrict__ out_coords) {
    const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= blocks * 4) return;
    const uint4 w = bits[t / 4];
    const int quarter = (int)(t & 3);
    uint32_t word = quarter == 0 ? w.x : (quarter == 1 ? w.y : (quarter == 2 ? w.z : w.w));
    if (word == 0u) return;
    size_t rank = counts[t / 4];
    rank += (quarter > 0 ? __popc(w.x) : 0) + (quarter > 1 ? __popc(w.y) : 0) + (quarter > 2 ? __popc(w.z) : 0);
    uint32_t rest = (uint32_t)(t * 32);
    int z = (int)(rest % (uint32_t)D);
    rest /= (uint32_t)D;
    int y = (int)(rest % (uint32_t)H);
    rest /= (uint32_t)H;
    int x = (int)(rest % (uint32_t)W);
    int b = (int)(rest / (uint32_t)W);
    int passed = 0;                             // cells the coordinates above have moved on from the word's first
    while (word) {
        const int at = __ffs((int)word) - 1;
        word &= word - 1u;
        z += at - passed;
        passed = at;
        while (z >= D) {
            z -= D;
            if (++y == H) {
                y = 0;
                if (++x == W) {
                    x = 0;
                    ++b;
                }
            }
        }
        if (rank < count) reinterpret_cast<int4*>(out_coords)[rank] = make_int4(b, x, y, z);
        ++rank;
    }
}

int check_query(const char* who, int Kw, int Kh, int Kd) {
    FGX_CHECK_ARG(Kw > 0 && Kh > 0 && Kd > 0, "%s: kernel sizes must be positive, got (%d,%d,%d)", who, Kw, Kh, Kd);
    FGX_CHECK_ARG((long long)Kw * Kh * Kd <= kMaxStageV, "%s: kernel volumes up to %d, got (%d,%d,%d)", who, kMaxStageV, Kw, Kh, Kd);
    return FGX_OK;
}

int launch_clear(void* zero, size_t zero_bytes, uint32_t* fill, size_t fill_words, hipStream_t s, const char* what) {
    const size_t most = zero_bytes > fill_words * 4 ? zero_bytes : fill_words * 4;
    unsigned grid = cdiv(most / 16 + 1, 256);
    if (grid > 4096u) grid = 4096u;
    clear_kernel<<<grid, 256, 0, s>>>((uint4*)zero, zero_bytes / 16, (uint4*)fill, fill_words);
    FGX_CHECK_LAUNCH(what);
    return FGX_OK;
}

template <typename Total>
int launch_count(const char* ws, const GridIndexLayout& L, Total* total, hipStream_t s, const char* what) {
    const ulonglong2* bits = (const ulonglong2*)(ws + L.bits);
    uint32_t* state = (uint32_t*)(ws + L.state);
    uint32_t* counts = (uint32_t*)(ws + L.counts);
    const unsigned tiles = (unsigned)L.tiles;
    const int per = count_rows(L.blocks);
    if (per == kCountRowsLong) count_bits_kernel<kCountRowsLong><<<tiles, kCountThreads, 0, s>>>(bits, L.blocks, tiles, state, counts, total);
    else if (per == kCountRowsShort) count_bits_kernel<kCountRowsShort><<<tiles, kCountThreads, 0, s>>>(bits, L.blocks, tiles, state, counts, total);
    else count_bits_kernel<kCountRowsFew><<<tiles, kCountThreads, 0, s>>>(bits, L.blocks, tiles, state, counts, total);
    FGX_CHECK_LAUNCH(what);
    return FGX_OK;
}

// Bit map of a grid: in bricks and cubes of 2^shift bricks each way (the index), or cells in their order (`in_order`: the output
// coordinates, which leave in that order).  The cubes are the largest whose padding adds no more than a quarter to the bricks'.
bool bits_layout(size_t n_rows, int B, int W, int H, int D, bool in_order, GridIndexLayout* out) {
    GridIndexLayout L{};
    if (B < 1 || W < 1 || H < 1 || D < 1) return false;
    const double cells = (double)B * W * H * D;
    if (cells > 8.0 * (double)kBitsMaxBytes || n_rows >= ((size_t)1 << 30)) return false;
    L.cells = (size_t)B * W * H * D;
    L.blocks = (L.cells + 127) / 128;
    if (!in_order) {
        const double bricks = (double)B * cdiv(W, 2) * cdiv(H, 2) * cdiv(D, 32);
        for (L.shift = 3;; --L.shift) {
            const uint32_t e = 2u << L.shift;
            const double padded = (double)B * cdiv(W, e) * cdiv(H, e) * cdiv(D, 32) * (double)(1u << (2 * L.shift));
            if (L.shift > 0 && padded > 1.25 * bricks) continue;
            if (padded > (double)kBitsMaxBytes / 16.0) return false;
            L.blocks = (size_t)padded;
            break;
        }
    }
    L.tiles = cdiv(L.blocks, (size_t)kCountThreads * count_rows(L.blocks));
    size_t off = 0;
    L.bits = off;
    off = align_up(off + L.blocks * 16, 256);
    L.state = off;
    off = align_up(off + (L.tiles + 4) * 4, 256);       // the tiles' words, the ticket, the number of losers, GridIndex::order
    L.losers = off;
    off = align_up(off + ((size_t)cdiv(n_rows, kLoserThreads * kLoserRows) + 1) * 4, 256);          // ... and of the tiles of rows, their ticket
    L.zero_bytes = off;
    L.counts = off;
    off = align_up(off + L.blocks * 4, 256);
    L.rows = off;
    off = align_up(off + n_rows * 4, 256);
    L.total = off;
    *out = L;
    return true;
}

}  // namespace

bool grid_index_plan(size_t n, int B, int W, int H, int D, GridIndexLayout* out) {
    GridIndexLayout L{};
    if (!bits_layout(n, B, W, H, D, false, &L)) return false;
    if (L.cells <= kDenseMaxCells) {
        L = GridIndexLayout{true, L.cells, 0, 0, 0, 0, 0, 0, 0, align_up(L.cells * 4, 256), 0, 0};
    }
    *out = L;
    return true;
}

bool grid_index_pays(size_t n, int B, int W, int H, int D) {
    GridIndexLayout L;
    if (!grid_index_plan(n, B, W, H, D, &L)) return false;
    const size_t bytes = L.blocks * 16;
    return L.dense || bytes <= kBitsAlwaysMaxBytes || bytes <= n * kBitsBytesPerVoxel;
}

int grid_index_build(const int32_t* coords, size_t n, int B, int W, int H, int D, const GridIndexLayout& L, void* workspace, uint32_t* walk,
                     uint32_t* plan_header, GridIndex* out, hipStream_t s, const char* what) {
    char* ws = (char*)workspace;
    GridIndex g{};
    g.B = B;
    g.W = W;
    g.H = H;
    g.D = D;
    const unsigned grid = cdiv(n, 256);
    if (L.dense) {
        uint32_t* cells = (uint32_t*)ws;
        int rc = launch_clear(nullptr, 0, cells, L.cells, s, what);
        if (rc != FGX_OK) return rc;
        g.cells = cells;
        if (n) insert_cells_kernel<<<grid, 256, 0, s>>>(coords, n, g, cells);
        FGX_CHECK_LAUNCH(what);
    } else {
        const uint32_t e = 2u << L.shift;
        g.shift = L.shift;
        g.step_y = (1u << (2 * L.shift)) * cdiv(D, 32);
        g.step_x = g.step_y * cdiv(H, e);
        g.step_b = g.step_x * cdiv(W, e);
        uint32_t* rows = walk != nullptr ? walk : (uint32_t*)(ws + L.rows);
        int rc = launch_clear(ws, L.zero_bytes, rows, n, s, what);
        if (rc != FGX_OK) return rc;
        uint32_t* order = (uint32_t*)(ws + L.state) + L.tiles + 2;
        g.order = order;
        if (n) set_bits_kernel<<<grid, 256, 0, s>>>(coords, n, g, (uint32_t*)(ws + L.bits), cdiv(grid, kOrderSamples), order + 1);
        FGX_CHECK_LAUNCH(what);
        rc = launch_count<uint32_t>(ws, L, order, s, what);
        if (rc != FGX_OK) return rc;
        g.bits = (const ulonglong2*)(ws + L.bits);
        g.counts = (const uint32_t*)(ws + L.counts);
        g.rows = rows;
        if (n) place_rows_kernel<<<grid, 256, 0, s>>>(coords, n, g, rows, walk != nullptr ? nullptr : (uint32_t*)(ws + L.state) + L.tiles + 1);
        FGX_CHECK_LAUNCH(what);
        if (n && walk != nullptr) {
            list_losers_kernel<<<cdiv(n, kLoserThreads * kLoserRows), kLoserThreads, 0, s>>>(coords, n, g, (uint32_t*)(ws + L.losers), rows,
                                                                                                              plan_header);
            FGX_CHECK_LAUNCH(what);
        }
    }
    *out = g;
    return FGX_OK;
}

int subm_map_grid(const int32_t* coords, size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dw, int Dh, int Dd,
                  const GridIndexLayout& L, void* workspace, uint32_t* walk, void* plan, uint32_t* out_map, int32_t* gray, int32_t* binary, uint32_t* counts,
                  bool* counted, hipStream_t s) {
    GridIndex index;
    phase_mark("grid index", s);
    int rc = grid_index_build(coords, n, B, W, H, D, L, workspace, walk, (uint32_t*)plan, &index, s, "fgx_subm_neighbor_map_grid(index)");
    if (rc != FGX_OK) return rc;
    phase_mark("grid map", s);
    const QueryGeom g{Kw, Kh, Kd, Kw * Kh * Kd, 1, 1, 1, 0, 0, 0, Dw, Dh, Dd};
    if (counted) *counted = L.dense && counts != nullptr;
    if (L.dense)
        return launch_map<true, kSubm>(coords, GridIndex{}, n, index, index, true, g, out_map, gray, binary, counts, s, "fgx_subm_neighbor_map_grid");
    if (plan != nullptr && n) {
        subm_map_plan_kernel<<<cdiv(n, kNarrowRows), kPlanThreads, 0, s>>>(coords, index, n, g, out_map, gray, binary, (unsigned char*)plan);
        FGX_CHECK_LAUNCH("fgx_subm_neighbor_map_grid(plan)");
        return FGX_OK;
    }
    return launch_map<false, kSubm>(coords, index, n, index, index, false, g, out_map, gray, binary, nullptr, s, "fgx_subm_neighbor_map_grid");
}

bool conv_maps_plan(size_t n_in, size_t n_out, int B, int W, int H, int D, int Wo, int Ho, int Do, bool with_bwd, ConvMapsLayout* P) {
    if (!grid_index_plan(n_in, B, W, H, D, &P->in)) return false;
    P->out_at = P->in.total;
    P->total = P->out_at;
    if (with_bwd) {
        if (!grid_index_plan(n_out, B, Wo, Ho, Do, &P->out)) return false;
        P->total += P->out.total;
    }
    return true;
}

int conv_maps_grid(const int32_t* in_coords, size_t n_in, const int32_t* out_coords, size_t n_out, int B, int W, int H, int D, int Wo, int Ho,
                   int Do, const int* k, const ConvMapsLayout& P, void* workspace, uint32_t* map_fwd, uint32_t* map_bwd, int32_t* gray,
                   int32_t* binary, uint32_t* counts, int32_t* gray_bwd, int32_t* binary_bwd, hipStream_t s) {
    const char* what = "fgx_spconv_neighbor_map_grid";
    char* ws = (char*)workspace;
    GridIndex in, out{};
    phase_mark("grid index", s);
    int rc = grid_index_build(in_coords, n_in, B, W, H, D, P.in, ws, nullptr, nullptr, &in, s, what);
    if (rc == FGX_OK && map_bwd != nullptr) rc = grid_index_build(out_coords, n_out, B, Wo, Ho, Do, P.out, ws + P.out_at, nullptr, nullptr, &out, s, what);
    if (rc != FGX_OK) return rc;
    phase_mark("grid map", s);
    const QueryGeom g{k[0], k[1], k[2], k[0] * k[1] * k[2], k[3], k[4], k[5], k[6], k[7], k[8], k[9], k[10], k[11]};
    if (n_out > 0)
        rc = P.in.dense ? launch_map<true, kConvFwd>(out_coords, GridIndex{}, n_out, in, in, true, g, map_fwd, gray, binary, counts, s, what)
                        : launch_map<false, kConvFwd>(out_coords, GridIndex{}, n_out, in, in, false, g, map_fwd, gray, binary, counts, s, what);
    if (rc != FGX_OK || map_bwd == nullptr || n_in == 0) return rc;
    const GridIndex walk = P.in.dense ? GridIndex{} : in;
    return P.out.dense ? launch_map<true, kConvBwd>(in_coords, walk, n_in, out, in, P.in.dense, g, map_bwd, gray_bwd, binary_bwd, nullptr, s, what)
                       : launch_map<false, kConvBwd>(in_coords, walk, n_in, out, in, P.in.dense, g, map_bwd, gray_bwd, binary_bwd, nullptr, s, what);
}

}  // namespace fgx

using namespace fgx;

extern "C" {

int fgx_grid_index_pays(size_t n, int B, int W, int H, int D) { return grid_index_pays(n, B, W, H, D) ? 1 : 0; }

int fgx_grid_index_walks(size_t n, int B, int W, int H, int D) {
    GridIndexLayout L;
    return grid_index_plan(n, B, W, H, D, &L) && !L.dense ? 1 : 0;
}

size_t fgx_subm_neighbor_map_grid_workspace_bytes(size_t n, int B, int W, int H, int D) {
    GridIndexLayout L;
    return grid_index_plan(n, B, W, H, D, &L) ? L.total : 0;
}

int fgx_subm_neighbor_map_grid(const int32_t* coords, size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dw, int Dh, int Dd,
                               void* workspace, size_t workspace_bytes, uint32_t* out_map, int32_t* gray, int32_t* binary, fgx_stream_t stream) {
    const char* who = "fgx_subm_neighbor_map_grid";
    int rc = check_query(who, Kw, Kh, Kd);
    if (rc != FGX_OK) return rc;
    FGX_CHECK_ARG((Kw & 1) && (Kh & 1) && (Kd & 1), "%s: kernel sizes must be odd, got (%d,%d,%d)", who, Kw, Kh, Kd);
    FGX_CHECK_ARG((gray == nullptr) == (binary == nullptr), "%s: gray and binary go together", who);
    FGX_CHECK_ARG(gray == nullptr || Kw * Kh * Kd <= 32, "%s: mask codes need a kernel volume <= 32, got (%d,%d,%d)", who, Kw, Kh, Kd);
    if (n == 0) return FGX_OK;
    GridIndexLayout L;
    FGX_CHECK_ARG(grid_index_plan(n, B, W, H, D, &L), "%s: no index over a grid of %d x %d x %d x %d cells and %zu voxels", who, B, W, H, D, n);
    FGX_CHECK_ARG(coords && workspace && out_map, "%s: null buffer", who);
    FGX_CHECK_ARG((((uintptr_t)coords & 15) | ((uintptr_t)workspace & 255)) == 0, "%s: coords must be 16-byte, workspace 256-byte aligned", who);
    FGX_CHECK_ARG(workspace_bytes >= L.total, "%s: workspace of %zu bytes, need %zu", who, workspace_bytes, L.total);
    PhaseEnd phases{(hipStream_t)stream};
    return subm_map_grid(coords, n, B, W, H, D, Kw, Kh, Kd, Dw, Dh, Dd, L, workspace, nullptr, nullptr, out_map, gray, binary, nullptr, nullptr, (hipStream_t)stream);
}

size_t fgx_spconv_neighbor_map_grid_workspace_bytes(size_t n_in, size_t n_out, int B, int W, int H, int D, int Wo, int Ho, int Do, int with_bwd) {
    ConvMapsLayout P;
    return conv_maps_plan(n_in, n_out, B, W, H, D, Wo, Ho, Do, with_bwd != 0, &P) ? P.total : 0;
}

int fgx_spconv_neighbor_map_grid(const int32_t* in_coords, size_t n_in, const int32_t* out_coords, size_t n_out, int B, int W, int H, int D,
                                 int Kw, int Kh, int Kd, int Sw, int Sh, int Sd, int Pw, int Ph, int Pd, int Dw, int Dh, int Dd,
                                 void* workspace, size_t workspace_bytes, uint32_t* map_fwd, uint32_t* map_bwd, int32_t* gray,
                                 int32_t* binary, fgx_stream_t stream) {
    const char* who = "fgx_spconv_neighbor_map_grid";
    int rc = check_query(who, Kw, Kh, Kd);
    if (rc != FGX_OK) return rc;
    FGX_CHECK_ARG((gray == nullptr) == (binary == nullptr), "%s: gray and binary go together", who);
    FGX_CHECK_ARG(gray == nullptr || Kw * Kh * Kd <= 32, "%s: mask codes need a kernel volume <= 32, got (%d,%d,%d)", who, Kw, Kh, Kd);
    int Wo, Ho, Do;
    rc = fgx_spconv_out_dims(W, H, D, Kw, Kh, Kd, Sw, Sh, Sd, Pw, Ph, Pd, Dw, Dh, Dd, &Wo, &Ho, &Do);
    if (rc != FGX_OK) return rc;
    FGX_CHECK_ARG(Sw > 0 && Sh > 0 && Sd > 0, "%s: strides must be positive", who);
    ConvMapsLayout P;
    FGX_CHECK_ARG(conv_maps_plan(n_in, n_out, B, W, H, D, Wo, Ho, Do, map_bwd != nullptr, &P), "%s: no index over a grid of this size", who);
    FGX_CHECK_ARG(workspace && (n_out == 0 || (out_coords && map_fwd)) && (n_in == 0 || in_coords), "%s: null buffer", who);
    FGX_CHECK_ARG((((uintptr_t)in_coords & 15) | ((uintptr_t)out_coords & 15) | ((uintptr_t)workspace & 255)) == 0,
                  "%s: coords must be 16-byte, workspace 256-byte aligned", who);
    FGX_CHECK_ARG(workspace_bytes >= P.total, "%s: workspace of %zu bytes, need %zu", who, workspace_bytes, P.total);
    const int k[12] = {Kw, Kh, Kd, Sw, Sh, Sd, Pw, Ph, Pd, Dw, Dh, Dd};
    PhaseEnd phases{(hipStream_t)stream};
    return conv_maps_grid(in_coords, n_in, out_coords, n_out, B, W, H, D, Wo, Ho, Do, k, P, workspace, map_fwd, map_bwd, gray, binary, nullptr,
                          nullptr, nullptr, (hipStream_t)stream);
}

size_t fgx_spconv_out_coords_grid_workspace_bytes(int B, int Wo, int Ho, int Do) {
    GridIndexLayout L;
    return bits_layout(0, B, Wo, Ho, Do, true, &L) ? L.total : 0;
}

int fgx_spconv_out_coords_grid_count(const int32_t* coords, size_t n_in, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Sw, int Sh,
                                     int Sd, int Pw, int Ph, int Pd, int Dw, int Dh, int Dd, void* workspace, size_t workspace_bytes,
                                     uint64_t* count, fgx_stream_t stream) {
    const char* who = "fgx_spconv_out_coords_grid_count";
    int Wo, Ho, Do;
    int rc = fgx_spconv_out_dims(W, H, D, Kw, Kh, Kd, Sw, Sh, Sd, Pw, Ph, Pd, Dw, Dh, Dd, &Wo, &Ho, &Do);
    if (rc != FGX_OK) return rc;
    GridIndexLayout L;
    FGX_CHECK_ARG(bits_layout(0, B, Wo, Ho, Do, true, &L), "%s: no bit map over an output grid of %d x %d x %d x %d cells", who, B, Wo, Ho, Do);
    FGX_CHECK_ARG(coords && n_in > 0 && workspace && count, "%s: null buffer", who);
    FGX_CHECK_ARG((double)n_in * Kw * Kh * Kd < (double)(1u << 30), "%s: too many candidates", who);
    FGX_CHECK_ARG((((uintptr_t)coords & 15) | ((uintptr_t)workspace & 255)) == 0, "%s: coords must be 16-byte, workspace 256-byte aligned", who);
    FGX_CHECK_ARG(workspace_bytes >= L.total, "%s: workspace of %zu bytes, need %zu", who, workspace_bytes, L.total);
    hipStream_t s = (hipStream_t)stream;
    char* ws = (char*)workspace;
    rc = launch_clear(ws, L.zero_bytes, nullptr, 0, s, who);
    if (rc != FGX_OK) return rc;
    GridIndex out{};
    out.B = B;
    out.W = Wo;
    out.H = Ho;
    out.D = Do;
    const QueryGeom g{Kw, Kh, Kd, Kw * Kh * Kd, Sw, Sh, Sd, Pw, Ph, Pd, Dw, Dh, Dd};
    if (Kw <= 3 && Kh <= 3 && Kd <= 3) set_output_bits_kernel<3><<<cdiv(n_in, 256), 256, 0, s>>>(coords, n_in, B, g, out, (uint32_t*)(ws + L.bits));
    else set_output_bits_kernel<0><<<cdiv(n_in, 256), 256, 0, s>>>(coords, n_in, B, g, out, (uint32_t*)(ws + L.bits));
    FGX_CHECK_LAUNCH(who);
    return launch_count(ws, L, count, s, who);
}

int fgx_spconv_out_coords_grid_emit(const void* workspace, int B, int Wo, int Ho, int Do, size_t count, int32_t* out_coords, fgx_stream_t stream) {
    const char* who = "fgx_spconv_out_coords_grid_emit";
    GridIndexLayout L;
    FGX_CHECK_ARG(bits_layout(0, B, Wo, Ho, Do, true, &L), "%s: no bit map over an output grid of %d x %d x %d x %d cells", who, B, Wo, Ho, Do);
    if (count == 0) return FGX_OK;
    FGX_CHECK_ARG(workspace && out_coords && ((uintptr_t)out_coords & 15) == 0, "%s: null or misaligned buffer", who);
    const char* ws = (const char*)workspace;
    emit_coords_kernel<<<cdiv(L.blocks * 4, 256), 256, 0, (hipStream_t)stream>>>((const uint4*)(ws + L.bits), (const uint32_t*)(ws + L.counts), L.blocks, Wo, Ho, Do, count,
                                                                   out_coords);
    FGX_CHECK_LAUNCH(who);
    return FGX_OK;
}

}  // extern "C"
