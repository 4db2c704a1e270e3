// The convolutions of a network's first layers (16-bit types, 8 or 16 channels on the gathered side, kernels of 17 ... 27 offsets):
// all offsets of a voxel side by side are one row of a matrix.  First the weight gradient:
//
//   grad_weight[co][v][ci] = sum over rows r with a neighbor at offset v of grad_out[r][co] * feats[map[r][v]][ci]
//
// As products per offset (wgrad_gemm.hip) every (row, offset) pair fetches a grad_out row of 2 * Co bytes for 16 or 32 bytes
// of features, and the 32-wide tile multiplies mostly padding.  Here the features of a row's V neighbors lie next to each other
// in LDS (a missing neighbor: zeros), [rows][V * Ci], and one product with the rows' own grad_out gives every offset at
// once: the features are gathered once per 64 or 128 of its columns, the pair lists not read at all.  What bounds it are the 16-byte gathers, one
// per (row, offset): 1 792 pieces for 64 rows, 0.88 us of a CU.  Four wavefronts do nothing but load and eight nothing but multiply: with both in one
// (issue a step's loads, then multiply another's) the address pipeline stood still while all of them multiplied, 1.4 us a step.  424 000 voxels
// 6 -> 48 channels 38 -> 29 us, 16 -> 48 67 -> 52.  A last piece per row holds a one: its column is the bias gradient.
// A workgroup keeps all accumulators over its contiguous run of rows and writes one partial product; a second kernel adds the
// partial products in workgroup order (same bits on every run).
#include "lane_swap.h"
#include "wgrad_device.h"

namespace fgx {
namespace {

__device__ __attribute__((aligned(256))) unsigned char g_zero_block_s[256];
// the piece (16 bytes) that starts with a one
__device__ __attribute__((aligned(256))) uint16_t g_one_f16[8] = {0x3C00, 0, 0, 0, 0, 0, 0, 0};
__device__ __attribute__((aligned(256))) uint16_t g_one_bf16[8] = {0x3F80, 0, 0, 0, 0, 0, 0, 0};

constexpr int kStemWaves = 8, kStemLoaders = 4;                // wavefronts that multiply, and that only load (one per SIMD)
constexpr int kStemThreads = 64 * (kStemWaves + kStemLoaders), kStemStages = 3;
constexpr int kStemMaxV = 27;

// P: 16-byte pieces of a feature row (Ci = 8 P)
// COLS: columns of grad_out that a workgroup of the weight gradient takes
template <int P, int COLS_ = 64>
struct StemCfg {
    static constexpr int COLS = COLS_, MT = COLS / 64;         // tiles of 32 of them per wavefront (2 share them)
    static constexpr int ROWS = 64 / P;                        // rows of a step
    static constexpr int PIECES = 28 * P;                      // of an LDS row: the offsets', the ones, padding
    static constexpr int N = PIECES * 8, NT = N / 32;          // columns of the product, in tiles of 32
    static constexpr int NT_PER = (NT + 3) / 4;                // ... per wavefront (4 share them, 2 the rows of the product)
    static constexpr int ROWB = PIECES * 16;
    static constexpr int F_BYTES = ROWS * ROWB, G_BYTES = ROWS * COLS * 2;
    static constexpr int F_INST = F_BYTES / 1024, G_INST = G_BYTES / 1024;
    static constexpr int F_PER = F_INST / kStemLoaders, G_PER = G_INST / kStemLoaders;     // loads per loader and step
    static constexpr int IDX_BYTES = ROWS * kStemMaxV * 4;
    static constexpr int IDX_SLOT = (IDX_BYTES + 1023) / 1024 * 1024;
    // A step's slot is written again IDX_SLOTS steps on.  The loaders' prologue reads the first steps' map words and asks for those of 2 (stages - 1)
    // steps in all: with one slot fewer (128 columns leave LDS for no more) the last ones go where the first step's were, which every loader
    // has to have read by then (PROLOGUE_BARRIER).  In the loop a barrier lies between the two either way.
    static constexpr int IDX_AHEAD = 2 * (kStemStages - 1), IDX_SLOTS = COLS == 64 ? IDX_AHEAD : IDX_AHEAD - 1;
    static constexpr bool PROLOGUE_BARRIER = IDX_SLOTS < IDX_AHEAD;
    static_assert(IDX_SLOTS >= IDX_AHEAD - 1, "the barrier stands before the prologue's last load of map words: only the first step's slot is free then");
    static constexpr int IDX_INST = IDX_SLOT / 1024, IDX_PER = (IDX_INST + kStemLoaders - 1) / kStemLoaders;
    static constexpr int STAGE = F_BYTES + G_BYTES;
    static constexpr size_t LDS = (size_t)kStemStages * STAGE + IDX_SLOTS * IDX_SLOT + 16;    // ... and the word that asks for a second pass
    static_assert(F_INST % kStemLoaders == 0 && G_INST % kStemLoaders == 0 && F_BYTES % 1024 == 0, "every loader has as many loads");
    static_assert(NT_PER % 2 == 0, "fragments are waited for in fours");
    static_assert(LDS <= 160 * 1024, "LDS");
    // XOR key on the 16-byte pieces of a grad_out row (8 or 16 of them): four rows of a transposing read on distinct banks.  Rows of
    // the feature side are 448 bytes (or 896) apart: 7 * 64 bytes put any four on distinct banks by themselves (two and two).
    static constexpr int key(int row) { return 2 * MT * (row & 3); }
};

// Map words of step j: ROWS * V of them in a row, 16 bytes per lane; past the map's end, and in the steps after the last one, zeros
// that nobody reads.
template <int P>
__device__ __forceinline__ void stem_issue_idx(const uint32_t* map, unsigned long long map_bytes, unsigned lo, int nsteps, int j, int V, int loader,
                                               int lane, unsigned char* slot, const unsigned char* zero_b) {
    using C = StemCfg<P>;
#pragma unroll
    for (int i = 0; i < C::IDX_PER; ++i) {
        const int inst = i * kStemLoaders + loader;            // wave-uniform
        if (inst >= C::IDX_INST) break;
        const int byte = inst * 1024 + lane * 16;
        const unsigned long long at = (unsigned long long)(lo + (unsigned)j) * (unsigned)(C::ROWS * V * 4) + (unsigned)byte;
        const bool real = j < nsteps && byte < C::ROWS * V * 4 && at + 16 <= map_bytes;
        const unsigned char* p = real ? (const unsigned char*)map + at : zero_b;
        __builtin_amdgcn_global_load_lds(FGX_GLOBAL_PTR(p), FGX_LDS_PTR(slot + inst * 1024), 16, 0, 0);
    }
}

// Where piece `at` of row `row` comes from in the last step, which has `rows` rows: map rows are read where they are (16 bytes of
// them may end past the map).
template <int P>
__device__ __forceinline__ const unsigned char* stem_piece(const unsigned char* feats, const uint32_t* map, const unsigned char* one_b,
                                                           const unsigned char* zero_b, unsigned long long base, int row, int rows, int at, int V) {
    const int v = at / P, part = at - v * P;
    if (row >= rows) return zero_b;
    if (v < V) {
        const uint32_t m = map[(base + (unsigned)row) * (unsigned)V + (unsigned)v];
        return m != FGX_EMPTY32 ? feats + (size_t)m * (16 * P) + part * 16 : zero_b;
    }
    return at == StemCfg<P>::PIECES - 1 ? one_b : zero_b;
}

// A loader's loads of a whole step's pieces: load i covers the 64 pieces from (i * loaders + loader) * 64 on.  Which map word names a lane's row, or
// which constant the piece is instead, is the same for every step; the words of all loads are read before the first address is needed.
template <int P>
struct StemPieces {
    static constexpr int N = StemCfg<P>::F_PER;
    uint32_t word[N];
    uint32_t offsets = 0, second = 0, ones = 0;                // bit i: load i's piece belongs to a kernel position; is the row's second one; is the ones'
    template <typename Key>
    __device__ __forceinline__ void init(int loader, int lane, int V, Key key) {
        using C = StemCfg<P>;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int piece = (i * kStemLoaders + loader) * 64 + lane, row = piece / C::PIECES, at = (piece - row * C::PIECES) ^ key(row), v = at / P;
            const bool offset = v < V;
            word[i] = offset ? (uint32_t)(row * V + v) : 0u;
            offsets |= (uint32_t)offset << i;
            second |= (uint32_t)(at - v * P) << i;
            ones |= (uint32_t)(at == C::PIECES - 1) << i;
        }
    }
    __device__ __forceinline__ void read(const uint32_t* words, uint32_t (&m)[N]) const {
#pragma unroll
        for (int i = 0; i < N; ++i) m[i] = words[word[i]];
    }
    __device__ __forceinline__ const unsigned char* source(int i, uint32_t m, const unsigned char* feats, const unsigned char* one_b,
                                                           const unsigned char* zero_b) const {
        const unsigned char* otherwise = (ones >> i) & 1u ? one_b : zero_b;
        return ((offsets >> i) & 1u) & (uint32_t)(m != FGX_EMPTY32) ? feats + (size_t)m * (16 * P) + (P == 2 ? ((second >> i) & 1u) * 16 : 0u) : otherwise;
    }
};

template <typename Tag, int P, int COLS>
__global__ void __launch_bounds__(kStemThreads)
stem_wgrad_kernel(const typename Tag::type* __restrict__ gout, const typename Tag::type* __restrict__ feats, const uint32_t* __restrict__ map,
                  uint32_t n, int V, int Co, unsigned steps_total, unsigned groups, float* __restrict__ partial) {
    using C = StemCfg<P, COLS>;
    using T = typename Tag::type;
    using T4 = T __attribute__((ext_vector_type(4)));
    constexpr int S = kStemStages;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    unsigned char* ring = lds;                                 // [S][features | grad_out]
    unsigned char* idx_ring = lds + S * C::STAGE;              // [IDX_SLOTS] map rows
    volatile uint32_t& again = *reinterpret_cast<volatile uint32_t*>(idx_ring + C::IDX_SLOTS * C::IDX_SLOT);       // some sum is not finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave & 1, wave_n = (wave >> 1) & 3;     // (of a multiplier)
    const int g = lane >> 5, l32 = lane & 31, s16 = lane & 15, mb = (lane >> 4) & 1;
    const int m0 = (int)blockIdx.y * COLS;

    // workgroups of one XCD take neighboring runs of steps
    const unsigned per_xcd = (groups + kXcds - 1) / kXcds;
    const unsigned group = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (group >= groups) return;
    const unsigned lo = (unsigned)((unsigned long long)steps_total * group / groups);
    const unsigned hi = (unsigned)((unsigned long long)steps_total * (group + 1) / groups);
    const int nsteps = (int)(hi - lo);

    const unsigned char* gout_b = (const unsigned char*)gout;
    const unsigned char* feats_b = (const unsigned char*)feats;
    const unsigned char* one_b = (const unsigned char*)(__is_same(typename Tag::type, _Float16) ? g_one_f16 : g_one_bf16);
    const unsigned char* zero_b = g_zero_block_s;
    const unsigned long long map_bytes = (unsigned long long)n * V * 4;

    // The loaders' walk over the steps; the multipliers meet them at its barriers.
    auto load_run = [&](const int lane) __attribute__((always_inline)) {
        const int lw = wave - kStemWaves;
        StemPieces<P> pieces;
        pieces.init(lw, lane, V, [](int) { return 0; });
        const int step_loads = C::F_PER + C::G_PER + (C::IDX_INST - lw + kStemLoaders - 1) / kStemLoaders;
        auto issue_idx = [&](int j) __attribute__((always_inline)) {
            stem_issue_idx<P>(map, map_bytes, lo, nsteps, j, V, lw, lane, idx_ring + ((unsigned)j % C::IDX_SLOTS) * C::IDX_SLOT, zero_b);
        };
        auto issue_rows_of = [&](int j, auto whole) __attribute__((always_inline)) {
            constexpr bool WHOLE = decltype(whole)::value;
            unsigned char* stage = ring + (j % S) * C::STAGE;
            const uint32_t* words = (const uint32_t*)(idx_ring + ((unsigned)j % C::IDX_SLOTS) * C::IDX_SLOT);
            const unsigned long long base = (unsigned long long)(lo + (unsigned)j) * C::ROWS;
            const int rows = WHOLE ? C::ROWS : (j < nsteps && base < n ? (int)(n - base) : 0);
            uint32_t named[C::F_PER];
            if (WHOLE) pieces.read(words, named);
#pragma unroll
            for (int i = 0; i < C::G_PER; ++i) {
                const int inst = i * kStemLoaders + lw, piece = inst * 64 + lane;
                const int row = piece / (COLS / 8), c = (piece % (COLS / 8) ^ C::key(row)) * 8;       // first column
                const unsigned char* p = zero_b;
                if ((WHOLE || row < rows) && m0 + c < Co) p = gout_b + ((base + (unsigned)row) * (unsigned)Co + (unsigned)(m0 + c)) * 2;
                __builtin_amdgcn_global_load_lds(FGX_GLOBAL_PTR(p), FGX_LDS_PTR(stage + C::F_BYTES + inst * 1024), 16, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < C::F_PER; ++i) {
                const int inst = i * kStemLoaders + lw;
                const unsigned char* p;
                if constexpr (WHOLE) {
                    p = pieces.source(i, named[i], feats_b, one_b, zero_b);
                } else {
                    const int piece = inst * 64 + lane, row = piece / C::PIECES;
                    p = stem_piece<P>(feats_b, map, one_b, zero_b, base, row, rows, piece - row * C::PIECES, V);
                }
                __builtin_amdgcn_global_load_lds(FGX_GLOBAL_PTR(p), FGX_LDS_PTR(stage + inst * 1024), 16, 0, 0);
            }
        };
        auto issue_rows = [&](int j) __attribute__((always_inline)) {
            if (j < nsteps && (unsigned long long)(lo + (unsigned)j + 1) * C::ROWS <= n) issue_rows_of(j, std::true_type{});
            else issue_rows_of(j, std::false_type{});
        };
#pragma unroll
        for (int j = 0; j < S - 1; ++j) issue_idx(j);
        wait_vmcnt<0>();
        __syncthreads();
#pragma unroll
        for (int j = 0; j < S - 1; ++j) {
            issue_rows(j);
            if (C::PROLOGUE_BARRIER && j == S - 2) {
                asm volatile("" ::: "memory");
                __builtin_amdgcn_s_barrier();                  // (the words were read: the loads that they name are on their way)
                asm volatile("" ::: "memory");
            }
            issue_idx(j + S - 1);
        }
        for (int k = 0; k < nsteps; ++k) {
            // rows of step k and the map words of step k + S - 1 have landed
            wait_vmcnt_in<(S - 2) * (C::F_PER + C::G_PER), (S - 2) * (C::F_PER + C::G_PER + C::IDX_PER)>((S - 2) * step_loads);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();                      // ... everybody's; the stage of step k - 1 is free
            asm volatile("" ::: "memory");
            issue_rows(k + S - 1);
            issue_idx(k + 2 * (S - 1));
        }
        wait_vmcnt<0>();                                       // the loads of the steps past the end
    };

    f32x16 acc[C::MT][C::NT_PER];
    // APART: rows of grad_out that are not finite are added pair by pair (wgrad_device.h).  428 946 voxels, with the reduction, us: 8 -> 48 channels
    // all finite 33, one value infinite 86, a value in every thousandth row 90, every value 930;  16 -> 48 53, 120, 128, 1 460 (the
    // sums that are not finite taken again over all rows, by the reduction, 8 -> 48: 8 200 and 8 800 for the last two).
    auto run = [&](auto apart_rows) __attribute__((always_inline)) {
        constexpr bool APART = decltype(apart_rows)::value;
#pragma unroll
        for (int i = 0; i < C::MT; ++i)
#pragma unroll
            for (int t = 0; t < C::NT_PER; ++t)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][t][e] = 0.f;

        __syncthreads();
        if (C::PROLOGUE_BARRIER) {                                 // (the loaders' among themselves)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        constexpr int NK = C::ROWS / 16;
        for (int k = 0; k < nsteps; ++k) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();                          // the loaders saw the rows of step k land
            asm volatile("" ::: "memory");
            const unsigned char* f_cur = ring + (k % S) * C::STAGE;
            const unsigned char* g_cur = f_cur + C::F_BYTES;
#pragma unroll
            for (int kk = 0; kk < NK; ++kk) {
                const int row = kk * 16 + g * 8 + (s16 >> 2);      // (see wgrad_gemm.hip on the transposing read)
                i16x4 fr[4 + 2 * C::NT_PER];                       // (of grad_out, two of them unused with 64 columns: waited for in fours)
#pragma unroll
                for (int i = 0; i < C::MT; ++i) {
                    const int byte = ((wave_m * C::MT + i) * 32 + mb * 16 + (s16 & 3) * 4) * 2;
                    const unsigned char* at = g_cur + row * (COLS * 2) + (((byte >> 4) ^ C::key(row)) << 4) + (byte & 15);
                    fr[2 * i] = lds_read_tr16(at);
                    fr[2 * i + 1] = lds_read_tr16(at + 4 * COLS * 2);
                }
                if (C::MT == 1) fr[2] = fr[3] = i16x4{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < C::NT_PER; ++t) {
                    const int tile = wave_n * C::NT_PER + t < C::NT ? wave_n * C::NT_PER + t : 0;
                    const unsigned char* at = f_cur + row * C::ROWB + (tile * 32 + mb * 16 + (s16 & 3) * 4) * 2;
                    fr[4 + 2 * t] = lds_read_tr16(at);
                    fr[5 + 2 * t] = lds_read_tr16(at + 4 * C::ROWB);
                }
                lds_wait_all(fr);
                i16x8 af[C::MT];
                uint32_t apart = 0u;
#pragma unroll
                for (int i = 0; i < C::MT; ++i) {
                    af[i] = __builtin_shufflevector(fr[2 * i], fr[2 * i + 1], 0, 1, 2, 3, 4, 5, 6, 7);
                    if constexpr (APART) apart |= nonfinite_rows<Tag>(af[i]);
                }
                if (APART && apart) {
#pragma unroll
                    for (int i = 0; i < C::MT; ++i) drop_rows(af[i], apart, g);
                }
#pragma unroll
                for (int t = 0; t < C::NT_PER; ++t) {
                    i16x8 bf = __builtin_shufflevector(fr[4 + 2 * t], fr[5 + 2 * t], 0, 1, 2, 3, 4, 5, 6, 7);
                    if (APART && apart) drop_rows(bf, apart, g);
#pragma unroll
                    for (int i = 0; i < C::MT; ++i) mma16<Tag>(acc[i][t], af[i], bf);
                }
                while (APART && apart) {
                    const int row = kk * 16 + __ffs((int)apart) - 1;
                    apart &= apart - 1u;
                    // (a row past the end is zeros and never comes here)
                    const uint32_t* neighbors = map + ((unsigned long long)(lo + (unsigned)k) * C::ROWS + (unsigned)row) * (unsigned)V;
#pragma unroll
                    for (int i = 0; i < C::MT; ++i) {
                        T4 gv[4];
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            gv[q] = *reinterpret_cast<const T4*>(g_cur + row * (COLS * 2) + ((((wave_m * C::MT + i) * 4 + q) ^ C::key(row)) << 4) + g * 8);
#pragma unroll
                        for (int t = 0; t < C::NT_PER; ++t) {
                            const int col = (wave_n * C::NT_PER + t) * 32 + l32, v = col / (8 * P);
                            if (col >= C::N || (v < V ? neighbors[v] == FGX_EMPTY32 : col < C::N - 8)) continue;
                            const float x = (float)*reinterpret_cast<const T*>(f_cur + row * C::ROWB + col * 2);
#pragma unroll
                            for (int e = 0; e < 16; ++e) acc[i][t][e] += (float)gv[e >> 2][e & 3] * x;
                        }
                    }
                }
            }
        }
    };
    if (tid == 0) again = 0u;                                      // (seen behind the first barrier of either side's run)
    if (wave >= kStemWaves) {
        __builtin_amdgcn_s_setprio(3);
        for (int pass = 0; pass < 2; ++pass) {
            int own = lane;                                        // (made anew: what follows from it is not kept in registers over both passes, and
            asm volatile("" : "+v"(own));                          // beside a multiplier's sums; 32 of them spilled, 16 -> 48, one value infinite: 235 us)
            load_run(own);
            if (pass == 0) __syncthreads();
            if (again == 0u) break;
        }
        return;
    }
    run(std::false_type{});
    bool finite = true;
#pragma unroll
    for (int i = 0; i < C::MT; ++i)
#pragma unroll
        for (int t = 0; t < C::NT_PER; ++t) finite = finite && all_finite(acc[i][t]);
    if (__any(!finite) && lane == 0) again = 1u;
    __syncthreads();                                               // (the loaders' after their first pass)
    if (again != 0u) run(std::true_type{});

    // partial[column tile][group][COLS][N]
    float* dst = partial + ((size_t)blockIdx.y * groups + group) * ((size_t)COLS * C::N);
#pragma unroll
    for (int i = 0; i < C::MT; ++i)
#pragma unroll
        for (int t = 0; t < C::NT_PER; ++t) {
            const int tile = wave_n * C::NT_PER + t;
            if (tile >= C::NT) continue;
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const int m = (wave_m * C::MT + i) * 32 + (e >> 2) * 8 + g * 4 + (e & 3);
                dst[(size_t)m * C::N + tile * 32 + l32] = acc[i][t][e];
            }
        }
}

// grad_weight and grad_bias: 32 columns of blockDim.z rows of the product per workgroup, blockDim.y threads per element each adding
// every blockDim.y-th partial product, their sums added in order.
template <typename T>
__global__ void __launch_bounds__(1024) stem_reduce_kernel(const float* __restrict__ partial, unsigned groups, int V, int Ci, int out_ci, int Co, int N, int tile,
                                                           T* __restrict__ gw, T* __restrict__ gb) {
    __shared__ float sums[32][33];                             // [rows * slices][32]
    const int c = threadIdx.x, slices = blockDim.y, slice = threadIdx.y, at = threadIdx.z * slices;
    const int col = blockIdx.x * 32 + c, co = blockIdx.y * blockDim.z + threadIdx.z;
    const size_t per = (size_t)tile * N;                       // (tile: columns of grad_out in a partial product)
    const float* src = partial + (size_t)(co / tile) * groups * per + (size_t)(co % tile) * N + col;
    float s = 0.f;
    unsigned b = co < Co ? slice : groups;
    for (; b + 3 * slices < groups; b += 4 * slices) {
        const float x0 = src[b * per], x1 = src[(b + slices) * per], x2 = src[(b + 2 * slices) * per], x3 = src[(b + 3 * slices) * per];
        s += x0; s += x1; s += x2; s += x3;
    }
    for (; b < groups; b += slices) s += src[b * per];
    sums[at + slice][c] = s;
    __syncthreads();
    float r = sums[at][c];
    for (int q = 1; q < slices; ++q) r += sums[at + q][c];
    if (slice != 0 || co >= Co) return;
    if (col < V * Ci) {
        const int v = col / Ci, ci = col - v * Ci;             // (the channels that filled the rows up are nobody's)
        if (ci < out_ci) gw[((size_t)co * V + v) * out_ci + ci] = from_float<T>(r);
    } else if (gb != nullptr && col == N - 8) {
        gb[co] = from_float<T>(r);
    }
}

// Forward product and input gradient of such layers (8 or 16 channels on the gathered side): the neighbors' features of a row lie
// side by side as in the weight gradient, and one product with the weight, [V * K] x [columns], replaces V products that fill
// a quarter (8 channels) or half of a K-slab.  The wavefronts keep the weight in registers over the workgroup's run of rows; the
// piece with the one multiplies the bias.  Rows are walked as they come, nothing of the mask sort is read.  Loaders and multipliers as in the
// weight gradient; a step is bound by what follows its barrier in a multiplier, 14 reads of LDS, 14 products in a row, rounding and two stores.
// 424 000 voxels, us: 6 -> 48 channels fp16 52 -> 35, bf16 64 -> 34; 16 -> 48 bf16 120 -> 62.
template <int P, bool WIDE>
struct StemGemmCfg {
    using W = StemCfg<P>;
    static constexpr int COLS = WIDE ? 256 : 128;              // output columns of a workgroup: tiles of 32, one per wavefront column
    static constexpr int RT = W::ROWS / 32;                    // row tiles of a step: each a multiplier's own, or (WIDE) one after the other
    static constexpr int WAVES = WIDE ? 8 : 4 * RT, THREADS = 64 * (WAVES + kStemLoaders);        // (one that loads: see kStemLoaders)
    static constexpr int KK = W::PIECES / 2;                   // products of a tile: 16 K values each
    static constexpr int AHEAD = 14;              // ... whose row fragments a wavefront has registers for beside the weight's
    static constexpr int STAGES = 4, IDX_SLOTS = 2 * (STAGES - 1);     // (a slot is written again once its step's rows are on their way)
    static constexpr size_t LDS = (size_t)STAGES * W::F_BYTES + IDX_SLOTS * W::IDX_SLOT;
    static_assert(LDS <= 160 * 1024, "LDS");
    // XOR key on the low bits of a row's piece numbers: 16 rows' reads of one piece fall on distinct banks (rows are 28 or 56 pieces)
    static __device__ __forceinline__ int key(int row) { return P == 1 ? (row >> 2) & 3 : (row >> 1) & 7; }
};

// mode as in fgx_pack_weight: 0 weight [cols][V][K], 1 / 2 weight [K][V][cols] with mirrored offsets / as they are
template <typename Tag, int P, bool WIDE>
__global__ void __launch_bounds__((StemGemmCfg<P, WIDE>::THREADS))
stem_gemm_kernel(const typename Tag::type* __restrict__ src, const typename Tag::type* __restrict__ weight,
                 const typename Tag::type* __restrict__ bias, const uint32_t* __restrict__ map, uint32_t n, int V, int cols, int mode,
                 unsigned steps_total, unsigned groups, int relu, typename Tag::type* __restrict__ out, uint8_t* __restrict__ relu_mask) {
    using C = StemCfg<P>;
    using G = StemGemmCfg<P, WIDE>;
    using T = typename Tag::type;
    constexpr int S = G::STAGES;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    unsigned char* ring = lds;                                 // [S][rows' features]
    unsigned char* idx_ring = lds + S * C::F_BYTES;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 5, l32 = lane & 31;
    const int ct = WIDE ? wave : wave & 3;                     // column tile of a multiplier
    const int c0 = (int)blockIdx.y * G::COLS + ct * 32;
    const bool multiplies = c0 < cols;

    const unsigned per_xcd = (groups + kXcds - 1) / kXcds;
    const unsigned group = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (group >= groups) return;
    const unsigned lo = (unsigned)((unsigned long long)steps_total * group / groups);
    const unsigned hi = (unsigned)((unsigned long long)steps_total * (group + 1) / groups);
    const int nsteps = (int)(hi - lo);

    const unsigned char* src_b = (const unsigned char*)src;
    const unsigned char* one_b = (const unsigned char*)(__is_same(T, _Float16) ? g_one_f16 : g_one_bf16);
    const unsigned char* zero_b = g_zero_block_s;
    const unsigned long long map_bytes = (unsigned long long)n * V * 4;

    if (wave >= G::WAVES) {
        __builtin_amdgcn_s_setprio(3);
        const int lw = wave - G::WAVES;
        StemPieces<P> pieces;
        pieces.init(lw, lane, V, [](int row) { return G::key(row); });
        const int step_loads = C::F_PER + (C::IDX_INST - lw + kStemLoaders - 1) / kStemLoaders;
        auto issue_idx = [&](int j) {
            stem_issue_idx<P>(map, map_bytes, lo, nsteps, j, V, lw, lane, idx_ring + (j % G::IDX_SLOTS) * C::IDX_SLOT, zero_b);
        };
        auto issue_rows_of = [&](int j, auto whole) {
            constexpr bool WHOLE = decltype(whole)::value;
            unsigned char* stage = ring + (j % S) * C::F_BYTES;
            const uint32_t* words = (const uint32_t*)(idx_ring + (j % G::IDX_SLOTS) * C::IDX_SLOT);
            const unsigned long long base = (unsigned long long)(lo + (unsigned)j) * C::ROWS;
            const int rows = WHOLE ? C::ROWS : (j < nsteps && base < n ? (int)(n - base) : 0);
            uint32_t named[C::F_PER];
            if (WHOLE) pieces.read(words, named);
#pragma unroll
            for (int i = 0; i < C::F_PER; ++i) {
                const int inst = i * kStemLoaders + lw;
                const unsigned char* p;
                if constexpr (WHOLE) {
                    p = pieces.source(i, named[i], src_b, one_b, zero_b);
                } else {
                    const int piece = inst * 64 + lane, row = piece / C::PIECES;
                    p = stem_piece<P>(src_b, map, one_b, zero_b, base, row, rows, (piece - row * C::PIECES) ^ G::key(row), V);
                }
                __builtin_amdgcn_global_load_lds(FGX_GLOBAL_PTR(p), FGX_LDS_PTR(stage + inst * 1024), 16, 0, 0);
            }
        };
        auto issue_rows = [&](int j) {
            if (j < nsteps && (unsigned long long)(lo + (unsigned)j + 1) * C::ROWS <= n) issue_rows_of(j, std::true_type{});
            else issue_rows_of(j, std::false_type{});
        };
#pragma unroll
        for (int j = 0; j < S - 1; ++j) issue_idx(j);
        wait_vmcnt<0>();
        __syncthreads();
#pragma unroll
        for (int j = 0; j < S - 1; ++j) {
            issue_rows(j);
            issue_idx(j + S - 1);
        }
        for (int k = 0; k < nsteps; ++k) {
            // rows of step k and the map words of step k + S - 1 have landed
            wait_vmcnt_in<(S - 2) * C::F_PER, (S - 2) * (C::F_PER + C::IDX_PER)>((S - 2) * step_loads);
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();                      // ... everybody's; the stage of step k - 1 is free
            asm volatile("" ::: "memory");
            issue_rows(k + S - 1);
            issue_idx(k + 2 * (S - 1));
        }
        wait_vmcnt<0>();
        return;
    }

    // The weight's fragments: lane l32 is a column, a piece its 8 consecutive K values.  Every load goes out before the first is waited for:
    // what a lane has no value for it reads from an address that exists and drops.
    i16x8 wf[G::KK];
    {
        const int col = c0 + l32, safe_col = col < cols ? col : 0;
        const short b0 = bias != nullptr ? ((const short*)bias)[safe_col] : (short)0;
#pragma unroll
        for (int kk = 0; kk < G::KK; ++kk) {
            const int at = kk * 2 + g, v = at / P, part = at - v * P, safe_v = v < V ? v : 0;
            if (mode == 0) {
                wf[kk] = *reinterpret_cast<const i16x8*>((const short*)weight + ((size_t)safe_col * V + safe_v) * (8 * P) + part * 8);
            } else {
                const int from = mode == 1 ? V - 1 - safe_v : safe_v;
#pragma unroll
                for (int e = 0; e < 8; ++e) wf[kk][e] = ((const short*)weight)[((size_t)(part * 8 + e) * V + from) * cols + safe_col];
            }
        }
#pragma unroll
        for (int kk = 0; kk < G::KK; ++kk) {
            const int at = kk * 2 + g, v = at / P;
            const bool live = multiplies && col < cols;
            if (!live || v >= V) wf[kk] = i16x8{0, 0, 0, 0, 0, 0, 0, 0};
            if (live && at == C::PIECES - 1) wf[kk][0] = b0;
        }
    }
    __syncthreads();
    for (int k = 0; k < nsteps; ++k) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();                          // the loaders saw the rows of step k land
        asm volatile("" ::: "memory");
        if (!multiplies) continue;
#pragma unroll
        for (int t = 0; t < (WIDE ? G::RT : 1); ++t) {
            const int rt = WIDE ? t : wave >> 2, frag_row = rt * 32 + l32;
            const unsigned char* row_at = ring + (k % S) * C::F_BYTES + frag_row * C::ROWB;
            f32x16 acc;
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[e] = 0.f;
#pragma unroll
            for (int k0 = 0; k0 < G::KK; k0 += G::AHEAD) {
                // (a group's reads all out before its first product: left to itself the compiler keeps two of them in flight)
                i16x8 rf[G::AHEAD];
#pragma unroll
                for (int kk = 0; kk < G::AHEAD; ++kk) rf[kk] = *reinterpret_cast<const i16x8*>(row_at + ((((k0 + kk) * 2 + g) ^ G::key(frag_row)) << 4));
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int kk = 0; kk < G::AHEAD; ++kk) mma16<Tag>(acc, wf[k0 + kk], rf[kk]);     // [column][row]: a lane ends up with columns of one row
            }
            // Element e of lane l: column 8 * (e / 4) + 4 * (l / 32) + e % 4, row l % 32.  Two exchanges between lanes make that 16-byte pieces, four
            // lanes a row: a store covers the 64 bytes of 16 rows.  (8 bytes a lane as they are: 16-byte writes at 110 G/s, 64 bytes each are a
            // quarter as many.)
            uint32_t w[4][2];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                using T4 = T __attribute__((ext_vector_type(4)));
                T4 four;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float x = acc[q * 4 + e];
                    four[e] = from_float<T>(relu ? __builtin_elementwise_maximum(x, 0.f) : x);
                }
                const uint64_t bits = __builtin_bit_cast(uint64_t, four);
                w[q][0] = (uint32_t)bits;
                w[q][1] = (uint32_t)(bits >> 32);
            }
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                swap_halves(w[0][d], w[1][d]);                     // lanes 0 - 31: pieces 0 and 2, lanes 32 - 63: 1 and 3
                swap_halves(w[2][d], w[3][d]);
            }
#pragma unroll
            for (int d = 0; d < 2; ++d) {
                swap_rows(w[0][d], w[2][d]);                       // rows 0 - 15 in the first piece, 16 - 31 in the second
                swap_rows(w[1][d], w[3][d]);
            }
            const int col = c0 + (((lane >> 4) & 1) * 2 + g) * 8;
            // (cols is a multiple of 8; all lanes stay for the next row tile)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                using T8 = T __attribute__((ext_vector_type(8)));
                const unsigned long long row = (unsigned long long)(lo + (unsigned)k) * C::ROWS + (unsigned)(rt * 32 + h * 16 + (lane & 15));
                if (row >= n || col >= cols) continue;
                const u32x4 piece = {w[2 * h][0], w[2 * h][1], w[2 * h + 1][0], w[2 * h + 1][1]};
                *reinterpret_cast<u32x4*>(out + row * (unsigned)cols + col) = piece;
                if (relu_mask != nullptr) {
                    const T8 x = __builtin_bit_cast(T8, piece);
                    uint32_t bits = 0;
#pragma unroll
                    for (int e = 0; e < 8; ++e) bits |= (uint32_t)((float)x[e] > 0.f) << e;
                    relu_mask[(row * (unsigned)cols + col) >> 3] = (uint8_t)bits;
                }
            }
        }
    }
}

// Columns of grad_out that a workgroup takes: 128 of 8 channels gather the rows half as often (with the forward pass, kept, 667 763 voxels, bf16: 8 -> 128 145 ->
// 137 us, 4 -> 136 301 -> 178, 6 -> 256 283 -> 250, 8 -> 384 695 -> 451); of 16 channels' product they would be 128 sums a lane.
int stem_cols(int Ci, int Co) { return Ci == 8 && Co > 64 ? 128 : 64; }

// Workgroups per column tile of grad_out: the chip full, and at least four steps each -- a partial product of 57 KB (Ci = 16: 115)
// is written and read for every one.
unsigned stem_groups(size_t n, int Ci, int Co) {
    const size_t runs = cdiv(n, 4 * (64 / (Ci / 8)));
    const unsigned col_tiles = cdiv(Co, stem_cols(Ci, Co));
    const size_t most = col_tiles >= 256 ? 1 : 256 / col_tiles;
    return (unsigned)(runs < most ? (runs ? runs : 1) : most);
}

template <typename Tag, int P, int COLS>
int stem_launch(const void* gout, const void* feats, const uint32_t* map, size_t n, int out_ci, int Co, int V, float* scratch, void* gw, void* gb,
                hipStream_t s) {
    using C = StemCfg<P, COLS>;
    using T = typename Tag::type;
    auto kern = stem_wgrad_kernel<Tag, P, COLS>;
    static thread_local bool lds_raised = false;
    if (!lds_raised) {
        FGX_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)C::LDS));
        lds_raised = true;
    }
    const unsigned groups = stem_groups(n, 8 * P, Co), col_tiles = cdiv(Co, COLS);
    const dim3 grid(cdiv(groups, kXcds) * kXcds, col_tiles);
    kern<<<grid, kStemThreads, C::LDS, s>>>((const T*)gout, (const T*)feats, map, (uint32_t)n, V, Co, cdiv(n, C::ROWS), groups, scratch);
    FGX_CHECK_LAUNCH("fgx_conv_wgrad_stem");
    unsigned slices = 1;
    while (slices < 32 && slices * 8 < groups) slices *= 2;
    const unsigned rows = slices >= 8 ? 1 : 8 / slices;
    stem_reduce_kernel<T><<<dim3(C::N / 32, cdiv(Co, rows)), dim3(32, slices, rows), 0, s>>>(scratch, groups, V, 8 * P, out_ci, Co, C::N, COLS, (T*)gw, (T*)gb);
    FGX_CHECK_LAUNCH("fgx_conv_wgrad_stem(reduce)");
    return FGX_OK;
}

template <typename Tag, int P, bool WIDE>
int stem_gemm_launch(int mode, const void* src, const void* weight, const void* bias, const uint32_t* map, size_t n, int cols, int V, int relu,
                     void* out, uint8_t* relu_mask, hipStream_t s) {
    using C = StemCfg<P>;
    using G = StemGemmCfg<P, WIDE>;
    using T = typename Tag::type;
    auto kern = stem_gemm_kernel<Tag, P, WIDE>;
    static thread_local bool lds_raised = false;
    if (!lds_raised) {
        FGX_CHECK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)G::LDS));
        lds_raised = true;
    }
    const unsigned steps = cdiv(n, C::ROWS), col_tiles = cdiv(cols, G::COLS);
    const unsigned most = col_tiles >= 256 ? 1 : 256 / col_tiles, groups = steps < most ? steps : most;
    const dim3 grid(cdiv(groups, kXcds) * kXcds, col_tiles);
    kern<<<grid, G::THREADS, G::LDS, s>>>((const T*)src, (const T*)weight, (const T*)bias, map, (uint32_t)n, V, cols, mode, steps, groups, relu,
                                            (T*)out, relu_mask);
    FGX_CHECK_LAUNCH("fgx_conv_gemm_stem");
    return FGX_OK;
}

bool stem_wgrad_takes(int dtype, size_t n, int Ci, int Co, int V) {
    return (dtype == FGX_F16 || dtype == FGX_BF16) && (Ci == 8 || Ci == 16) && Co > 0 && Co % 8 == 0 && Co <= 65535 && V >= 17 && V <= kStemMaxV &&
           n > 0 && n < 0xFFFFFFFFull;
}

bool stem_gemm_takes(int dtype, size_t n, int K, int cols, int V) {
    return (dtype == FGX_F16 || dtype == FGX_BF16) && (K == 8 || K == 16) && cols > 0 && cols % 8 == 0 && cols <= 65535 * 128 && V >= 17 &&
           V <= kStemMaxV && n > 0 && n < 0xFFFFFFFFull;
}

}  // namespace
}  // namespace fgx

using namespace fgx;

extern "C" {

// Weight gradient, ms: 424 000 voxels 6 (padded to 8) -> 48 channels 0.132 on the streaming kernel, 0.043 here; 143 616 voxels
// 8 -> 64 0.053 and 0.023, 16 -> 64 0.057 and 0.036; 848 voxels 8 -> 48 0.013 and 0.011.  With 16 channels and few voxels the partial
// products weigh as much as the pairs: level up to 64 columns, behind over more (15 192 voxels 16 -> 128 0.027 and 0.028).
int fgx_wgrad_stem_pays(int dtype, size_t n, int Ci, int Co, int V) {
    return stem_wgrad_takes(dtype, n, Ci, Co, V) && (Ci == 8 || Co <= 64 || n >= 24576);
}

size_t fgx_wgrad_stem_scratch_bytes(size_t n, int Ci, int Co) {
    if ((Ci != 8 && Ci != 16) || Co <= 0) return 0;
    return (size_t)stem_groups(n, Ci, Co) * align_up((size_t)Co, (size_t)stem_cols(Ci, Co)) * (size_t)(28 * Ci) * sizeof(float);
}

int fgx_conv_wgrad_stem(int dtype, const void* grad_out, const void* feats, const uint32_t* map, size_t n, int Ci, int Co, int V, void* scratch,
                        void* grad_weight, void* grad_bias, fgx_stream_t stream) {
    return fgx_conv_wgrad_stem_cut(dtype, grad_out, feats, map, n, Ci, Ci, Co, V, scratch, grad_weight, grad_bias, stream);
}

int fgx_conv_wgrad_stem_cut(int dtype, const void* grad_out, const void* feats, const uint32_t* map, size_t n, int Ci, int out_ci, int Co, int V,
                            void* scratch, void* grad_weight, void* grad_bias, fgx_stream_t stream) {
    FGX_CHECK_ARG(stem_wgrad_takes(dtype, n, Ci, Co, V), "fgx_conv_wgrad_stem: dtype %d, n=%zu, Ci=%d, Co=%d, V=%d is not for this kernel", dtype, n,
                  Ci, Co, V);
    FGX_CHECK_ARG(out_ci >= 1 && out_ci <= Ci, "fgx_conv_wgrad_stem: %d of %d channels", out_ci, Ci);
    FGX_CHECK_ARG(grad_out && feats && map && scratch && grad_weight, "fgx_conv_wgrad_stem: null buffer");
    FGX_CHECK_ARG((((uintptr_t)grad_out | (uintptr_t)feats | (uintptr_t)map | (uintptr_t)scratch) & 15) == 0,
                  "fgx_conv_wgrad_stem: grad_out, feats, map and scratch must be 16-byte aligned");
    hipStream_t s = (hipStream_t)stream;
#define FGX_STEM(Tag)                                                                                                                          \
    return Ci == 16                  ? stem_launch<Tag, 2, 64>(grad_out, feats, map, n, out_ci, Co, V, (float*)scratch, grad_weight, grad_bias, s)  \
           : stem_cols(Ci, Co) == 64 ? stem_launch<Tag, 1, 64>(grad_out, feats, map, n, out_ci, Co, V, (float*)scratch, grad_weight, grad_bias, s)  \
                                     : stem_launch<Tag, 1, 128>(grad_out, feats, map, n, out_ci, Co, V, (float*)scratch, grad_weight, grad_bias, s)
    if (dtype == FGX_F16) FGX_STEM(F16);
    FGX_STEM(BF16);
#undef FGX_STEM
}

// Where it is ahead of the general kernels (us, scan order, bf16: general, this):
//            forward                                                                       input gradient
//   rows     8 -> 16    8 -> 64   16 -> 16  16 -> 64  16 -> 256       rows     8 -> 16  16 -> 16  16 -> 32  16 -> 64  16 -> 96  16 -> 256
//       187  11.7  6.1  11.0  6.2  11.6  6.6  11.5  6.6  11.5  7.0        187  10.5  9.1  10.5 13.1           10.2 13.5            10.7 13.3
//     3 758  12.7  6.2  14.3  6.2  13.1  6.6  14.0  6.6  20.4  6.8      2 047  12.5  9.6  10.4 13.3           11.7 13.8  12.5 13.3 16.9 13.8
//    38 407  19.0  7.3  21.3  7.9  20.1  9.2  21.6  9.8  33.3 16.6      3 758  11.3  9.2  11.6 13.4           13.8 13.4  14.6 13.2 19.9 13.5
//   428 946  76.2 29.9  86.5 32.9  83.3 50.1  92.9 52.5   203  108     15 467  13.4  9.3  13.7 13.9 15.5 14.0 19.0 14.3  26.6 14.3 33.9 16.9
// 2 669 444   398  158   434  173   418  274   451  287  1130  694  2 669 444   389  164   416  288 417 291   428  304   571  320 1107  711
// An input gradient fetches its fragments of the weight one value at a time, 3 us more per launch under 8 channels and 6 under 16.
int fgx_conv_gemm_stem_pays(int dtype, int mode, size_t n, int K, int cols, int V) {
    if (mode < 0 || mode > 2 || !stem_gemm_takes(dtype, n, K, cols, V)) return 0;
    return mode == 0 || K == 8 || n >= 16384 || (n >= 3072 && cols >= 64);
}

int fgx_conv_gemm_stem(int dtype, int mode, const void* src, const void* weight, const void* bias, const uint32_t* map, size_t n, int Ci, int Co,
                       int V, int activation, void* out, uint8_t* relu_mask, fgx_stream_t stream) {
    FGX_CHECK_ARG(mode >= 0 && mode <= 2, "fgx_conv_gemm_stem: mode must be 0 (forward), 1 (dgrad, mirrored offsets) or 2 (dgrad)");
    const int K = mode == 0 ? Ci : Co, cols = mode == 0 ? Co : Ci;
    FGX_CHECK_ARG(stem_gemm_takes(dtype, n, K, cols, V), "fgx_conv_gemm_stem: dtype %d, n=%zu, K=%d, cols=%d, V=%d is not for this kernel", dtype, n, K,
                  cols, V);
    FGX_CHECK_ARG(activation == FGX_ACT_NONE || activation == FGX_ACT_RELU, "fgx_conv_gemm_stem: unknown activation %d", activation);
    FGX_CHECK_ARG(relu_mask == nullptr || activation == FGX_ACT_RELU, "fgx_conv_gemm_stem: a ReLU mask needs the ReLU epilogue");
    FGX_CHECK_ARG(src && weight && map && out, "fgx_conv_gemm_stem: null buffer");
    FGX_CHECK_ARG((((uintptr_t)src | (uintptr_t)weight | (uintptr_t)map | (uintptr_t)out) & 15) == 0,
                  "fgx_conv_gemm_stem: src, weight, map and out must be 16-byte aligned");
    const int relu = activation == FGX_ACT_RELU;
    hipStream_t s = (hipStream_t)stream;
    // 256 columns a workgroup from 129 on: the rows are gathered half as often (667 763 voxels, bf16: 8 -> 128 72 us, 4 -> 160 117 -> 91, 6 -> 256 149 -> 127,
    // 8 -> 320 287 -> 160, 8 -> 384 344 -> 181, 8 -> 560 520 -> 391).  16 channels' weight does not fit beside such a wavefront's fragments (16 -> 160 154, 419).
#define FGX_STEM(Tag)                                                                                                                    \
    return K == 16      ? stem_gemm_launch<Tag, 2, false>(mode, src, weight, bias, map, n, cols, V, relu, out, relu_mask, s)             \
           : cols > 128 ? stem_gemm_launch<Tag, 1, true>(mode, src, weight, bias, map, n, cols, V, relu, out, relu_mask, s)              \
                        : stem_gemm_launch<Tag, 1, false>(mode, src, weight, bias, map, n, cols, V, relu, out, relu_mask, s)
    if (dtype == FGX_F16) FGX_STEM(F16);
    FGX_STEM(BF16);
#undef FGX_STEM
}

}  // extern "C"
