// Gather GEMM of few voxels under wide weights, offset by offset over the pairs that exist (forward and dgrad, gfx950).
//
//   partial[p, :] = src[in(p), :] x W_v          for the pairs p = (r, v) of one offset v after the other
//   out[r, :]     = sum over v of partial[pair(r, v), :] (+ bias)
//
// The masked kernels multiply a tile of output rows with every offset that any of its rows has.  A few hundred or thousand voxels
// of a surface have nearly as many masks as voxels, so a tile carries almost all offsets and 2 to 2.5 rows are multiplied per
// pair (864 voxels of a thick shell: 0.42 of the rows of a 256-row tile have the offset; 3 758 voxels 0.51; 41 700 voxels 0.58).  Here the rows
// of a tile are 128 pairs of ONE offset: 0.89 and 0.96 of what is multiplied exists.  What that costs is the partial sums, 4 bytes
// per pair and output column written and read once, which the 256 MB memory-side cache holds for as many voxels as this
// pays for.  The product itself has no masks, bands or index stream left: a tile's source rows are known before its first step.
//
// fgx_pair_plan lists the pairs: per offset how many, their source rows in row order, and for each (row, offset) its place in the
// offset's list.  Nothing is read back: the launch covers the most tiles there can be, and a workgroup finds its tile -- or that
// there is none for it -- from the counts.
#include <type_traits>

#include "gemm_device.h"
#include "lds_read.h"

namespace fgx {
namespace {

constexpr int kPairRows = 128;                      // pairs of a tile
constexpr int kPairMaxV = 32;
constexpr uint32_t kOobOffset = 0xFF000000u;        // buffer offset no operand reaches: the load returns zeros

using rsrc_t = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}

constexpr int kPairChunk = 256;     // rows a workgroup of the plan places

// plan: counts[kPairMaxV] | place[n][V] | rows[V][n] | the chunks' counts [chunks][kPairMaxV] (while it is made)
__host__ __device__ inline size_t pair_place_at() { return kPairMaxV; }
__host__ __device__ inline size_t pair_rows_at(size_t n, int V) { return kPairMaxV + n * (size_t)V; }
__host__ __device__ inline size_t pair_chunks_at(size_t n, int V) { return kPairMaxV + 2 * n * (size_t)V; }

// Up to kPairColumnRows rows in one launch: a workgroup per offset, four words of its column in flight per thread, one barrier to hand
// the wavefronts' counts round.  It waits for the scattered words (a wave-wide load takes 64 lines): 864 rows 4.2 us, 3 758 rows 8.2.
constexpr int kPairColumnRows = 4096;
__global__ void __launch_bounds__(1024) pair_plan_columns_kernel(const uint32_t* __restrict__ map, uint32_t n, int V, uint32_t* __restrict__ plan) {
    __shared__ uint32_t counts[64];             // of (quarter of the rows, wavefront)
    const int v = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t m[4];
    unsigned long long have[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t r = q * 1024 + threadIdx.x;
        m[q] = r < n ? map[(size_t)r * V + v] : FGX_EMPTY32;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        have[q] = __ballot(m[q] != FGX_EMPTY32);
        if (lane == 0) counts[q * 16 + wave] = (uint32_t)__popcll(have[q]);
    }
    __syncthreads();
    const uint32_t mine = counts[lane];
    uint32_t to = mine;
#pragma unroll
    for (int d = 1; d < 64; d *= 2) {
        const uint32_t other = (uint32_t)__shfl_up((int)to, d, 64);
        if (lane >= d) to += other;
    }
    uint32_t* place = plan + pair_place_at();
    uint32_t* rows = plan + pair_rows_at(n, V) + (size_t)v * n;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const uint32_t r = q * 1024 + threadIdx.x;
        const uint32_t at = (uint32_t)__shfl((int)(to - mine), q * 16 + wave, 64) + (uint32_t)__popcll(have[q] & ((1ull << lane) - 1ull));
        if (r < n) place[(size_t)r * V + v] = m[q] != FGX_EMPTY32 ? at : FGX_EMPTY32;
        if (m[q] != FGX_EMPTY32) rows[at] = m[q];
    }
    if (threadIdx.x == 63) plan[v] = to;
}

// More rows: a workgroup takes kPairChunk of them through LDS, a thread a row, so the map comes in and the places go out as whole
// lines; a launch of its own counts the chunks first (COUNT).  38 407 rows 12.6 us (column by column in chunks of 4096: 22.6), 3 758 rows 10.9.
template <bool COUNT, int VC>
__global__ void __launch_bounds__(kPairChunk) pair_plan_kernel(const uint32_t* __restrict__ map, uint32_t n, int v_arg, uint32_t* __restrict__ plan) {
    constexpr int kWaves = kPairChunk / 64, VM = VC > 0 ? VC : kPairMaxV;
    extern __shared__ uint32_t words[];                         // [kPairChunk][V]
    __shared__ uint32_t counts[kPairMaxV][kWaves], before[kPairMaxV];
    const int V = VC > 0 ? VC : v_arg;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t* chunks = plan + pair_chunks_at(n, V);
    const uint32_t base = blockIdx.x * (uint32_t)kPairChunk, here = n - base < (uint32_t)kPairChunk ? n - base : (uint32_t)kPairChunk;
    const uint32_t* from = map + (size_t)base * V;
    {
        uint32_t w[VM];
#pragma unroll
        for (int i = 0; i < VM; ++i) w[i] = i < V && i * kPairChunk + tid < (int)here * V ? from[i * kPairChunk + tid] : FGX_EMPTY32;
#pragma unroll
        for (int i = 0; i < VM; ++i)
            if (i < V) words[i * kPairChunk + tid] = w[i];      // (rows past the end: no neighbors)
    }
    if constexpr (!COUNT) {                                     // pairs of the chunks before this one, 8 threads on each offset
        static_assert(kPairChunk == 8 * kPairMaxV, "a thread for every eighth of an offset's chunks");
        const int v = tid >> 3;
        uint32_t sum = 0;
        for (uint32_t c0 = 0; c0 < blockIdx.x; c0 += 64) {      // (eight loads in flight)
#pragma unroll
            for (uint32_t q = 0; q < 64; q += 8) {
                const uint32_t c = c0 + q + (uint32_t)(tid & 7);
                sum += v < V && c < blockIdx.x ? chunks[(size_t)c * kPairMaxV + v] : 0u;
            }
        }
#pragma unroll
        for (int d = 4; d > 0; d /= 2) sum += (uint32_t)__shfl_xor((int)sum, d, 64);
        if ((tid & 7) == 0) before[v] = sum;
    }
    __syncthreads();
    uint32_t m[VM];
#pragma unroll
    for (int v = 0; v < VM; ++v) m[v] = v < V ? words[tid * V + v] : FGX_EMPTY32;
    uint32_t have_mine = 0;
#pragma unroll
    for (int v = 0; v < VM; ++v) {
        const uint32_t c = (uint32_t)__popcll(__ballot(m[v] != FGX_EMPTY32));
        have_mine = lane == v ? c : have_mine;
    }
    if (lane < VM) counts[lane][wave] = have_mine;
    __syncthreads();
    if (tid < V) {                                              // up to each wavefront, and all of them
        uint32_t to = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const uint32_t c = counts[tid][w];
            if constexpr (!COUNT) counts[tid][w] = before[tid] + to;
            to += c;
        }
        if constexpr (COUNT) chunks[(size_t)blockIdx.x * kPairMaxV + tid] = to;
        else if (blockIdx.x == gridDim.x - 1) plan[tid] = before[tid] + to;
    }
    if constexpr (!COUNT) {
        __syncthreads();
        uint32_t* rows = plan + pair_rows_at(n, V);
#pragma unroll
        for (int v = 0; v < VM; ++v) {
            if (v >= V) break;
            const unsigned long long have = __ballot(m[v] != FGX_EMPTY32);
            const uint32_t at = counts[v][wave] + (uint32_t)__popcll(have & ((1ull << lane) - 1ull));
            if (m[v] != FGX_EMPTY32) rows[(size_t)v * n + at] = m[v];
            words[tid * V + v] = m[v] != FGX_EMPTY32 ? at : FGX_EMPTY32;
        }
        __syncthreads();
        uint32_t* place = plan + pair_place_at() + (size_t)base * V;
#pragma unroll
        for (int i = 0; i < VM; ++i)
            if (i < V && i * kPairChunk + tid < (int)here * V) place[i * kPairChunk + tid] = words[i * kPairChunk + tid];
    }
}

// Lane v < 32 of a wavefront holds offset v's number of pairs: the pairs and the tiles of the offsets up to and with it (lanes above: nothing).
__device__ __forceinline__ void scan_counts(const uint32_t* __restrict__ plan, int V, int lane, uint32_t& pairs, uint32_t& tiles, uint32_t& count) {
    count = lane < V ? plan[lane] : 0u;
    pairs = count;
    tiles = (count + kPairRows - 1) / kPairRows;
#pragma unroll
    for (int d = 1; d < kPairMaxV; d *= 2) {
        const uint32_t p = (uint32_t)__shfl_up((int)pairs, d, 64), t = (uint32_t)__shfl_up((int)tiles, d, 64);
        if (lane >= d) {
            pairs += p;
            tiles += t;
        }
    }
}

// Bytes of a row that a step multiplies, and workgroups on a CU, by the size of the type (see the kernel).
constexpr int pair_slab(int es) { return es == 4 ? 64 : 128; }
constexpr int pair_groups(int es) { return es == 4 ? 4 : 2; }

// Where the weight is read from: as in the tiled gather GEMM, lines of one (offset, K-slab).
//   TR = false: a line is an output column, its K values side by side;  TR = true: a line is a K value, its columns side by side.
struct PairWeight {
    const unsigned char* base;
    uint32_t bytes, v_stride, slab_stride, line_stride;
    int mirrored;           // offset v multiplies the weight of V - 1 - v
};

template <typename Tag, bool TR, int BN_, int WAVES_M>
struct PairCfg {
    using T = typename Tag::type;
    static constexpr int ES = (int)sizeof(T), SLAB = pair_slab(ES), CH = SLAB / 16, SK = SLAB / ES, RPL = 64 / CH;     // (RPL: rows a wave-wide load covers)
    static constexpr int BM = kPairRows, BN = BN_, NW = 4, NT = 256, WAVES_N = NW / WAVES_M;
    static constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N, TM = WM / 32, TN = WN / 32;
    static constexpr int A_PER = BM / RPL / NW;
    static constexpr int LCOLS = BN == 96 ? 128 : BN;               // columns of a transposed line in LDS: whole loads of whole lines
    static constexpr int TCH = LCOLS * ES / 16, LINES = 64 / TCH;   // 16-byte pieces of a transposed line, lines a load covers
    static constexpr int B_PER = TR ? SK / LINES / NW : (BN / RPL + NW - 1) / NW;
    static constexpr int BROWS = TR ? LCOLS : B_PER * NW * RPL;     // (whole loads on every wavefront: of 96 columns' fp32 the last fetch nothing)
    static constexpr int LPS = A_PER + B_PER;
    static constexpr int STAGE = (BM + BROWS) * SLAB, S = 2;
    static constexpr int tr_key(int line) { return ES != 2 ? 0 : (TCH >= 16 ? 4 * (line & 3) : 2 * (line & 3)); }   // 4 lines of a transposing read, 4 bank groups
    static constexpr int PITCH = 32 * 4 + 16;                       // epilogue band of a wavefront: 32 rows of 32 sums
    static constexpr size_t lds_bytes = S * STAGE;
    static_assert(NW * 32 * PITCH <= S * STAGE, "the epilogue bands lie in the ring");
    static_assert(pair_groups(ES) * lds_bytes <= 160 * 1024, "workgroups that share a CU: one multiplies while the others wait for loads");
};

// One tile of 128 pairs x 128 columns (fp32: 96 or 64) per workgroup, four wavefronts of 64 x 64, K in slabs of 128 bytes through two stages: a
// stage's fragments are taken into registers, the loads two slabs on go out into it, and the products run meanwhile.  Two
// workgroups per CU cover each other's barriers.  XCD x takes the x-th eighth of the (column tile, row tile) list, so a part of
// the weight -- the larger operand here -- crosses to one XCD only.
// 864 voxels x 1024 channels (11 022 pairs, 57 MB of weight) 44 us, 513 TFLOP/s; 3 758 voxels 146 us, 695 TFLOP/s.  Tiles of 128 x 256 and 256 x 128 on
// eight wavefronts, rings of three to five slabs, slabs of 64 bytes, and loads by wavefronts of their own in a persistent workgroup came out between
// 0.9 and 1.2 of that time, ahead only for the second, behind for everything smaller.
// fp32 multiplies three bf16 parts of every value (split3.h), six products for one: half as long a slab is enough work for a barrier, and its
// stages and fragments let four workgroups share a CU, which cover the few slabs' start and end (96 channels have three of 128 bytes). It is bound by making
// the parts (208 vector instructions to 18 products of a wavefront's 32 x 96) and by what it writes: 38 407 voxels, 96 channels, with the sums
// 130 us on the fp32 units (141 in two workgroups of 128-byte slabs, 125 with the sums leaving in bands of 32 columns), 110 in parts (105 before
// both operands were scaled); 16 400 voxels, 128 channels 76 -> 71, 256 channels 227 -> 208; error against 64 bits 1.90e-7 -> 1.56e-7. A tile with a sum that the parts cannot stand for is multiplied
// a second time, on the fp32 units.
template <typename Tag, bool TR, int BN, int WAVES_M>
__global__ void __launch_bounds__(256, pair_groups((int)sizeof(typename Tag::type)))
pair_gemm_kernel(const typename Tag::type* __restrict__ src, PairWeight b, const uint32_t* __restrict__ plan, uint32_t n, int K, int cols,
                 int V, uint32_t src_bytes, float* __restrict__ partial) {
    using C = PairCfg<Tag, TR, BN, WAVES_M>;
    constexpr int CH = C::CH;
    extern __shared__ __attribute__((aligned(16))) unsigned char ring[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave_m = wave / C::WAVES_N, wave_n = wave % C::WAVES_N;

    uint32_t pairs_to, tiles_to, count;
    scan_counts(plan, V, lane, pairs_to, tiles_to, count);
    const uint32_t row_tiles = (uint32_t)__builtin_amdgcn_readlane((int)tiles_to, kPairMaxV - 1);
    const uint32_t total = row_tiles * ((cols + C::BN - 1) / C::BN), per_xcd = (total + kXcds - 1) / kXcds;
    const uint32_t logical = (blockIdx.x % kXcds) * per_xcd + blockIdx.x / kXcds;
    if (blockIdx.x / kXcds >= per_xcd || logical >= total) return;      // whole workgroup
    const uint32_t col_tile = logical / row_tiles, row_tile = logical % row_tiles;
    const int v = __builtin_amdgcn_readfirstlane(__popc((uint32_t)__ballot(tiles_to <= row_tile)));
    const uint32_t have = (uint32_t)__builtin_amdgcn_readlane((int)count, v);
    const uint32_t first = (row_tile - ((uint32_t)__builtin_amdgcn_readlane((int)tiles_to, v) - (have + C::BM - 1) / C::BM)) * C::BM;
    const uint32_t live = have - first < (uint32_t)C::BM ? have - first : (uint32_t)C::BM;              // pairs of this tile
    const size_t pair0 = (size_t)((uint32_t)__builtin_amdgcn_readlane((int)pairs_to, v) - have + first);
    const int col0 = (int)col_tile * C::BN;

    const rsrc_t src_rs = make_rsrc(src, src_bytes), b_rs = make_rsrc(b.base, b.bytes);
    const uint32_t* rows = plan + pair_rows_at(n, V) + (size_t)v * n + first;
    const uint32_t row_bytes = (uint32_t)K * C::ES;
    const int slabs = (int)((row_bytes + C::SLAB - 1) / C::SLAB);
    const bool ragged = row_bytes % C::SLAB != 0;

    uint32_t a_off[C::A_PER], a_at[C::A_PER], b_off[C::B_PER], b_at[C::B_PER];      // ..._at: byte (TR: K value) inside the slab
#pragma unroll
    for (int i = 0; i < C::A_PER; ++i) {
        const uint32_t r = (uint32_t)((i * C::NW + wave) * C::RPL + lane / CH);
        a_at[i] = (uint32_t)(((lane & (CH - 1)) ^ swz_key<CH>((int)r)) << 4);
        a_off[i] = r < live ? rows[r] * row_bytes + a_at[i] : kOobOffset;
    }
    const int wv = b.mirrored ? V - 1 - v : v;
#pragma unroll
    for (int i = 0; i < C::B_PER; ++i) {
        if constexpr (TR) {
            const int line = (i * C::NW + wave) * C::LINES + lane / C::TCH;
            const int piece = (lane % C::TCH) ^ C::tr_key(line);
            b_at[i] = (uint32_t)line;
            b_off[i] = piece * (16 / C::ES) < BN && col0 + piece * (16 / C::ES) < cols ? (uint32_t)line * b.line_stride + (uint32_t)(col0 * C::ES + (piece << 4)) : kOobOffset;
        } else {
            const int col = (i * C::NW + wave) * C::RPL + lane / CH;
            b_at[i] = (uint32_t)(((lane & (CH - 1)) ^ swz_key<CH>(col)) << 4);
            b_off[i] = col < BN && col0 + col < cols ? (uint32_t)(col0 + col) * b.line_stride + b_at[i] : kOobOffset;
        }
    }
    uint32_t b_soff = 0;
    auto issue = [&](int slab) {
        unsigned char* stage = ring + (slab & 1) * C::STAGE;
        const bool tail = ragged && slab == slabs - 1;
        const uint32_t a_soff = (uint32_t)slab * C::SLAB;
#pragma unroll
        for (int i = 0; i < C::A_PER; ++i) {
            const uint32_t vo = tail && a_soff + a_at[i] >= row_bytes ? kOobOffset : a_off[i];
            __builtin_amdgcn_raw_ptr_buffer_load_lds(src_rs, FGX_LDS_PTR(stage + (i * C::NW + wave) * 1024), 16, vo, a_soff, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < C::B_PER; ++i) {
            const bool past = tail && (TR ? slab * C::SK + (int)b_at[i] >= K : a_soff + b_at[i] >= row_bytes);
            const uint32_t vo = past ? kOobOffset : b_off[i];
            __builtin_amdgcn_raw_ptr_buffer_load_lds(b_rs, FGX_LDS_PTR(stage + C::BM * C::SLAB + (i * C::NW + wave) * 1024), 16, vo, b_soff, 0, 0);
        }
        b_soff += b.slab_stride;
    };

    const int g = lane >> 5, l32 = lane & 31, s16 = lane & 15, half = (lane >> 4) & 1;
    int a_frag[CH / 2][C::TM], b_frag[CH / 2][C::TN];
#pragma unroll
    for (int kk = 0; kk < CH / 2; ++kk)
#pragma unroll
        for (int i = 0; i < C::TM; ++i) a_frag[kk][i] = swz<CH>(wave_m * C::WM + i * 32 + l32, kk * 2 + g);
#pragma unroll
    for (int kk = 0; kk < CH / 2; ++kk)
#pragma unroll
        for (int i = 0; i < C::TN; ++i) {
            if constexpr (TR && C::ES == 2) {
                const int line = kk * 16 + g * 8 + (s16 >> 2), byte = (wave_n * C::WN + i * 32 + half * 16 + (s16 & 3) * 4) * C::ES;
                b_frag[kk][i] = C::BM * C::SLAB + line * (C::TCH * 16) + (((byte >> 4) ^ C::tr_key(line)) << 4) + (byte & 15);
            } else if constexpr (TR) {
                b_frag[kk][i] = C::BM * C::SLAB + (kk * 8 + g * 4) * (C::TCH * 16) + (wave_n * C::WN + i * 32 + l32) * C::ES;
            } else {
                b_frag[kk][i] = C::BM * C::SLAB + swz<CH>(wave_n * C::WN + i * 32 + l32, kk * 2 + g);
            }
        }
    f32x16 acc[C::TM][C::TN];
    // fp32: which way the columns and the sums count at present.  What the matrix unit drops of its sums points downwards, the more the larger they are; turned after
    // two thirds of the slabs, nine tenths of it cancel, and every other offset starts with the other sign.  Mean error of the outputs over their root mean
    // square, 1 976 voxels, 1024 channels: -1.9e-7 -> 7e-11, 2-norm 5.3e-7 -> 4.9e-7 (fp32 units 5.8e-7).
    float scale = wv & 1 ? -kSplit3Scale : kSplit3Scale;
    const int turn_at = (2 * slabs + 1) / 3;
    auto multiply = [&](auto on_fp32_units) __attribute__((always_inline)) {
        constexpr bool SPLIT = C::ES == 4 && !decltype(on_fp32_units)::value;
        b_soff = (uint32_t)wv * b.v_stride;
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
#pragma unroll
            for (int j = 0; j < C::TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

        issue(0);
        if (slabs > 1) issue(1);
        for (int s = 0; s < slabs; ++s) {
            if (SPLIT && s == turn_at) {
                scale = -scale;
                asm volatile("" ::: "memory");         // (a branch, not a choice per sum in every step)
#pragma unroll
                for (int i = 0; i < C::TM; ++i)
#pragma unroll
                    for (int j = 0; j < C::TN; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[i][j][e] = -acc[i][j][e];
            }
            if (s + 1 < slabs) wait_vmcnt<C::LPS>();        // all but the newest slab's loads have landed
            else wait_vmcnt<0>();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            const unsigned char* cur = ring + (s & 1) * C::STAGE;
            u32x4 af[CH / 2][C::TM], bf[CH / 2][C::TN];
            i16x4 tr[TR && C::ES == 2 ? CH * C::TN : 4];
#pragma unroll
            for (int kk = 0; kk < CH / 2; ++kk) {
#pragma unroll
                for (int i = 0; i < C::TM; ++i) af[kk][i] = *(const u32x4*)(cur + a_frag[kk][i]);
#pragma unroll
                for (int j = 0; j < C::TN; ++j) {
                    if constexpr (TR && C::ES == 2) {       // (K rows 4 apart share a key)
                        tr[(kk * C::TN + j) * 2] = lds_read_tr16(cur + b_frag[kk][j]);
                        tr[(kk * C::TN + j) * 2 + 1] = lds_read_tr16(cur + b_frag[kk][j] + 4 * C::TCH * 16);
                    } else if constexpr (TR) {
#pragma unroll
                        for (int e = 0; e < 4; ++e) bf[kk][j][e] = *(const uint32_t*)(cur + b_frag[kk][j] + e * C::TCH * 16);
                    } else {
                        bf[kk][j] = *(const u32x4*)(cur + b_frag[kk][j]);
                    }
                }
            }
            if constexpr (TR && C::ES == 2) {
                lds_wait_all(tr);
#pragma unroll
                for (int kk = 0; kk < CH / 2; ++kk)
#pragma unroll
                    for (int j = 0; j < C::TN; ++j)
                        bf[kk][j] = __builtin_bit_cast(u32x4, __builtin_shufflevector(tr[(kk * C::TN + j) * 2], tr[(kk * C::TN + j) * 2 + 1], 0, 1, 2, 3, 4, 5, 6, 7));
            }
            if (s + 2 < slabs) {
                // every wavefront's fragments are in registers before the stage is written again
                asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                issue(s + 2);
            }
            if constexpr (SPLIT) {
#pragma unroll
                for (int kk = 0; kk < CH / 2; kk += 2) {        // (16 values of K a product)
                    Split3 rows3[C::TM];
#pragma unroll
                    for (int i = 0; i < C::TM; ++i) rows3[i] = split3(af[kk][i], af[kk + 1][i]);
#pragma unroll
                    for (int j = 0; j < C::TN; ++j) {
                        const Split3 cols3 = split3(bf[kk][j], bf[kk + 1][j], scale);
#pragma unroll
                        for (int i = 0; i < C::TM; ++i) mma_split3(acc[i][j], cols3, rows3[i]);     // transposed tile
                    }
                }
            } else {
#pragma unroll
                for (int kk = 0; kk < CH / 2; ++kk)
#pragma unroll
                    for (int i = 0; i < C::TM; ++i)
#pragma unroll
                        for (int j = 0; j < C::TN; ++j) mma<Tag>(acc[i][j], bf[kk][j], af[kk][i]);      // transposed tile
            }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();           // the ring is reused below
        asm volatile("" ::: "memory");
    };
    multiply(std::false_type{});
    if constexpr (C::ES == 4) {
        bool fine = true;
#pragma unroll
        for (int i = 0; i < C::TM; ++i)
#pragma unroll
            for (int j = 0; j < C::TN; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) fine = fine && split3_holds(acc[i][j][e]);
        volatile uint32_t* told = (volatile uint32_t*)ring;
        const bool all = __ballot(!fine) == 0;
        if (lane == 0) told[wave] = all;
        __syncthreads();
        const bool every = told[0] & told[1] & told[2] & told[3];
        __syncthreads();
        if (!every) {
            multiply(std::true_type{});
        } else {
            const float unscale = scale < 0.f ? -kSplit3Unscale : kSplit3Unscale;
#pragma unroll
            for (int i = 0; i < C::TM; ++i)
#pragma unroll
                for (int j = 0; j < C::TN; ++j)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[i][j][e] *= unscale;
        }
    }

    // element e of lane l: pair l % 32, column 8 * (e / 4) + 4 * (l / 32) + e % 4.  Through the wavefront's band in LDS, 32 columns at a time, out as
    // 16-byte pieces of 128 bytes a pair.
    unsigned char* band = ring + wave * 32 * C::PITCH;
    constexpr int QUADS = 8;            // 16-byte pieces of a band row
#pragma unroll
    for (int i = 0; i < C::TM; ++i) {
#pragma unroll
        for (int j = 0; j < C::TN; ++j) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const f32x4 four = {acc[i][j][q * 4], acc[i][j][q * 4 + 1], acc[i][j][q * 4 + 2], acc[i][j][q * 4 + 3]};
                *(f32x4*)(band + l32 * C::PITCH + (q * 8 + g * 4) * 4) = four;
            }
            // (written and read by the same wavefront: program order suffices)
#pragma unroll
            for (int pass = 0; pass < 32 * QUADS / 64; ++pass) {
                const int r = (pass * 64 + lane) / QUADS, quad = (pass * 64 + lane) % QUADS, col = col0 + wave_n * C::WN + j * 32 + quad * 4;
                const uint32_t row = (uint32_t)(wave_m * C::WM + i * 32 + r);
                if (row < live && col < cols) *(f32x4*)(partial + (pair0 + row) * cols + col) = *(const f32x4*)(band + r * C::PITCH + quad * 16);
            }
        }
    }
}

// out[r] = act(sum over the offsets of row r, in order, of its partial sums + bias): tpr = min(cols / 4, 256) threads a row, four columns
// each, four partial sums in flight.  It waits for memory: 45 MB
// of sums in 9.5 us (4.7 TB/s).
template <typename T>
__global__ void __launch_bounds__(256) pair_reduce_kernel(const float* __restrict__ partial, const uint32_t* __restrict__ plan, uint32_t n, int cols,
                                                          int V, const T* __restrict__ bias, int act, T* __restrict__ out,
                                                          uint8_t* __restrict__ relu_mask) {
    using Out = T __attribute__((ext_vector_type(4)));
    __shared__ uint32_t pair_of[256 / 8][kPairMaxV];
    __shared__ int pairs[256 / 8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int quads = cols / 4, tpr = quads < 256 ? quads : 256;
    const int rows = 256 / tpr < 32 ? 256 / tpr : 32;
    uint32_t pairs_to, tiles_to, count;
    scan_counts(plan, V, lane, pairs_to, tiles_to, count);
    const uint32_t* place = plan + pair_place_at();
    const uint32_t r0 = blockIdx.x * (uint32_t)rows;
    for (int i = wave; i < rows; i += 4) {
        const uint32_t at = r0 + i < n && lane < V ? place[(size_t)(r0 + i) * V + lane] : FGX_EMPTY32;
        const unsigned long long have = __ballot(at != FGX_EMPTY32);
        if (at != FGX_EMPTY32) pair_of[i][__popcll(have & ((1ull << lane) - 1ull))] = pairs_to - count + at;
        if (lane == 0) pairs[i] = __popcll(have);
    }
    __syncthreads();
    const int mine = (int)threadIdx.x / tpr;
    const uint32_t r = r0 + mine;
    if (mine >= rows || r >= n) return;
    const int m = pairs[mine];
    const f32x4* from = (const f32x4*)partial;
    for (int c = (int)threadIdx.x % tpr; c < quads; c += tpr) {
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        int u = 0;
        for (; u + 4 <= m; u += 4) {
            f32x4 x[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) x[q] = from[(size_t)pair_of[mine][u + q] * quads + c];
#pragma unroll
            for (int q = 0; q < 4; ++q) s += x[q];
        }
        for (; u < m; ++u) s += from[(size_t)pair_of[mine][u] * quads + c];
        Out rounded;
        uint32_t bits = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float bv = bias != nullptr ? to_float<T>(bias[c * 4 + e]) : 0.f;
            rounded[e] = from_float<T>(activate(s[e] + bv, act));
            bits |= (uint32_t)(to_float<T>(rounded[e]) > 0.f) << e;
        }
        const size_t i = (size_t)r * quads + c;
        ((Out*)out)[i] = rounded;
        if (relu_mask != nullptr) {
            const uint32_t other = (uint32_t)__shfl_xor((int)bits, 1, 64);
            if ((i & 1) == 0) relu_mask[i >> 1] = (uint8_t)(bits | other << 4);
        }
    }
}

size_t most_tiles(size_t n, int V) { return (size_t)V * cdiv(n, kPairRows); }

template <typename Tag, bool TR, int BN, int WAVES_M>
int launch_gemm(const void* src, const PairWeight& b, const uint32_t* plan, size_t n, size_t n_src, int K, int cols, int V, float* partial, hipStream_t s) {
    using C = PairCfg<Tag, TR, BN, WAVES_M>;
    using T = typename Tag::type;
    const unsigned grid = cdiv(most_tiles(n, V) * cdiv(cols, BN), kXcds) * kXcds;
    pair_gemm_kernel<Tag, TR, BN, WAVES_M><<<grid, C::NT, C::lds_bytes, s>>>((const T*)src, b, plan, (uint32_t)n, K, cols, V,
                                                                   (uint32_t)(n_src * (size_t)K * sizeof(T)), partial);
    FGX_CHECK_LAUNCH("fgx_conv_gemm_pairs");
    return FGX_OK;
}

template <typename Tag, bool TR>
int launch_pairs(const void* src, const PairWeight& b, const void* bias, const uint32_t* plan, size_t n, size_t n_src, int K, int cols, int V,
                 float* partial, int act, void* out, uint8_t* relu_mask, hipStream_t s) {
    using T = typename Tag::type;
    // Columns of a tile.  fp32 is bound by what it multiplies: 96 where that pads less, else 64, whose smaller pieces even out better (96
    // channels, 38 407 voxels 0.126 ms, 64 columns 0.148; 512 channels, 3 758 voxels 0.240, 128 columns 0.245; 1024 channels, 864 voxels 0.241 and 0.257;
    // 256 channels, 15 467 voxels 0.273 and 0.262).  16-bit types load half as much per product
    // with 128: those unless they pad by a sixth or leave CUs without a tile (864 voxels: 256 channels 64 columns 16.4 us, 128 16.8; 288 channels
    // 18.1 and 19.3; 512 channels 24.5 and 22.9; 3 758 voxels, 1024 channels 217 and 177).
    int rc;
    if constexpr (sizeof(T) == 4) {
        rc = cdiv(cols, 96) * 96 < cdiv(cols, 64) * 64 ? launch_gemm<Tag, TR, 96, 4>(src, b, plan, n, n_src, K, cols, V, partial, s)
                                                       : launch_gemm<Tag, TR, 64, 2>(src, b, plan, n, n_src, K, cols, V, partial, s);
    } else {
        const size_t tiles = (size_t)V * cdiv(n * 9, 20 * kPairRows) * cdiv(cols, 128);     // (a little under half of a row's offsets exist)
        const bool narrow = tiles < 224 || cdiv(cols, 128) * 128 * 6 > cdiv(cols, 64) * 64 * 7;
        rc = narrow ? launch_gemm<Tag, TR, 64, 2>(src, b, plan, n, n_src, K, cols, V, partial, s)
                    : launch_gemm<Tag, TR, 128, 2>(src, b, plan, n, n_src, K, cols, V, partial, s);
    }
    if (rc != FGX_OK) return rc;
    const int quads = cols / 4, tpr = quads < 256 ? quads : 256, rows = 256 / tpr < 32 ? 256 / tpr : 32;
    pair_reduce_kernel<T><<<cdiv(n, rows), 256, 0, s>>>(partial, plan, (uint32_t)n, cols, V, (const T*)bias, act, (T*)out, relu_mask);
    FGX_CHECK_LAUNCH("fgx_conv_gemm_pairs(sums)");
    return FGX_OK;
}

}  // namespace
}  // namespace fgx

using namespace fgx;

extern "C" {

// Where the products of the pairs and their sums are ahead of the masked kernels.  Pairs of figures: masked kernels, this, us a call without
// their plans; a plan costs 4 for 864 rows, 8 for 3 758, 13 for 38 407, and stands for the tile masks or gather plan (3 to 15) and, at inference,
// for the mask sort.
// 16-bit types.  Per pair the sums are 8 bytes an output column, the products 2 K: rows of 256 channels and more.  The lead goes where the tiles
// pad less and the streaming kernel sets in, at rows that depend little on K: up to 6 000 under as many columns as channels or fewer, up to
// 5 000 under more, of which the sums are larger beside the masked kernels' traffic.
//   K x columns    864 rows   2 047    3 758    4 753    5 914    6 543      K x columns    3 758     4 753     5 318     5 914
//    256 x  256      26  17   32  24   39  32   51  36   53  45   52  48      256 x  512    54  54    70  62    69  68    70  77
//    512 x  512      36  24   49  39   77  67  128  84  120  97               384 x  768    98  83   100 103   100 114   115 130
//    768 x  768      58  37  103  67  178 116  179 144  277 180  298 200      512 x 1024   134 122   200 159   151 181   158 208
//   1024 x 1024      76  49  144  98  242 182  385 231  299 301  317 338      768 x 1024   194 151   288 193   228 222   226 251
//   1024 x  128      33  18   35  22   48  30   73  34   74  45              1024 x 2048   447 379   809 480   814 542   829 609
// 64 columns (256 x 64: 15 12, 20 14, 24 19, 33 20, 34 21) gain little more than the plan: a training step whose input gradient still wants the
// masks is up to 5 % slower for it, a pass at inference 1.16 to 1.44 times as fast.
// fp32 (figures of the fp32 units on both sides; in three bf16 parts both are shorter, and level where they were: 49 976 rows, kept, 64 x 64 81 76, 96 x 96
// 167 127, 128 x 128 219 209, 160 x 160 340 340):  what is not multiplied counts for more than in 16 bits: from 64 channels on, up to a number of rows and as long as the sums,
// with 0.45 of a row's offsets, stay below 5 MB a channel.  Their traffic, which outgrows the 256 MB memory-side cache, costs what the products
// save from 4.5 MB on, and by 5 MB also the 30 to 50 us of tables that a fresh cache is spared (64 x 256, cache and one layer, 27 200 rows: forward
// 248 230, training 552 543;  38 400 rows: 354 325, 765 750;  24 400 rows, training 500 459).  Beyond: 96 x 96, 71 359 rows 244 250,
// 84 634 rows 250 297;  128 x 128 438 378, 451 453;  160 x 160 595 617, 732 739;  256 x 96, 99 042 rows 857 631.
// Kernels of more than 8 offsets: 65 536 rows, 98 304 under at most half as many columns as channels.  The masked kernels multiply whole slabs of 32
// channels, two of which 64 channels fill where 65 ... 96 are padded to three: 28 800 and 32 768 rows a slab (one layer, its cache included or kept,
// inference fresh, kept, training fresh, kept:  64 x 64, 56 428 rows 165 126, 106 103, 375 334, 292 289, 64 090 rows 166 139, 105 117, 383 375, 299 326;
// 64 x 32, 56 428 rows 124 105, 75 80, 305 321, 223 226, 96 531 rows 174 165, 119 131, 431 466, 331 350;  72 x 72, 64 090 rows 269 204, 206 179,
// 658 569, 570 516, 83 458 rows 277 274, 210 242, 713 742, 621 679;  72 x 32, 83 458 rows 186 161, 134 131, 524 539, 431 433;  128 x 32 249 210, 196 179,
// 613 619, 523 508).
// Up to 8 offsets, whose masks the sort brings together almost without padding: 45 000 rows, under at most half as many columns 65 536, 22 500 a slab (2 x 2 x 2,
// stride 2, kept: 96 x 96, 60 500 rows 56 77, 76 600 rows 67 91;  128 x 128 132 105, 107 131;  96 x 192, 48 000 rows 82 101;  64 x 64, 48 149 input rows,
// training 56 60, 54 406 rows 58 88;  128 x 64, 64 600 rows 93 68, 76 600 rows 68 78;  256 x 128 180 179, 201 216;  64 x 32, fresh, 48 000 rows 95 102).
//   K x columns    855 rows   8 589    15 474    24 372    38 323    48 203    63 137      up to
//     64 x   64      16  13    38  29    54  38    67  55    89  75   111  87   111 112      57 600 rows
//     64 x  256      23  17    96  66   116 108   192 178   259                               25 720 (the sums' bound)
//     96 x   96      21  15    66  39   108  62   158  87   157 126   260 158   244 217      65 536
//     96 x  192      27  18   104  64   151 101   217 153   260 263   356 330   365          51 440 (the sums' bound)
//    128 x  256      32  22   165  93   216 156   367 254   493 407   492                    38 836 (1 GiB)
//    128 x  512      52  33   302 179   354 324   541       824                              19 418 (the same)
//    256 x  128      32  20   193  84   317 136   412 209   618 328   639 416   720 544      77 672 (the same)
//    256 x  256      52  30   331 151   417 264   715 414   962 658   953                    38 836 (the same)
// The sums at most 1 GiB at their bound.
int fgx_conv_gemm_pairs_pays(int dtype, int mode, size_t n, int Ci, int Co, int V) {
    if (mode < 0 || mode > 2 || V < 1 || V > kPairMaxV || Ci <= 0 || Co <= 0 || n == 0) return 0;
    const int es = dtype == FGX_F32 ? 4 : 2, K = mode == 0 ? Ci : Co, cols = mode == 0 ? Co : Ci;
    if (Ci % (16 / es) != 0 || Co % (16 / es) != 0 || (size_t)V * Ci * Co * es >= ((size_t)1 << 31)) return 0;
    if (n > 98304 || fgx_conv_gemm_pairs_scratch_bytes(n, cols, V) > ((size_t)1 << 30)) return 0;
    if (es == 4) {
        const size_t slabs = cdiv(K, 32);
        const bool half = cols * 2 <= K;
        size_t rows = V <= 8 ? (half ? 22500 * slabs : 45000) : (half ? 32768 : 28800) * slabs;
        if (rows > 65536 && (V <= 8 || !half)) rows = 65536;
        return K >= 64 && n <= rows && 0.45 * (double)fgx_conv_gemm_pairs_scratch_bytes(n, cols, V) <= 5e6 * K;
    }
    return K >= 256 && cols >= 64 && cols <= 2 * K && n <= (cols <= K ? 6000u : 5000u);
}

size_t fgx_pair_plan_words(size_t n, int V) {
    return V >= 1 && V <= kPairMaxV ? pair_chunks_at(n, V) + (size_t)cdiv(n, kPairChunk) * kPairMaxV : 0;
}

int fgx_pair_plan(const uint32_t* map, size_t n, int V, uint32_t* plan, fgx_stream_t stream) {
    FGX_CHECK_ARG(V >= 1 && V <= kPairMaxV && n < ((size_t)1 << 26), "fgx_pair_plan: %zu rows, V=%d out of range", n, V);
    FGX_CHECK_ARG(plan != nullptr && (n == 0 || map != nullptr), "fgx_pair_plan: null buffer");
    if (n <= (size_t)kPairColumnRows) {
        pair_plan_columns_kernel<<<V, 1024, 0, (hipStream_t)stream>>>(map, (uint32_t)n, V, plan);
        FGX_CHECK_LAUNCH("fgx_pair_plan");
        return FGX_OK;
    }
    const unsigned chunks = cdiv(n, kPairChunk);
    const size_t lds = (size_t)kPairChunk * V * sizeof(uint32_t);
#define FGX_PLAN(VC)                                                                                                                \
    do {                                                                                                                            \
        pair_plan_kernel<true, VC><<<chunks, kPairChunk, lds, (hipStream_t)stream>>>(map, (uint32_t)n, V, plan);    \
        pair_plan_kernel<false, VC><<<chunks, kPairChunk, lds, (hipStream_t)stream>>>(map, (uint32_t)n, V, plan);                   \
    } while (0)
    if (V == 27) FGX_PLAN(27);
    else if (V == 8) FGX_PLAN(8);
    else FGX_PLAN(0);
#undef FGX_PLAN
    FGX_CHECK_LAUNCH("fgx_pair_plan");
    return FGX_OK;
}

size_t fgx_conv_gemm_pairs_scratch_bytes(size_t n, int cols, int V) { return n * (size_t)V * (size_t)(cols > 0 ? cols : 0) * sizeof(float); }

int fgx_conv_gemm_pairs(int dtype, int mode, const void* src, const void* weight, const void* bias, const uint32_t* plan, size_t n, size_t n_src,
                        int Ci, int Co, int V, void* scratch, int activation, void* out, uint8_t* relu_mask, fgx_stream_t stream) {
    FGX_CHECK_ARG(activation == FGX_ACT_NONE || activation == FGX_ACT_RELU, "fgx_conv_gemm_pairs: unknown activation %d", activation);
    FGX_CHECK_ARG(dtype == FGX_F16 || dtype == FGX_BF16 || dtype == FGX_F32, "fgx_conv_gemm_pairs: unknown dtype %d", dtype);
    FGX_CHECK_ARG(mode >= 0 && mode <= 2 && V >= 1 && V <= kPairMaxV && Ci > 0 && Co > 0, "fgx_conv_gemm_pairs: bad shape, mode %d Ci=%d Co=%d V=%d",
                  mode, Ci, Co, V);
    const int es = dtype == FGX_F32 ? 4 : 2, K = mode == 0 ? Ci : Co, cols = mode == 0 ? Co : Ci;
    FGX_CHECK_ARG(Ci % (16 / es) == 0 && Co % (16 / es) == 0, "fgx_conv_gemm_pairs: rows of %d and %d elements are not whole 16-byte pieces", Ci, Co);
    FGX_CHECK_ARG(relu_mask == nullptr || (activation == FGX_ACT_RELU && es == 2), "fgx_conv_gemm_pairs: a ReLU mask needs the ReLU and a 16-bit type");
    if (n == 0) return FGX_OK;
    FGX_CHECK_ARG(src && weight && plan && scratch && out, "fgx_conv_gemm_pairs: null buffer");
    FGX_CHECK_ARG((((uintptr_t)src | (uintptr_t)weight | (uintptr_t)scratch | (uintptr_t)out) & 15) == 0, "fgx_conv_gemm_pairs: buffers must be 16-byte aligned");
    const size_t weight_bytes = (size_t)V * Ci * Co * es, src_bytes = n_src * (size_t)K * es;
    FGX_CHECK_ARG(weight_bytes < ((size_t)1 << 31) && src_bytes <= kOobOffset && n * (size_t)V < 0xFFFFFFFFull && n < 0x7FFFFFFFull &&
                      most_tiles(n, V) * cdiv(cols, 64) < 0x7FFFFFF0ull,
                  "fgx_conv_gemm_pairs: an operand exceeds the 32-bit offset range");
    PairWeight b;                                           // [Co][V][Ci]
    b.base = (const unsigned char*)weight;
    b.bytes = (uint32_t)weight_bytes;
    b.v_stride = (uint32_t)(Ci * es);
    b.line_stride = (uint32_t)((size_t)V * Ci * es);
    b.slab_stride = mode == 0 ? (uint32_t)pair_slab(es) : (uint32_t)(pair_slab(es) / es) * b.line_stride;
    b.mirrored = mode == 1;
    hipStream_t s = (hipStream_t)stream;
#define FGX_PAIRS(Tag)                                                                                                                              \
    return mode == 0 ? launch_pairs<Tag, false>(src, b, bias, plan, n, n_src, K, cols, V, (float*)scratch, activation, out, relu_mask, s)           \
                     : launch_pairs<Tag, true>(src, b, bias, plan, n, n_src, K, cols, V, (float*)scratch, activation, out, relu_mask, s)
    if (dtype == FGX_F16) FGX_PAIRS(F16);
    if (dtype == FGX_BF16) FGX_PAIRS(BF16);
    FGX_PAIRS(F32);
#undef FGX_PAIRS
}

}  // extern "C"
