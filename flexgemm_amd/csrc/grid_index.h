// Which row holds the voxel at a cell of the grid: the index the neighbor maps of surfaces and blocks are looked up in.
//
// Two forms, chosen by the grid's size alone (grid_index_plan):
//   cells   one word per cell, the row of its voxel or EMPTY.  Two launches (clear, insert) and one load per question; the
//           clear is what it costs, so up to kDenseMaxCells cells (32 MiB, which the last-level cache holds).
//   bits    one bit per cell, a running count of the set bits for every 128 of them, and the rows in cell order: five
//           launches, an eighth of a byte per cell.  A question reads 16 bytes of bits and 4 of counts, and a row when
//           the bit is set.  128 cells are a brick of 2 x 2 x 32, and bricks follow a Z-order curve across columns of 8 x 8: a
//           bit map's word still is 32 cells along z, which voxels in scan order fill together, but the 27 cells around a voxel
//           lie in 4 bricks instead of 9 rows, a surface's voxels in fewer lines, and any 128 of the rows in cell order are a
//           compact patch -- the row order that the narrow layers' plan wants (narrow_plan.h), without a sort.  2 667 120 voxels
//           of a 1024^3 surface: the cache in scan order 0.407 -> 0.367 ms against cells in their own order, in random order
//           0.735 -> 0.687, and the plan's four sorting passes (0.26 ms) gone.  (Bricks of 4 x 4 x 8: 0.402 and 0.675, but 0.010
//           more in scan order at 400 000 voxels, where four times as many words are set.)
//           Map rows are walked in cell order when the voxels come in no order of their own.
// A voxel given several times is found under its smallest row number, and voxels outside the grid are not found; the `bits`
// form lists the rows that lost their cell behind the others (in row order where the walk is the caller's), so that its walk
// visits every row once.
//
// Against the hash table (hash_build.hip) a question is one or two reads of a few neighboring lines instead of a probe at a
// pseudo-random place; against sort and merge (neighbor_sorted.hip) nothing is sorted.
#pragma once
#include "fgx_common.h"

namespace fgx {

struct GridIndex {
    const uint32_t* cells;          // `cells` form (bits == nullptr)
    const ulonglong2* bits;         // `bits` form: 128 cells each
    const uint32_t* counts;         // set bits before each 128
    const uint32_t* rows;           // rows in cell order, then the rows without a cell
    const uint32_t* order;          // [0] set bits, [1] neighboring rows that step back, of the looked-at ones (grid_in_scan_order)
    int B, W, H, D;
    uint32_t shift;                 // `bits` form: bricks per edge of a column, as a power of two
    uint32_t step_b, step_x, step_y;        // ... and bricks from one column to the next along an axis
};

constexpr size_t kDenseMaxCells = (size_t)1 << 23;
// bit maps of up to 16 MiB cost a few microseconds to clear and count; larger ones (up to 512 MiB) as long as they are no
// more than 64 bytes per voxel -- a surface's is 50 bytes at 1024^3 -- since clearing and counting then costs about what the
// look-ups do.  Beyond, the hash and the sorted builders do not depend on the grid's volume.
constexpr size_t kBitsAlwaysMaxBytes = (size_t)16 << 20, kBitsMaxBytes = (size_t)512 << 20, kBitsBytesPerVoxel = 64;

struct GridIndexLayout {
    bool dense;
    size_t cells;                   // B * W * H * D
    size_t blocks, tiles;           // `bits` form: 128-bit blocks, tiles of the count
    size_t bits, counts, state, losers, rows, total;        // byte offsets; [bits, losers + its bytes) is cleared to 0, rows to EMPTY
    size_t zero_bytes;
    uint32_t shift;                 // as in GridIndex
};

// false: the grid is too large for either form
bool grid_index_plan(size_t n, int B, int W, int H, int D, GridIndexLayout* out);
// the rule of the "auto" builder: forms that fit are also worth their clears
bool grid_index_pays(size_t n, int B, int W, int H, int D);
// walk (optional, `bits` form): n words for the rows in cell order, in place of the workspace's.  plan_header (optional, with a walk): the header
// of a narrow layer's plan, cleared on the way
int grid_index_build(const int32_t* coords, size_t n, int B, int W, int H, int D, const GridIndexLayout& L, void* workspace, uint32_t* walk,
                     uint32_t* plan_header, GridIndex* out, hipStream_t s, const char* what);

// Submanifold map over a planned index.  counts (optional, [V][ceil(n / kPairSubRows)]): set mask bits per kPairSubRows rows;
// *counted says whether they were written (the `cells` form does).  plan (optional, with a walk, 3 x 3 x 3 kernels that grid_plan_fits): the narrow layers'
// plan along the walk, made with the map.
inline bool grid_plan_fits(const GridIndexLayout& L, int Kw, int Kh, int Kd, int Dd) { return !L.dense && Kw == 3 && Kh == 3 && Kd == 3 && Dd <= 16; }
int subm_map_grid(const int32_t* coords, size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dw, int Dh, int Dd,
                  const GridIndexLayout& L, void* workspace, uint32_t* walk, void* plan, uint32_t* out_map, int32_t* gray, int32_t* binary, uint32_t* counts,
                  bool* counted, hipStream_t s);

// Both maps of a generic convolution: an index of the inputs, and of the outputs for the backward map.
struct ConvMapsLayout {
    GridIndexLayout in, out;
    size_t out_at, total;
};
bool conv_maps_plan(size_t n_in, size_t n_out, int B, int W, int H, int D, int Wo, int Ho, int Do, bool with_bwd, ConvMapsLayout* P);
// k: kernel, stride, padding, dilation (three each).  counts as above, of the forward map; written whenever given.
int conv_maps_grid(const int32_t* in_coords, size_t n_in, const int32_t* out_coords, size_t n_out, int B, int W, int H, int D, int Wo, int Ho,
                   int Do, const int* k, const ConvMapsLayout& P, void* workspace, uint32_t* map_fwd, uint32_t* map_bwd, int32_t* gray,
                   int32_t* binary, uint32_t* counts, int32_t* gray_bwd, int32_t* binary_bwd, hipStream_t s);

#if defined(__HIPCC__)
__device__ __forceinline__ size_t grid_cell(const GridIndex& g, int b, int x, int y, int z) {
    return (((size_t)(uint32_t)b * (uint32_t)g.W + (uint32_t)x) * (uint32_t)g.H + (uint32_t)y) * (uint32_t)g.D + (uint32_t)z;
}

// Where a cell's entry is: the sum of one part per axis, so that a kernel's few coordinates along each are taken apart once.
template <bool DENSE>
struct GridPlace;
template <>
struct GridPlace<true> {
    size_t cell;
    __device__ __forceinline__ GridPlace operator+(const GridPlace& o) const { return {cell + o.cell}; }
};
template <>
struct GridPlace<false> {
    uint32_t brick, at;             // 128 cells, and which of them
    __device__ __forceinline__ GridPlace operator+(const GridPlace& o) const { return {brick + o.brick, at + o.at}; }
};

__device__ __forceinline__ uint32_t every_other_bit(uint32_t v) { return (v & 1u) | ((v & 2u) << 1) | ((v & 4u) << 2); }
// part of a brick coordinate: its column's, and its own along the curve within the column
__device__ __forceinline__ uint32_t brick_part(const GridIndex& g, uint32_t v, uint32_t step, int bit) {
    return (v >> g.shift) * step + (every_other_bit(v & ((1u << g.shift) - 1u)) << bit);
}

template <bool DENSE>
__device__ __forceinline__ GridPlace<DENSE> place_bx(const GridIndex& g, int b, int x) {
    if constexpr (DENSE) return {((size_t)(uint32_t)b * (uint32_t)g.W + (uint32_t)x) * (uint32_t)g.H * (uint32_t)g.D};
    else return {(uint32_t)b * g.step_b + brick_part(g, (uint32_t)x >> 1, g.step_x, 1), ((uint32_t)x & 1u) << 6};
}
template <bool DENSE>
__device__ __forceinline__ GridPlace<DENSE> place_y(const GridIndex& g, int y) {
    if constexpr (DENSE) return {(size_t)(uint32_t)y * (uint32_t)g.D};
    else return {brick_part(g, (uint32_t)y >> 1, g.step_y, 0), ((uint32_t)y & 1u) << 5};
}
template <bool DENSE>
__device__ __forceinline__ GridPlace<DENSE> place_z(const GridIndex& g, int z) {
    if constexpr (DENSE) return {(size_t)(uint32_t)z};
    else return {((uint32_t)z >> 5) << (2u * g.shift), (uint32_t)z & 31u};
}
template <bool DENSE>
__device__ __forceinline__ GridPlace<DENSE> grid_place(const GridIndex& g, int b, int x, int y, int z) {
    return place_bx<DENSE>(g, b, x) + place_y<DENSE>(g, y) + place_z<DENSE>(g, z);
}

// Whether the voxels come in scan order, or nearly: one in sixteen of the sampled steps from row to row at most goes back.
constexpr size_t kOrderSamples = 256;           // workgroups of 256 rows that are looked at
__device__ __forceinline__ bool grid_in_scan_order(const GridIndex& g, size_t n) {
    const size_t most = kOrderSamples * 256;
    return (size_t)g.order[1] * 16 <= (n < most ? n : most);
}

// set bits before bit `at` of a brick
__device__ __forceinline__ uint32_t bits_before(const ulonglong2& w, uint32_t at) {
    const unsigned long long below = (at & 64u ? w.y : w.x) & ((1ull << (at & 63u)) - 1ull);
    return (uint32_t)__popcll(below) + (at & 64u ? (uint32_t)__popcll(w.x) : 0u);
}

// row of the voxel at a cell inside the grid, or EMPTY
template <bool DENSE>
__device__ __forceinline__ uint32_t grid_find(const GridIndex& g, const GridPlace<DENSE>& p) {
    if constexpr (DENSE) {
        return g.cells[p.cell];
    } else {
        const ulonglong2 w = g.bits[p.brick];
        if ((((p.at & 64u ? w.y : w.x) >> (p.at & 63u)) & 1ull) == 0ull) return FGX_EMPTY32;
        return g.rows[g.counts[p.brick] + bits_before(w, p.at)];
    }
}
#endif

}  // namespace fgx
