// Which row holds the voxel at a cell of the grid: the index the neighbor maps of surfaces and blocks are looked up in.
//
// Two forms, chosen by the grid's size alone (grid_index_plan):
//   cells   one word per cell, the row of its voxel or EMPTY.  Two launches (clear, insert) and one load per question; the
//           clear is what it costs, so up to kDenseMaxCells cells (32 MiB, which the last-level cache holds).
//   bits    one bit per cell, a running count of the set bits for every 128 of them, and the rows in cell order: five
//           launches, an eighth of a byte per cell.  A question reads 16 bytes of bits and 4 of counts, and a row when
//           the bit is set.  The rows in cell order double as a walk over the voxels on which neighboring questions fall
//           into the same lines, whatever order the voxels come in.
// A voxel given several times is found under its smallest row number, and voxels outside the grid are not found; the `bits`
// form lists the rows that lost their cell behind the others, so that its walk visits every row once.
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
    int B, W, H, D;
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
    size_t bits, counts, state, rows, total;        // byte offsets; [bits, state + state bytes) is cleared to 0, rows to EMPTY
    size_t zero_bytes;
};

// false: the grid is too large for either form
bool grid_index_plan(size_t n, int B, int W, int H, int D, GridIndexLayout* out);
// the rule of the "auto" builder: forms that fit are also worth their clears
bool grid_index_pays(size_t n, int B, int W, int H, int D);
int grid_index_build(const int32_t* coords, size_t n, int B, int W, int H, int D, const GridIndexLayout& L, void* workspace, GridIndex* out,
                     hipStream_t s, const char* what);

// Submanifold map over a planned index.  counts (optional, [V][ceil(n / kPairSubRows)]): set mask bits per kPairSubRows rows;
// *counted says whether they were written (the `cells` form does).
int subm_map_grid(const int32_t* coords, size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dw, int Dh, int Dd,
                  const GridIndexLayout& L, void* workspace, uint32_t* out_map, int32_t* gray, int32_t* binary, uint32_t* counts,
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

// row of the voxel at a cell inside the grid, or EMPTY
template <bool DENSE>
__device__ __forceinline__ uint32_t grid_find(const GridIndex& g, size_t cell) {
    if constexpr (DENSE) {
        return g.cells[cell];
    } else {
        const size_t block = cell >> 7;
        const ulonglong2 w = g.bits[block];
        const unsigned at = (unsigned)cell & 127u;
        const unsigned long long word = at & 64u ? w.y : w.x;
        if (((word >> (at & 63u)) & 1ull) == 0ull) return FGX_EMPTY32;
        const unsigned long long below = word & ((1ull << (at & 63u)) - 1ull);
        const uint32_t rank = g.counts[block] + (uint32_t)__popcll(below) + (at & 64u ? (uint32_t)__popcll(w.x) : 0u);
        return g.rows[rank];
    }
}
#endif

}  // namespace fgx
