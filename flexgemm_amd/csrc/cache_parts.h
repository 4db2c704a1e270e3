// Steps of the neighbor cache shared by its builders (defined in neighbor_post.hip).
#pragma once
#include "fgx_common.h"

namespace fgx {

constexpr int kPairRows = 256;          // voxels per block of the pair lists
constexpr int kPairSubRows = 64;        // voxels per count when the map's kernel counts as it goes

// Pair lists from counts[V][m] of the set mask bits of every kPairRows rows, or of every kPairSubRows when `sub` is set
// (m = rows / that, rounded up): scan and fill, the segment table written on the way.  offsets: V * ceil(n / kPairRows)
// words, totals: 32 words.  seg_host (optional): pinned host memory the table is written to as well.
int pair_lists_from_counts(const uint32_t* map, const int32_t* gray, size_t n, int V, const uint32_t* counts, size_t m, bool sub,
                           uint32_t* offsets, uint32_t* totals, uint32_t* seg, uint32_t* seg_host, uint32_t* sig_i, uint32_t* sig_o,
                           hipStream_t s);
int pair_counts(const int32_t* gray, size_t n, int V, uint32_t* counts, hipStream_t s);

}  // namespace fgx
