// The neighbor cache of a convolution in one call: the map and its mask codes (grid index or sort-and-merge builder), the
// mask sort, and for a training cache the pair lists -- the calls a host would otherwise make one after the other, each
// with its allocations and argument marshalling in between while the GPU waits.  The pair lists and the mask sort both
// start from the map and need nothing of each other; from a few hundred thousand voxels on the lists are enqueued on a
// second stream of the library's own (default priority, one per device, made on first use), which the caller's stream
// waits for before the call returns.
#include <mutex>

#include "cache_parts.h"
#include "fgx_common.h"
#include "grid_index.h"

namespace fgx {
namespace {

constexpr int kMaxCacheDevices = 64;
constexpr size_t kTwoStreamsMinRows = 393216;      // below, the second stream's events cost more than the overlap gives

hipStream_t g_side_stream[kMaxCacheDevices];
std::mutex g_side_mutex;

int side_stream(hipStream_t* out) {
    int dev = 0;
    FGX_CHECK_HIP(hipGetDevice(&dev));
    FGX_CHECK_ARG(dev >= 0 && dev < kMaxCacheDevices, "fgx_subm_cache_build: device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_side_mutex);
    if (g_side_stream[dev] == nullptr) FGX_CHECK_HIP(hipStreamCreateWithFlags(&g_side_stream[dev], hipStreamNonBlocking));
    *out = g_side_stream[dev];
    return FGX_OK;
}

struct CacheLayout {
    size_t map_ws, map_bytes, sort_ws, sort_bytes, pair_ws, pair_bytes, total;
};

CacheLayout cache_layout(size_t n, int key_bits, int Kw, int Kh, int V, int with_pairs) {
    CacheLayout L{};
    L.map_bytes = fgx_subm_neighbor_map_sorted_workspace_bytes(n, key_bits, Kw, Kh);
    L.sort_bytes = fgx_sort_workspace_bytes(n);
    L.pair_bytes = with_pairs ? fgx_pair_workspace_bytes(n, V) : 0;
    size_t off = 0;
    L.map_ws = off;
    off = align_up(off + L.map_bytes, 256);
    L.sort_ws = off;
    off = align_up(off + L.sort_bytes, 256);
    L.pair_ws = off;
    off = align_up(off + L.pair_bytes, 256);
    L.total = off;
    return L;
}

// The mask sort on `s` (none without sorted_idx) and, with_pairs, the pair lists (enqueued by `lists` on the stream it is given) -- beside it on the second
// stream for many rows, outside a capture (which would have to own that stream); `s` waits for both.
template <typename Lists>
int sort_beside_pairs(size_t n, int V, const int32_t* binary, int64_t* sorted_idx, void* sort_ws, size_t sort_bytes, bool with_pairs,
                      hipStream_t s, const char* who, Lists lists) {
    bool two_streams = with_pairs && sorted_idx != nullptr && n >= kTwoStreamsMinRows;
    if (two_streams) {
        hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
        FGX_CHECK_HIP(hipStreamIsCapturing(s, &capturing));
        two_streams = capturing == hipStreamCaptureStatusNone;
    }
    hipStream_t side = nullptr;
    hipEvent_t map_made = nullptr, lists_made = nullptr;
    int rc = FGX_OK;
    if (two_streams) {
        rc = side_stream(&side);
        if (rc != FGX_OK) return rc;
        FGX_CHECK_HIP(hipEventCreateWithFlags(&map_made, hipEventDisableTiming));
        hipError_t e = hipEventCreateWithFlags(&lists_made, hipEventDisableTiming);
        if (e == hipSuccess) e = hipEventRecord(map_made, s);
        if (e != hipSuccess) {
            (void)hipEventDestroy(map_made);
            if (lists_made) (void)hipEventDestroy(lists_made);
            return fail_hip(e, who);
        }
    }
    // the mask sort first: it is the longer of the two chains
    if (sorted_idx != nullptr) rc = fgx_sort_by_code(binary, n, V, sorted_idx, sort_ws, sort_bytes, (fgx_stream_t)s);
    if (rc == FGX_OK && with_pairs) {
        hipError_t e = two_streams ? hipStreamWaitEvent(side, map_made, 0) : hipSuccess;
        if (e != hipSuccess) rc = fail_hip(e, who);
        if (rc == FGX_OK) rc = lists(two_streams ? side : s);
        if (two_streams) {
            // whatever was enqueued on the second stream, the caller's stream waits for it: its buffers are the caller's
            e = hipEventRecord(lists_made, side);
            if (e == hipSuccess) e = hipStreamWaitEvent(s, lists_made, 0);
            if (e != hipSuccess && rc == FGX_OK) rc = fail_hip(e, who);
        }
    }
    if (map_made) (void)hipEventDestroy(map_made);
    if (lists_made) (void)hipEventDestroy(lists_made);
    return rc;
}

// what follows the map: [counts][offsets][totals] of the pair lists, the sort, a code array of the backward map
struct PostLayout {
    size_t counts, offsets, totals, sort_ws, sort_bytes, sort2_ws, sort2_bytes, codes, total;
};

PostLayout post_layout(size_t at, size_t n, int V, bool with_pairs, size_t n_bwd) {
    PostLayout L{};
    size_t off = align_up(at, 256);
    if (with_pairs) {
        L.counts = off;
        off = align_up(off + (size_t)cdiv(n, kPairSubRows) * V * 4, 256);
        L.offsets = off;
        off = align_up(off + (size_t)cdiv(n, kPairRows) * V * 4, 256);
        L.totals = off;
        off += 256;
    }
    L.sort_ws = off;
    L.sort_bytes = fgx_sort_workspace_bytes(n);
    off = align_up(off + L.sort_bytes, 256);
    if (n_bwd) {
        L.codes = off;
        off = align_up(off + n_bwd * 4, 256);
        L.sort2_ws = off;
        L.sort2_bytes = fgx_sort_workspace_bytes(n_bwd);
        off = align_up(off + L.sort2_bytes, 256);
    }
    L.total = off;
    return L;
}

}  // namespace
}  // namespace fgx

using namespace fgx;

extern "C" size_t fgx_subm_cache_workspace_bytes(size_t n, int key_bits, int Kw, int Kh, int Kd, int with_pairs) {
    if ((key_bits != 32 && key_bits != 64) || Kw < 1 || Kh < 1 || Kd < 1 || (long long)Kw * Kh * Kd > 32) return 0;
    if (fgx_subm_neighbor_map_sorted_workspace_bytes(n, key_bits, Kw, Kh) == 0) return 0;
    return cache_layout(n, key_bits, Kw, Kh, Kw * Kh * Kd, with_pairs).total;
}

extern "C" int fgx_subm_cache_build(const int32_t* coords, size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dw,
                                    int Dh, int Dd, int key_bits, int presorted, int with_pairs, void* workspace,
                                    size_t workspace_bytes, uint32_t* out_map, int32_t* gray, int32_t* binary,
                                    int64_t* sorted_idx, uint32_t* seg, uint32_t* sig_i, uint32_t* sig_o, fgx_stream_t stream) {
    FGX_CHECK_ARG(Kw > 0 && Kh > 0 && Kd > 0 && (long long)Kw * Kh * Kd <= 32,
                  "fgx_subm_cache_build: mask codes need a kernel volume <= 32, got (%d,%d,%d)", Kw, Kh, Kd);
    const int V = Kw * Kh * Kd;
    FGX_CHECK_ARG(!with_pairs || seg != nullptr, "fgx_subm_cache_build: null segment table");
    FGX_CHECK_ARG(n * (size_t)V < 0xFFFFFFFFull, "fgx_subm_cache_build: pair offsets must fit in 32 bits");
    hipStream_t s = (hipStream_t)stream;
    if (n == 0) return with_pairs ? fgx_pair_count(nullptr, 0, V, seg, nullptr, 0, stream) : FGX_OK;
    FGX_CHECK_ARG(key_bits == 32 || key_bits == 64, "fgx_subm_cache_build: key_bits must be 32 or 64, got %d", key_bits);
    FGX_CHECK_ARG(coords && workspace && out_map && gray && binary && sorted_idx, "fgx_subm_cache_build: null buffer");
    FGX_CHECK_ARG(!with_pairs || (sig_i && sig_o), "fgx_subm_cache_build: null pair list");
    FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0, "fgx_subm_cache_build: workspace must be 256-byte aligned");
    const CacheLayout L = cache_layout(n, key_bits, Kw, Kh, V, with_pairs);
    FGX_CHECK_ARG(L.map_bytes != 0, "fgx_subm_cache_build: kernel of %d x %d rows is too large for the sorted builder", Kw, Kh);
    FGX_CHECK_ARG(workspace_bytes >= L.total, "fgx_subm_cache_build: workspace of %zu bytes, need %zu", workspace_bytes, L.total);
    char* ws = (char*)workspace;

    int rc = fgx_subm_neighbor_map_sorted(coords, n, B, W, H, D, Kw, Kh, Kd, Dw, Dh, Dd, key_bits, presorted, ws + L.map_ws,
                                          L.map_bytes, out_map, gray, binary, stream);
    if (rc != FGX_OK) return rc;

    return sort_beside_pairs(n, V, binary, sorted_idx, ws + L.sort_ws, L.sort_bytes, with_pairs != 0, s, "fgx_subm_cache_build",
                             [&](hipStream_t on) {
                                 const int r = fgx_pair_count(gray, n, V, seg, ws + L.pair_ws, L.pair_bytes, (fgx_stream_t)on);
                                 return r != FGX_OK ? r : fgx_pair_fill(out_map, gray, n, V, ws + L.pair_ws, sig_i, sig_o, (fgx_stream_t)on);
                             });
}

extern "C" size_t fgx_subm_cache_grid_workspace_bytes(size_t n, int B, int W, int H, int D, int V, int with_pairs) {
    GridIndexLayout G;
    if (V < 1 || V > 32 || !grid_index_plan(n, B, W, H, D, &G)) return 0;
    return post_layout(G.total, n, V, with_pairs != 0, 0).total;
}

extern "C" int fgx_subm_cache_build_grid(const int32_t* coords, size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dw,
                                         int Dh, int Dd, int with_pairs, void* workspace, size_t workspace_bytes, uint32_t* out_map,
                                         int32_t* gray, int32_t* binary, int64_t* sorted_idx, uint32_t* seg, uint32_t* sig_i,
                                         uint32_t* sig_o, uint32_t* seg_host, uint32_t* walk, fgx_stream_t stream) {
    return fgx_subm_cache_build_grid_plan(coords, n, B, W, H, D, Kw, Kh, Kd, Dw, Dh, Dd, with_pairs, workspace, workspace_bytes, out_map, gray, binary,
                                          sorted_idx, seg, sig_i, sig_o, seg_host, walk, nullptr, stream);
}

extern "C" int fgx_subm_cache_plan_fits(size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dd) {
    GridIndexLayout G;
    return n > 0 && grid_index_plan(n, B, W, H, D, &G) && grid_plan_fits(G, Kw, Kh, Kd, Dd) ? 1 : 0;
}

extern "C" int fgx_subm_cache_build_grid_plan(const int32_t* coords, size_t n, int B, int W, int H, int D, int Kw, int Kh, int Kd, int Dw,
                                              int Dh, int Dd, int with_pairs, void* workspace, size_t workspace_bytes, uint32_t* out_map,
                                              int32_t* gray, int32_t* binary, int64_t* sorted_idx, uint32_t* seg, uint32_t* sig_i,
                                              uint32_t* sig_o, uint32_t* seg_host, uint32_t* walk, void* plan, fgx_stream_t stream) {
    const char* who = "fgx_subm_cache_build_grid";
    FGX_CHECK_ARG(Kw > 0 && Kh > 0 && Kd > 0 && (long long)Kw * Kh * Kd <= 32 && (Kw & 1) && (Kh & 1) && (Kd & 1),
                  "%s: mask codes need odd kernel sizes and a volume <= 32, got (%d,%d,%d)", who, Kw, Kh, Kd);
    const int V = Kw * Kh * Kd;
    FGX_CHECK_ARG(!with_pairs || seg != nullptr, "%s: null segment table", who);
    FGX_CHECK_ARG(n * (size_t)V < 0xFFFFFFFFull, "%s: pair offsets must fit in 32 bits", who);
    hipStream_t s = (hipStream_t)stream;
    if (n == 0) return with_pairs ? fgx_pair_count(nullptr, 0, V, seg, nullptr, 0, stream) : FGX_OK;
    GridIndexLayout G;
    FGX_CHECK_ARG(grid_index_plan(n, B, W, H, D, &G), "%s: no index over a grid of %d x %d x %d x %d cells and %zu voxels", who, B, W, H, D, n);
    const PostLayout P = post_layout(G.total, n, V, with_pairs != 0, 0);
    FGX_CHECK_ARG(coords && workspace && out_map && gray && binary, "%s: null buffer", who);
    FGX_CHECK_ARG(!with_pairs || (sig_i && sig_o), "%s: null pair list", who);
    FGX_CHECK_ARG((((uintptr_t)coords & 15) | ((uintptr_t)workspace & 255)) == 0, "%s: coords must be 16-byte, workspace 256-byte aligned", who);
    FGX_CHECK_ARG(workspace_bytes >= P.total, "%s: workspace of %zu bytes, need %zu", who, workspace_bytes, P.total);
    FGX_CHECK_ARG(walk == nullptr || (!G.dense && ((uintptr_t)walk & 15) == 0), "%s: an index without a walk, or a misaligned one", who);
    FGX_CHECK_ARG(plan == nullptr || (walk != nullptr && grid_plan_fits(G, Kw, Kh, Kd, Dd) && ((uintptr_t)plan & 15) == 0),
                  "%s: no plan of a %d x %d x %d kernel without a walk, or a misaligned one", who, Kw, Kh, Kd);
    char* ws = (char*)workspace;
    PhaseEnd phases{s};
    uint32_t* counts = with_pairs ? (uint32_t*)(ws + P.counts) : nullptr;
    bool counted = false;
    int rc = subm_map_grid(coords, n, B, W, H, D, Kw, Kh, Kd, Dw, Dh, Dd, G, ws, walk, plan, out_map, gray, binary, counts, &counted, s);
    if (rc != FGX_OK) return rc;
    return sort_beside_pairs(n, V, binary, sorted_idx, ws + P.sort_ws, P.sort_bytes, with_pairs != 0, s, who, [&](hipStream_t on) {
        int r = counted ? FGX_OK : pair_counts(gray, n, V, counts, on);
        if (r != FGX_OK) return r;
        return pair_lists_from_counts(out_map, gray, n, V, counts, cdiv(n, counted ? kPairSubRows : kPairRows), counted,
                                      (uint32_t*)(ws + P.offsets), (uint32_t*)(ws + P.totals), seg, seg_host, sig_i, sig_o, on);
    });
}

extern "C" size_t fgx_cache_post_workspace_bytes(size_t n, int V, int with_pairs) {
    return V >= 1 && V <= 32 ? post_layout(0, n, V, with_pairs != 0, 0).total : 0;
}

extern "C" int fgx_cache_post(const uint32_t* map, const int32_t* gray, const int32_t* binary, size_t n, int V, int with_pairs, void* workspace,
                              size_t workspace_bytes, int64_t* sorted_idx, uint32_t* seg, uint32_t* sig_i, uint32_t* sig_o, uint32_t* seg_host,
                              fgx_stream_t stream) {
    const char* who = "fgx_cache_post";
    FGX_CHECK_ARG(V >= 1 && V <= 32 && n > 0 && n * (size_t)V < 0xFFFFFFFFull, "%s: %zu rows of %d offsets out of range", who, n, V);
    const PostLayout P = post_layout(0, n, V, with_pairs != 0, 0);
    FGX_CHECK_ARG(map && gray && binary && workspace && (!with_pairs || (seg && sig_i && sig_o)), "%s: null buffer", who);
    FGX_CHECK_ARG(((uintptr_t)workspace & 255) == 0 && workspace_bytes >= P.total, "%s: workspace of %zu bytes, need %zu, 256-byte aligned", who,
                  workspace_bytes, P.total);
    char* ws = (char*)workspace;
    hipStream_t s = (hipStream_t)stream;
    PhaseEnd phases{s};
    return sort_beside_pairs(n, V, binary, sorted_idx, ws + P.sort_ws, P.sort_bytes, with_pairs != 0, s, who, [&](hipStream_t on) {
        const int r = pair_counts(gray, n, V, (uint32_t*)(ws + P.counts), on);
        return r != FGX_OK ? r : pair_lists_from_counts(map, gray, n, V, (uint32_t*)(ws + P.counts), cdiv(n, kPairRows), false, (uint32_t*)(ws + P.offsets),
                                                        (uint32_t*)(ws + P.totals), seg, seg_host, sig_i, sig_o, on);
    });
}

extern "C" size_t fgx_spconv_cache_grid_workspace_bytes(size_t n_in, size_t n_out, int B, int W, int H, int D, int Wo, int Ho, int Do, int V,
                                                        int with_bwd, int with_bwd_order) {
    ConvMapsLayout M;
    if (V < 1 || V > 32 || !conv_maps_plan(n_in, n_out, B, W, H, D, Wo, Ho, Do, with_bwd != 0, &M)) return 0;
    return post_layout(M.total, n_out, V, with_bwd != 0, with_bwd_order ? n_in : 0).total;
}

extern "C" int fgx_spconv_cache_build_grid(const int32_t* in_coords, size_t n_in, const int32_t* out_coords, size_t n_out, int B, int W, int H,
                                           int D, int Kw, int Kh, int Kd, int Sw, int Sh, int Sd, int Pw, int Ph, int Pd, int Dw, int Dh,
                                           int Dd, void* workspace, size_t workspace_bytes, uint32_t* map_fwd, int32_t* gray,
                                           int32_t* binary, int64_t* sorted_idx, uint32_t* map_bwd, uint32_t* seg, uint32_t* sig_i,
                                           uint32_t* sig_o, uint32_t* seg_host, int32_t* gray_bwd, int64_t* sorted_idx_bwd, fgx_stream_t stream) {
    const char* who = "fgx_spconv_cache_build_grid";
    int Wo, Ho, Do;
    int rc = fgx_spconv_out_dims(W, H, D, Kw, Kh, Kd, Sw, Sh, Sd, Pw, Ph, Pd, Dw, Dh, Dd, &Wo, &Ho, &Do);
    if (rc != FGX_OK) return rc;
    FGX_CHECK_ARG((long long)Kw * Kh * Kd <= 32, "%s: mask codes need a kernel volume <= 32, got (%d,%d,%d)", who, Kw, Kh, Kd);
    const int V = Kw * Kh * Kd;
    const bool bwd = map_bwd != nullptr, order_bwd = sorted_idx_bwd != nullptr;
    FGX_CHECK_ARG(n_in > 0 && n_out > 0 && n_out * (size_t)V < 0xFFFFFFFFull, "%s: empty or too many voxels", who);
    ConvMapsLayout M;
    FGX_CHECK_ARG(conv_maps_plan(n_in, n_out, B, W, H, D, Wo, Ho, Do, bwd, &M), "%s: no index over a grid of this size", who);
    const PostLayout P = post_layout(M.total, n_out, V, bwd, order_bwd ? n_in : 0);
    FGX_CHECK_ARG(in_coords && out_coords && workspace && map_fwd && gray && binary && sorted_idx, "%s: null buffer", who);
    FGX_CHECK_ARG(!bwd || (seg && sig_i && sig_o), "%s: a backward map comes with pair lists", who);
    FGX_CHECK_ARG(order_bwd == (gray_bwd != nullptr) && (bwd || !order_bwd), "%s: codes and order of the backward map go together", who);
    FGX_CHECK_ARG((((uintptr_t)in_coords & 15) | ((uintptr_t)out_coords & 15) | ((uintptr_t)workspace & 255)) == 0,
                  "%s: coords must be 16-byte, workspace 256-byte aligned", who);
    FGX_CHECK_ARG(workspace_bytes >= P.total, "%s: workspace of %zu bytes, need %zu", who, workspace_bytes, P.total);
    char* ws = (char*)workspace;
    hipStream_t s = (hipStream_t)stream;
    PhaseEnd phases{s};
    const int k[12] = {Kw, Kh, Kd, Sw, Sh, Sd, Pw, Ph, Pd, Dw, Dh, Dd};
    uint32_t* counts = bwd ? (uint32_t*)(ws + P.counts) : nullptr;
    int32_t* binary_bwd = order_bwd ? (int32_t*)(ws + P.codes) : nullptr;
    rc = conv_maps_grid(in_coords, n_in, out_coords, n_out, B, W, H, D, Wo, Ho, Do, k, M, ws, map_fwd, map_bwd, gray, binary, counts, gray_bwd,
                        binary_bwd, s);
    if (rc != FGX_OK) return rc;
    rc = sort_beside_pairs(n_out, V, binary, sorted_idx, ws + P.sort_ws, P.sort_bytes, bwd, s, who, [&](hipStream_t on) {
        return pair_lists_from_counts(map_fwd, gray, n_out, V, counts, cdiv(n_out, kPairSubRows), true, (uint32_t*)(ws + P.offsets),
                                      (uint32_t*)(ws + P.totals), seg, seg_host, sig_i, sig_o, on);
    });
    if (rc != FGX_OK || !order_bwd) return rc;
    return fgx_sort_by_code(binary_bwd, n_in, V, sorted_idx_bwd, ws + P.sort2_ws, P.sort2_bytes, stream);
}
