// Weight gradient for narrow layers (16-bit types, up to 32 channels on both sides) with the gathered rows resident in
// LDS: the counterpart of conv_gemm_narrow.hip, on the same plan (narrow_plan.h).
//
//   grad_weight[co][v][ci] = sum over rows r with a neighbor at offset v of grad_out[r][co] * feats[source(r, v)][ci]
//
// The block-major kernel fetches two 64-byte rows per (row, offset) pair: 4.4 GB cross the L2 for the 0.65 GB that
// configuration 4 (2.67 M voxels, 32 channels) holds, at the fabric's read limit.  Here a chunk of 128 rows that are
// consecutive on a Z-order curve brings its own grad_out rows (8 KiB) and its ~220 distinct source rows into LDS once;
// the voxels are the K dimension, and the transposing LDS read (ds_read_b64_tr_b16), which takes an address per lane,
// does the gather: lane s of a 16-lane group names 4 channels of the row that the plan's table gives for (chunk row,
// offset) and receives 4 rows' values of one channel.  A missing neighbor is the row of zeros.
//
// Workgroup of kernel volumes other than 27: 4 multiplying wavefronts + 4 loading wavefronts, two LDS buffers, one barrier per chunk (as in the
// forward kernel).  Multiplier w owns the offsets 8 w ... 8 w + 7 (their 32 x 32 accumulators stay in registers over all the
// chunks of the workgroup; offsets from V on multiply zeros).  It walks the chunk's 128 rows in eight k-steps of 16; the
// grad_out fragment of a k-step is read once for the eight offsets.  3 x 3 x 3 kernels: narrow_wgrad27_kernel.  At the end every workgroup writes its partial
// products, and a second kernel adds them in workgroup order (fixed order: same bits on every run).
// An infinity or NaN in grad_out times the row of zeros is NaN where the sum over the pairs has no term: a workgroup whose sums are not
// all finite goes over its chunks again and adds such rows of grad_out pair by pair, until every sum is NaN (wgrad_device.h).  2.67 M
// voxels, 32 channels: all finite 0.165 ms, one value infinite 0.58, a value in every thousandth row 0.61, every value 0.51 (with four multipliers 0.236,
// 0.65, 0.67, 0.80; most where no sum ends as NaN, 6.1).
// The bias gradient comes for nothing: the offsets from V on are multiplied for no one, and the last of them by ones.  Column sums of
// their own read grad_out once more (2.67 M voxels, 32 channels: 29 us a layer and 4 for their reduction; a training pass of two
// layers 2.084 -> 2.022 ms).
// A plan with an overflowing chunk (more distinct sources than slots) is not for this kernel: the caller looks at the
// plan's header and takes the block-major kernel then.
#include "wgrad_device.h"
#include "narrow_walk.h"

namespace fgx {
namespace {

constexpr int kNwMult = 4, kNwLoad = 4, kNwThreads = 64 * (kNwMult + kNwLoad);
constexpr int kNwTaps = 8;                                                       // offsets per multiplier
constexpr int kNwGoutBytes = kNarrowRows * 64;                                   // the chunk's grad_out rows
constexpr int kNwBufferBytes = kNarrowRowBufPad + kNwGoutBytes + kNarrowTableBytes;
constexpr size_t kNwLdsBytes = 2 * (size_t)kNwBufferBytes + 16;                  // ... and the word that asks for a second pass
constexpr int kNwSrcGroups = kNarrowSlots / 16 / kNwLoad;                        // 7 wave-wide row loads per loader
constexpr int kNwOutGroups = kNarrowRows / 16 / kNwLoad;                         // 2
constexpr int kNwIds = kNwSrcGroups + kNwOutGroups;

// Kernel volumes other than 27.
template <typename Tag>
__global__ void __launch_bounds__(kNwThreads)
narrow_wgrad_kernel(const typename Tag::type* __restrict__ gout, const typename Tag::type* __restrict__ feats,
                    const unsigned char* __restrict__ plan, uint32_t chunks, uint32_t plan_bytes, uint32_t gout_bytes,
                    uint32_t feats_bytes, int V, int Ci, int Co, float* __restrict__ partial, float* __restrict__ bias_partial) {
    using T = typename Tag::type;
    using T4 = T __attribute__((ext_vector_type(4)));
    constexpr int TAPS = kNwTaps;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    volatile uint32_t& again = *reinterpret_cast<volatile uint32_t*>(lds + 2 * kNwBufferBytes);       // some sum is not finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const bool loader = wave >= kNwMult;
    if (tid == 0) again = 0u;
    const int src_row_bytes = Ci * 2, out_row_bytes = Co * 2;

    // chunks of this workgroup: XCD x owns the x-th eighth, its workgroups interleave
    const unsigned G = gridDim.x;
    const unsigned xcd = blockIdx.x % kXcds, slot_in_xcd = blockIdx.x / kXcds, per_round = G / kXcds;
    const unsigned per_xcd = (chunks + kXcds - 1) / kXcds;
    const unsigned range_lo = xcd * per_xcd, range_hi = (xcd + 1) * per_xcd < chunks ? (xcd + 1) * per_xcd : chunks;
    const unsigned first = range_lo + slot_in_xcd;

    // the slot of zeros of both buffers
    if (tid < 8) {
        const u32x4 zero = {0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4*>(lds + (size_t)(tid >> 2) * kNwBufferBytes + kNarrowSlots * 64 + (tid & 3) * 16) = zero;
    }

    const rsrc_t feats_rs = make_rsrc(feats, feats_bytes);
    const rsrc_t gout_rs = make_rsrc(gout, gout_bytes);
    const rsrc_t plan_rs = make_rsrc(plan, plan_bytes);

    // ---- loaders: per chunk, wavefront lw loads the source-row groups (j * 4 + lw), the grad_out-row groups likewise,
    // and every fourth KiB of the table; the row numbers of the next chunk but one are fetched while the loads fly ----
    const int lw = loader ? wave - kNwMult : 0;
    uint32_t ids[kNwIds];
    auto fetch_ids = [&](unsigned chunk) {
        const uint32_t base = (uint32_t)kNarrowHeader + chunk * (uint32_t)kNarrowPlanStride + (uint32_t)kNarrowTableBytes;
#pragma unroll
        for (int j = 0; j < kNwSrcGroups; ++j)
            ids[j] = __builtin_amdgcn_raw_buffer_load_b32(plan_rs, base + (uint32_t)((j * kNwLoad + lw) * 16 + (lane >> 2)) * 4u, 0, 0);
#pragma unroll
        for (int j = 0; j < kNwOutGroups; ++j)
            ids[kNwSrcGroups + j] = __builtin_amdgcn_raw_buffer_load_b32(
                plan_rs, base + (uint32_t)kNarrowSlots * 4u + (uint32_t)((j * kNwLoad + lw) * 16 + (lane >> 2)) * 4u, 0, 0);
    };
    auto enqueue = [&](unsigned chunk, int b) {
        unsigned char* buf = lds + (size_t)b * kNwBufferBytes;
#pragma unroll
        for (int j = 0; j < kNwSrcGroups; ++j) {
            const int group = j * kNwLoad + lw;
            const uint32_t s = (uint32_t)(group * 16 + (lane >> 2));
            const uint32_t piece = (uint32_t)(lane & 3) ^ narrow_piece_key(s);
            const bool live = ids[j] != FGX_EMPTY32 && (int)(piece * 16) < src_row_bytes;
            const uint32_t vo = live ? ids[j] * (uint32_t)src_row_bytes + piece * 16u : kNarrowOob;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(feats_rs, FGX_LDS_PTR(buf + group * 1024), 16, vo, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < kNwOutGroups; ++j) {
            const int group = j * kNwLoad + lw;
            const uint32_t s = (uint32_t)(group * 16 + (lane >> 2));
            const uint32_t piece = (uint32_t)(lane & 3) ^ narrow_piece_key(s);
            const uint32_t id = ids[kNwSrcGroups + j];
            const bool live = id != FGX_EMPTY32 && (int)(piece * 16) < out_row_bytes;
            const uint32_t vo = live ? id * (uint32_t)out_row_bytes + piece * 16u : kNarrowOob;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(gout_rs, FGX_LDS_PTR(buf + kNarrowRowBufPad + group * 1024), 16, vo, 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < kNarrowTableBytes / 1024 / kNwLoad; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(
                plan_rs, FGX_LDS_PTR(buf + kNarrowRowBufPad + kNwGoutBytes + (j * kNwLoad + lw) * 1024), 16,
                (uint32_t)kNarrowHeader + chunk * (uint32_t)kNarrowPlanStride + (uint32_t)((j * kNwLoad + lw) * 1024 + lane * 16), 0, 0, 0);
    };

    // ---- multipliers ----
    // Transposing read: in a 16-lane group, lane s supplies the address of 4 adjacent channels of row (s / 4) of a run of
    // four rows and receives those four rows' values of channel (group base + s).  Lanes 0-15 / 16-31 cover channels
    // 0-15 / 16-31, the two wave halves take rows [0, 8) / [8, 16) of a k-step, a second read the rows four further on.
    const int mw = loader ? 0 : wave;
    const int s16 = lane & 15, mb = (lane >> 4) & 1, g = lane >> 5;
    const int q = s16 >> 2;                                                      // row of the run of four
    const int chan_byte = mb * 32 + (s16 & 3) * 8;                               // the lane's 4 channels inside a row
    const uint32_t cpiece = (uint32_t)(chan_byte >> 4), cw = (uint32_t)(chan_byte & 15);
    // The two roles run loops of their own (with the same number of barriers): the multipliers' accumulators then take
    // no registers from the loaders and the other way round.
    if (loader) {
        for (int pass = 0; pass < 2; ++pass) {
            if (first < range_hi) {
                fetch_ids(first);
                enqueue(first, 0);
                if (first + per_round < range_hi) fetch_ids(first + per_round);
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
                int b = 0;
                for (unsigned chunk = first; chunk < range_hi; chunk += per_round, b ^= 1) {
                    const unsigned next = chunk + per_round;
                    const bool enqueues = next < range_hi, fetches = next + per_round < range_hi;
                    if (enqueues) {
                        enqueue(next, b ^ 1);
                        if (fetches) fetch_ids(next + per_round);
                    }
                    if (fetches) wait_vmcnt<kNwIds>();
                    else wait_vmcnt<0>();
                    __syncthreads();
                }
            }
            if (pass == 0) __syncthreads();
            if (again == 0u) break;
        }
        return;
    }
    f32x16 acc[TAPS];
    // a row's entries for the wavefront's offsets, 16 bytes
    auto entries_of = [&](const unsigned char* table, int r) __attribute__((always_inline)) -> u32x4 {
        return *reinterpret_cast<const u32x4*>((const uint16_t*)(table + r * (kNarrowTableStride * 2)) + mw * 8);
    };
    auto offset_of = [&](int t) -> int { return mw * kNwTaps + t; };
    // the last offset of the last multiplier, past every V: ones in place of whatever its table entry names
    static_assert(kNarrowMaxV < kNwMult * kNwTaps, "an offset is free for the column sums");
    const uint32_t bias_bits = bias_partial != nullptr && mw == kNwMult - 1 ? (std::is_same<Tag, F16>::value ? 0x3C003C00u : 0x3F803F80u) : 0u;
    auto run = [&](auto apart_rows) __attribute__((always_inline)) {
        constexpr bool APART = decltype(apart_rows)::value;
#pragma unroll
        for (int t = 0; t < TAPS; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;
        if (first < range_hi) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
            int b = 0;
            bool done = false;                                                   // (second pass) every sum is NaN
            for (unsigned chunk = first; chunk < range_hi; chunk += per_round, b ^= 1) {
                const unsigned char* buf = lds + (size_t)b * kNwBufferBytes;
                const unsigned char* gbuf = buf + kNarrowRowBufPad;
                const unsigned char* table = gbuf + kNwGoutBytes;
                // grad_out rows sit in the slots of their chunk row numbers: row r = kk * 16 + g * 8 + q (+ 4) has the
                // piece key (g * 2 (+ 1)) & 3, whatever kk
                const uint32_t g_lo = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)gbuf +
                                      (uint32_t)((g * 8 + q) * 64) + ((cpiece ^ (uint32_t)((g * 2) & 3)) << 4) + cw;
                const uint32_t g_hi = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)gbuf +
                                      (uint32_t)((g * 8 + q + 4) * 64) + ((cpiece ^ (uint32_t)((g * 2 + 1) & 3)) << 4) + cw;
                const uint32_t row_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)buf + cw;
#pragma unroll 1
                for (int kk = 0; kk < kNarrowRows / 16 && !done; ++kk) {
                    const int r0 = kk * 16 + g * 8 + q;
                    const u32x4 e_lo = entries_of(table, r0), e_hi = entries_of(table, r0 + 4);
                    i16x4 gfr[2], ffr[2 * TAPS];                                 // grad_out (lo, hi); the offsets (lo, hi)
                    gfr[0] = lds_read_tr16_at<0>(g_lo + (uint32_t)(kk * 16 * 64));
                    gfr[1] = lds_read_tr16_at<0>(g_hi + (uint32_t)(kk * 16 * 64));
                    auto entry = [](const u32x4& e, int t) -> uint32_t { return (t & 1) ? e[t >> 1] >> 16 : e[t >> 1] & 0xFFFFu; };
                    auto at = [&](const u32x4& e, int t) -> uint32_t { return row_base + (entry(e, t) ^ (cpiece << 4)); };
#pragma unroll
                    for (int t = 0; t < 6; ++t) {                                // (at most 15 reads are counted in flight)
                        ffr[t * 2] = lds_read_tr16_at<0>(at(e_lo, t));
                        ffr[t * 2 + 1] = lds_read_tr16_at<0>(at(e_hi, t));
                    }
                    // every fragment register is tied to the wait: the compiler must not touch one before it
                    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(gfr[0]), "+v"(gfr[1]));
                    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(ffr[0]), "+v"(ffr[1]), "+v"(ffr[2]), "+v"(ffr[3]));
                    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(ffr[4]), "+v"(ffr[5]), "+v"(ffr[6]), "+v"(ffr[7]));
                    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(ffr[8]), "+v"(ffr[9]), "+v"(ffr[10]), "+v"(ffr[11]));
#pragma unroll
                    for (int t = 6; t < TAPS; ++t) {
                        ffr[t * 2] = lds_read_tr16_at<0>(at(e_lo, t));
                        ffr[t * 2 + 1] = lds_read_tr16_at<0>(at(e_hi, t));
                    }
                    i16x8 gf = __builtin_shufflevector(gfr[0], gfr[1], 0, 1, 2, 3, 4, 5, 6, 7);
                    uint32_t apart = 0u;
                    if constexpr (APART) {
#pragma unroll
                        for (int t = 12; t < 2 * TAPS; ++t) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(ffr[t]));
                        apart = nonfinite_rows<Tag>(gf);
                        if (apart) drop_rows(gf, apart, g);
                    }
#pragma unroll
                    for (int t = 0; t < 6; ++t) {
                        i16x8 ff = __builtin_shufflevector(ffr[t * 2], ffr[t * 2 + 1], 0, 1, 2, 3, 4, 5, 6, 7);
                        if (APART && apart) drop_rows(ff, apart, g);
                        mma16<Tag>(acc[t], gf, ff);
                    }
#pragma unroll
                    for (int t = 12; t < 2 * TAPS; ++t) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(ffr[t]));
#pragma unroll
                    for (int t = 6; t < TAPS; ++t) {
                        i16x8 ff = __builtin_shufflevector(ffr[t * 2], ffr[t * 2 + 1], 0, 1, 2, 3, 4, 5, 6, 7);
                        if (!APART && t == TAPS - 1 && bias_bits != 0u) ff = __builtin_bit_cast(i16x8, u32x4{bias_bits, bias_bits, bias_bits, bias_bits});
                        if (APART && apart) drop_rows(ff, apart, g);
                        mma16<Tag>(acc[t], gf, ff);
                    }
                    while (APART && apart) {
                        const int r = kk * 16 + __ffs((int)apart) - 1;
                        apart &= apart - 1u;
                        T4 gv[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            gv[e] = *reinterpret_cast<const T4*>(gbuf + r * 64 + (((uint32_t)e ^ narrow_piece_key((uint32_t)r)) << 4) + g * 8);
                        const u32x4 entries = entries_of(table, r);
                        T x[TAPS];                                            // (all reads in flight together; a missing neighbor's: zeros)
#pragma unroll
                        for (int t = 0; t < TAPS; ++t)
                            x[t] = *reinterpret_cast<const T*>(buf + (entry(entries, t) ^ ((uint32_t)((lane & 31) >> 3) << 4)) + (lane & 7) * 2);
#pragma unroll
                        for (int t = 0; t < TAPS; ++t) {
                            if (__builtin_amdgcn_readfirstlane((int)entry(entries, t)) >> 6 == (int)kNarrowZeroSlot) continue;
#pragma unroll
                            for (int e = 0; e < 16; ++e) acc[t][e] += (float)gv[e >> 2][e & 3] * (float)x[t];
                        }
                    }
                }
                if constexpr (APART) {
                    bool nan = true;
#pragma unroll
                    for (int t = 0; t < TAPS; ++t) nan = nan && (offset_of(t) >= V || all_nan(acc[t], lane, 0, Co, 0, Ci));
                    done = __all(nan);
                }
                __builtin_amdgcn_s_waitcnt(0);
                __syncthreads();
            }
        }
    };
    run(std::false_type{});
    // (whatever the second pass does: a column's sum has a term for every row)
    if (bias_bits != 0u && (lane & 31) == 0)
#pragma unroll
        for (int e = 0; e < 16; ++e) bias_partial[blockIdx.x * 32 + (e >> 2) * 8 + g * 4 + (e & 3)] = acc[TAPS - 1][e];
    bool finite = true;
#pragma unroll
    for (int t = 0; t < TAPS; ++t) finite = finite && (offset_of(t) >= V || all_finite(acc[t]));
    if (__any(!finite) && lane == 0) again = 1u;
    __syncthreads();                                                             // (the loaders' after their first pass)
    if (again != 0u) run(std::true_type{});
    // partial[workgroup][v][co][ci] (32 x 32 per offset): accumulator element e of lane (l32, g) is co = (e >> 2) * 8 +
    // g * 4 + (e & 3), ci = l32
    {
        const int l32 = lane & 31;
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
            const int v = offset_of(t);
            if (v < V) {
                float* dst = partial + ((size_t)blockIdx.x * V + v) * 1024;
#pragma unroll
                for (int e = 0; e < 16; ++e) dst[((e >> 2) * 8 + g * 4 + (e & 3)) * 32 + l32] = acc[t][e];
            }
        }
    }
}

// 3 x 3 x 3 kernels: seven multipliers of four offsets, the last one with three and the column sums, and four loaders (narrow_walk.h).  Four multipliers of
// seven, one per SIMD, waited for every k-step's reads before its products: 2 667 120 voxels, 32 channels 0.207 ms -> 0.168 (in random order
// 0.212 -> 0.182), 667 763 voxels, 16 channels 60 -> 46 us, 166 977 voxels, 32 channels 27.7 -> 24.3.  Eight multipliers of seven offsets, four for either
// half of a chunk's rows, 0.180, and 32 us for the last.  The memory's share is 0.108 ms (561 MB, 219 of them the plan).
constexpr int kNw27Mult = 7, kNw27Taps = 4, kNw27Threads = 64 * (kNw27Mult + kWalkLoad);
constexpr size_t kNw27LdsBytes = (size_t)kWalkBuffers * kNwBufferBytes + (size_t)kWalkMetas * kWalkMetaBytes + 16;
static_assert(kNw27LdsBytes <= 160 * 1024 && kNw27Mult * kNw27Taps == kNarrowCubeV + 1, "LDS; a place for the column sums");

template <typename Tag>
__global__ void __launch_bounds__(kNw27Threads)
narrow_wgrad27_kernel(const typename Tag::type* __restrict__ gout, const typename Tag::type* __restrict__ feats,
                      const unsigned char* __restrict__ plan, uint32_t chunks, uint32_t plan_bytes, uint32_t gout_bytes,
                      uint32_t feats_bytes, int Ci, int Co, float* __restrict__ partial, float* __restrict__ bias_partial) {
    using T = typename Tag::type;
    using T4 = T __attribute__((ext_vector_type(4)));
    constexpr int V = kNarrowCubeV, TAPS = kNw27Taps, STEPS = kNarrowRows / 16;
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
    unsigned char* meta = lds + kWalkBuffers * kNwBufferBytes;
    volatile uint32_t& again = *reinterpret_cast<volatile uint32_t*>(meta + kWalkMetas * kWalkMetaBytes);       // some sum is not finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (tid == 0) again = 0u;
    const NarrowWalk walk(chunks, kXcds);
    if (tid < 4 * kWalkBuffers) {                                                // the rows of zeros
        const u32x4 zero = {0u, 0u, 0u, 0u};
        *reinterpret_cast<u32x4*>(lds + (size_t)(tid >> 2) * kNwBufferBytes + kNarrowSlots * 64 + (tid & 3) * 16) = zero;
    }
    const rsrc_t feats_rs = make_rsrc(feats, feats_bytes), gout_rs = make_rsrc(gout, gout_bytes), plan_rs = make_rsrc(plan, plan_bytes);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                           // (the zeros and the word: met by the first barrier)

    if (wave >= kNw27Mult) {
        for (int pass = 0; pass < 2; ++pass) {
            if (walk.count > 0)
                narrow_load_walk<true, false>(walk, wave - kNw27Mult, lane, feats_rs, Ci * 2, gout_rs, Co * 2, plan_rs, lds, kNwBufferBytes,
                                              kNarrowRowBufPad + kNwGoutBytes, meta);
            if (pass == 0) __syncthreads();
            if (again == 0u) break;
        }
        return;
    }

    // (the lanes' part in a transposing read: narrow_wgrad_kernel)
    const int s16 = lane & 15, mb = (lane >> 4) & 1, g = lane >> 5, q = s16 >> 2;
    const int chan_byte = mb * 32 + (s16 & 3) * 8;
    const uint32_t cpiece = (uint32_t)(chan_byte >> 4), cw = (uint32_t)(chan_byte & 15);
    using Entries = uint32_t __attribute__((ext_vector_type(2)));                // of the wavefront's four offsets
    auto entries_of = [&](const unsigned char* table, int r) __attribute__((always_inline)) -> Entries {
        return *reinterpret_cast<const Entries*>(table + r * (kNarrowTableStride * 2) + wave * (TAPS * 2));
    };
    auto entry = [](const Entries& e, int t) -> uint32_t { return (t & 1) ? e[t >> 1] >> 16 : e[t >> 1] & 0xFFFFu; };
    const bool sums = bias_partial != nullptr && wave == kNw27Mult - 1;          // the last place: ones instead of what its table entry names
    const uint32_t ones = std::is_same<Tag, F16>::value ? 0x3C003C00u : 0x3F803F80u;
    f32x16 acc[TAPS];
#pragma unroll
    for (int t = 0; t < TAPS; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;

    // A k-step's reads in two groups, grad_out and two offsets, and the other two: while one is multiplied the next is on its way.
    auto lds_at = [](const unsigned char* p) { return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p; };
    const uint32_t g_lo = (uint32_t)((g * 8 + q) * 64) + ((cpiece ^ (uint32_t)((g * 2) & 3)) << 4) + cw;         // (row kk * 16 + g * 8 + q: piece key g * 2)
    const uint32_t g_hi = (uint32_t)((g * 8 + q + 4) * 64) + ((cpiece ^ (uint32_t)((g * 2 + 1) & 3)) << 4) + cw;
    if (walk.count > 0) {
        walk_barrier();
        walk_barrier();
        for (unsigned i = 0; i < walk.count; ++i) {
            const unsigned char* buf = lds + (i % kWalkBuffers) * kNwBufferBytes;
            const unsigned char* table = buf + kNarrowRowBufPad + kNwGoutBytes;
            const uint32_t g_at = lds_at(buf + kNarrowRowBufPad), row_at = lds_at(buf) + cw;
            Entries lo[STEPS], hi[STEPS];
#pragma unroll
            for (int kk = 0; kk < STEPS; ++kk) {
                lo[kk] = entries_of(table, kk * 16 + g * 8 + q);
                hi[kk] = entries_of(table, kk * 16 + g * 8 + q + 4);
            }
            i16x4 gf[2][2], f[2][4];
            auto issue = [&](int kk, int half) __attribute__((always_inline)) {
                if (half == 0) {
                    gf[kk & 1][0] = lds_read_tr16_at<0>(g_at + g_lo + (uint32_t)(kk * 16 * 64));
                    gf[kk & 1][1] = lds_read_tr16_at<0>(g_at + g_hi + (uint32_t)(kk * 16 * 64));
                }
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    f[half][2 * t] = lds_read_tr16_at<0>(row_at + (entry(lo[kk], half * 2 + t) ^ (cpiece << 4)));
                    f[half][2 * t + 1] = lds_read_tr16_at<0>(row_at + (entry(hi[kk], half * 2 + t) ^ (cpiece << 4)));
                }
            };
            issue(0, 0);
            issue(0, 1);
#pragma unroll
            for (int kk = 0; kk < STEPS; ++kk) {
                lds_wait_but<4>(f[0]);                                           // (everything but the other group)
                asm volatile("" : "+v"(gf[kk & 1][0]), "+v"(gf[kk & 1][1]));
                const i16x8 gg = __builtin_shufflevector(gf[kk & 1][0], gf[kk & 1][1], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                for (int t = 0; t < 2; ++t) mma16<Tag>(acc[t], gg, __builtin_shufflevector(f[0][2 * t], f[0][2 * t + 1], 0, 1, 2, 3, 4, 5, 6, 7));
                if (kk + 1 < STEPS) {
                    issue(kk + 1, 0);
                    lds_wait_but<6>(f[1]);
                } else {
                    lds_wait_but<0>(f[1]);
                }
                i16x8 last = __builtin_shufflevector(f[1][2], f[1][3], 0, 1, 2, 3, 4, 5, 6, 7);
                if (sums) last = __builtin_bit_cast(i16x8, u32x4{ones, ones, ones, ones});
                mma16<Tag>(acc[2], gg, __builtin_shufflevector(f[1][0], f[1][1], 0, 1, 2, 3, 4, 5, 6, 7));
                mma16<Tag>(acc[3], gg, last);
                if (kk + 1 < STEPS) issue(kk + 1, 1);
            }
            walk_barrier();
        }
    }
    // (whatever the second pass does: a column's sum has a term for every row)
    if (sums && (lane & 31) == 0)
#pragma unroll
        for (int e = 0; e < 16; ++e) bias_partial[blockIdx.x * 32 + (e >> 2) * 8 + g * 4 + (e & 3)] = acc[TAPS - 1][e];
    bool finite = true;
#pragma unroll
    for (int t = 0; t < TAPS; ++t) finite = finite && (wave * TAPS + t >= V || all_finite(acc[t]));
    if (__any(!finite) && lane == 0) again = 1u;
    __syncthreads();                                                             // (the loaders' after their first pass)
    if (again != 0u && walk.count > 0) {
        // the chunks once more, rows of grad_out that are not finite apart
#pragma unroll
        for (int t = 0; t < TAPS; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[t][e] = 0.f;
        walk_barrier();
        walk_barrier();
        bool done = false;                                                       // every sum is NaN
        for (unsigned i = 0; i < walk.count; ++i) {
            const unsigned char* buf = lds + (i % kWalkBuffers) * kNwBufferBytes;
            const unsigned char* gbuf = buf + kNarrowRowBufPad;
            const unsigned char* table = gbuf + kNwGoutBytes;
            const uint32_t g_at = lds_at(gbuf), row_at = lds_at(buf) + cw;
#pragma unroll 1
            for (int kk = 0; kk < STEPS && !done; ++kk) {
                const Entries lo = entries_of(table, kk * 16 + g * 8 + q), hi = entries_of(table, kk * 16 + g * 8 + q + 4);
                i16x4 f[4 + 2 * TAPS];
                f[0] = lds_read_tr16_at<0>(g_at + g_lo + (uint32_t)(kk * 16 * 64));
                f[1] = lds_read_tr16_at<0>(g_at + g_hi + (uint32_t)(kk * 16 * 64));
                f[2] = f[3] = i16x4{0, 0, 0, 0};
#pragma unroll
                for (int t = 0; t < TAPS; ++t) {
                    f[4 + 2 * t] = lds_read_tr16_at<0>(row_at + (entry(lo, t) ^ (cpiece << 4)));
                    f[5 + 2 * t] = lds_read_tr16_at<0>(row_at + (entry(hi, t) ^ (cpiece << 4)));
                }
                lds_wait_all(f);
                i16x8 gg = __builtin_shufflevector(f[0], f[1], 0, 1, 2, 3, 4, 5, 6, 7);
                uint32_t apart = nonfinite_rows<Tag>(gg);
                if (apart) drop_rows(gg, apart, g);
#pragma unroll
                for (int t = 0; t < TAPS; ++t) {
                    i16x8 ff = __builtin_shufflevector(f[4 + 2 * t], f[5 + 2 * t], 0, 1, 2, 3, 4, 5, 6, 7);
                    if (apart) drop_rows(ff, apart, g);
                    mma16<Tag>(acc[t], gg, ff);
                }
                while (apart) {
                    const int r = kk * 16 + __ffs((int)apart) - 1;
                    apart &= apart - 1u;
                    T4 gv[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        gv[e] = *reinterpret_cast<const T4*>(gbuf + r * 64 + (((uint32_t)e ^ narrow_piece_key((uint32_t)r)) << 4) + g * 8);
                    const Entries entries = entries_of(table, r);
                    T x[TAPS];                                                   // (all reads in flight together; a missing neighbor's: zeros)
#pragma unroll
                    for (int t = 0; t < TAPS; ++t)
                        x[t] = *reinterpret_cast<const T*>(buf + (entry(entries, t) ^ ((uint32_t)((lane & 31) >> 3) << 4)) + (lane & 7) * 2);
#pragma unroll
                    for (int t = 0; t < TAPS; ++t) {
                        if (__builtin_amdgcn_readfirstlane((int)entry(entries, t)) >> 6 == (int)kNarrowZeroSlot) continue;
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[t][e] += (float)gv[e >> 2][e & 3] * (float)x[t];
                    }
                }
            }
            bool nan = true;
#pragma unroll
            for (int t = 0; t < TAPS; ++t) nan = nan && (wave * TAPS + t >= V || all_nan(acc[t], lane, 0, Co, 0, Ci));
            done = __all(nan);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            walk_barrier();
        }
    }
    // partial[workgroup][v][co][ci] (32 x 32 per offset): accumulator element e of lane (l32, g) is co = (e >> 2) * 8 +
    // g * 4 + (e & 3), ci = l32
#pragma unroll
    for (int t = 0; t < TAPS; ++t) {
        const int v = wave * TAPS + t;
        if (v >= V) continue;
        float* dst = partial + ((size_t)blockIdx.x * V + v) * 1024;
#pragma unroll
        for (int e = 0; e < 16; ++e) dst[((e >> 2) * 8 + g * 4 + (e & 3)) * 32 + (lane & 31)] = acc[t][e];
    }
}

// grad_weight[co][v][ci] = sum over the workgroups' partial products.  A workgroup owns 64 consecutive elements of the
// padded (v, co, ci) tiles; four groups of 64 threads each add a quarter of the partial products in ascending order
// (eight loads in flight), and the four sums are added in ascending order: a fixed order, whatever the timing.
template <typename T>
__global__ void __launch_bounds__(256) narrow_wgrad_reduce_kernel(const float* __restrict__ partial, unsigned groups, int V, int Ci,
                                                                  int Co, T* __restrict__ gw, const float* __restrict__ bias_partial,
                                                                  T* __restrict__ gb) {
    __shared__ float part[4][64];
    if (blockIdx.x == (unsigned)V * 16) {                                        // the last workgroup: the column sums
        __shared__ float sums[8][32];
        const unsigned co = threadIdx.x & 31, eighth = threadIdx.x >> 5;
        float s = 0.f;
#pragma unroll 8
        for (unsigned w = eighth; w < groups; w += 8) s += bias_partial[w * 32 + co];
        sums[eighth][co] = s;
        __syncthreads();
        if (eighth == 0 && (int)co < Co) {
            float total = sums[0][co];
#pragma unroll
            for (int q = 1; q < 8; ++q) total += sums[q][co];
            gb[co] = from_float<T>(total);
        }
        return;
    }
    const unsigned i = blockIdx.x * 64 + (threadIdx.x & 63);                     // (v, co, ci) of the padded 32 x 32 tiles
    const unsigned quarter = threadIdx.x >> 6, per = (groups + 3) / 4;
    const unsigned lo = quarter * per, hi = lo + per < groups ? lo + per : groups;
    const size_t stride = (size_t)V * 1024;
    float s = 0.f;
    unsigned w = lo;
    for (; w + 8 <= hi; w += 8) {
        float x[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) x[j] = partial[(size_t)(w + j) * stride + i];
#pragma unroll
        for (int j = 0; j < 8; ++j) s += x[j];
    }
    for (; w < hi; ++w) s += partial[(size_t)w * stride + i];
    part[quarter][threadIdx.x & 63] = s;
    __syncthreads();
    if (quarter == 0) {
        const float total = ((part[0][threadIdx.x] + part[1][threadIdx.x]) + part[2][threadIdx.x]) + part[3][threadIdx.x];
        const int v = i >> 10, co = (i >> 5) & 31, ci = i & 31;
        if (co < Co && ci < Ci) gw[((size_t)co * V + v) * Ci + ci] = from_float<T>(total);
    }
}

int narrow_wgrad_groups(unsigned* out) {
    int dev = 0, cus = 0;
    FGX_CHECK_HIP(hipGetDevice(&dev));
    FGX_CHECK_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    unsigned groups = (unsigned)(cus > 0 ? cus : 256);
    groups = groups / kXcds * kXcds;
    if (groups < (unsigned)kXcds) groups = kXcds;
    *out = groups;
    return FGX_OK;
}

template <typename Tag>
int launch_narrow_wgrad(const void* gout, const void* feats, const void* plan, size_t n, size_t n_src, int V, int Ci, int Co,
                        void* scratch, void* gw, void* gb, hipStream_t s) {
    using T = typename Tag::type;
    unsigned groups = 0;
    int rc = narrow_wgrad_groups(&groups);
    if (rc != FGX_OK) return rc;
    const uint32_t chunks = (uint32_t)((n + kNarrowRows - 1) / kNarrowRows);
    float* bias_partial = gb ? (float*)scratch + (size_t)groups * V * 1024 : nullptr;
    static thread_local bool raised = false;
    if (!raised) {
        FGX_CHECK_HIP(hipFuncSetAttribute((const void*)narrow_wgrad27_kernel<Tag>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kNw27LdsBytes));
        FGX_CHECK_HIP(hipFuncSetAttribute((const void*)narrow_wgrad_kernel<Tag>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kNwLdsBytes));
        raised = true;
    }
    const uint32_t plan_bytes = (uint32_t)(kNarrowHeader + (size_t)chunks * kNarrowPlanStride);
    const uint32_t gout_bytes = (uint32_t)(n * (size_t)Co * 2), feats_bytes = (uint32_t)(n_src * (size_t)Ci * 2);
    if (V == kNarrowCubeV)
        narrow_wgrad27_kernel<Tag><<<groups, kNw27Threads, kNw27LdsBytes, s>>>((const T*)gout, (const T*)feats, (const unsigned char*)plan, chunks, plan_bytes,
                                                                             gout_bytes, feats_bytes, Ci, Co, (float*)scratch, bias_partial);
    else
        narrow_wgrad_kernel<Tag><<<groups, kNwThreads, kNwLdsBytes, s>>>((const T*)gout, (const T*)feats, (const unsigned char*)plan, chunks, plan_bytes,
                                                                         gout_bytes, feats_bytes, V, Ci, Co, (float*)scratch, bias_partial);
    FGX_CHECK_LAUNCH("fgx_conv_narrow_wgrad");
    narrow_wgrad_reduce_kernel<T><<<(unsigned)V * 16 + (gb ? 1u : 0u), 256, 0, s>>>((const float*)scratch, groups, V, Ci, Co, (T*)gw, bias_partial, (T*)gb);
    FGX_CHECK_LAUNCH("fgx_conv_narrow_wgrad(reduce)");
    return FGX_OK;
}

}  // namespace
}  // namespace fgx

using namespace fgx;

extern "C" {

size_t fgx_narrow_wgrad_scratch_bytes(int V) {
    if (V < 1 || V > kNwMult * kNwTaps) return 0;
    unsigned groups = 0;
    if (narrow_wgrad_groups(&groups) != FGX_OK) return 0;
    return (size_t)groups * (V * 1024 + 32) * sizeof(float);
}

int fgx_conv_narrow_wgrad(int dtype, const void* grad_out, const void* feats, const void* plan, size_t n, size_t n_src, int Ci,
                          int Co, int V, void* scratch, void* grad_weight, fgx_stream_t stream) {
    return fgx_conv_narrow_wgrad_bias(dtype, grad_out, feats, plan, n, n_src, Ci, Co, V, scratch, grad_weight, nullptr, stream);
}

int fgx_conv_narrow_wgrad_bias(int dtype, const void* grad_out, const void* feats, const void* plan, size_t n, size_t n_src, int Ci,
                               int Co, int V, void* scratch, void* grad_weight, void* grad_bias, fgx_stream_t stream) {
    FGX_CHECK_ARG(dtype == FGX_F16 || dtype == FGX_BF16, "fgx_conv_narrow_wgrad: 16-bit types only, got dtype %d", dtype);
    FGX_CHECK_ARG(V >= 1 && V <= kNarrowMaxV && V <= kNwMult * kNwTaps, "fgx_conv_narrow_wgrad: bad kernel volume %d", V);
    FGX_CHECK_ARG(Ci >= 8 && Ci <= 32 && Ci % 8 == 0 && Co >= 8 && Co <= 32 && Co % 8 == 0,
                  "fgx_conv_narrow_wgrad: Ci = %d and Co = %d must be 8, 16, 24 or 32", Ci, Co);
    FGX_CHECK_ARG(n > 0 && n < 0xFFFFFFFFull, "fgx_conv_narrow_wgrad: bad row count %zu", n);
    FGX_CHECK_ARG((double)n * Co * 2 < (double)0xFF000000u && (double)n_src * Ci * 2 < (double)0xFF000000u,
                  "fgx_conv_narrow_wgrad: operand too large for 32-bit offsets");
    FGX_CHECK_ARG(grad_out && feats && plan && scratch && grad_weight, "fgx_conv_narrow_wgrad: null buffer");
    FGX_CHECK_ARG((((uintptr_t)grad_out | (uintptr_t)feats | (uintptr_t)plan | (uintptr_t)scratch) & 15) == 0,
                  "fgx_conv_narrow_wgrad: buffers must be 16-byte aligned");
    FGX_CHECK_ARG(kNarrowHeader + ((n + kNarrowRows - 1) / kNarrowRows) * (size_t)kNarrowPlanStride < 0xFF000000ull,
                  "fgx_conv_narrow_wgrad: plan passes the 32-bit offset range");
    hipStream_t s = (hipStream_t)stream;
    if (dtype == FGX_F16) return launch_narrow_wgrad<F16>(grad_out, feats, plan, n, n_src, V, Ci, Co, scratch, grad_weight, grad_bias, s);
    return launch_narrow_wgrad<BF16>(grad_out, feats, plan, n, n_src, V, Ci, Co, scratch, grad_weight, grad_bias, s);
}

}  // extern "C"
