// Fixed gfx950 schedules for the masked implicit GEMM.
//
// The reference times every tile shape and every power-of-two SPLITK on first use and caches the
// winner per (2^floor(log2 N), Ci, Co, V) (flex_gemm/utils/autotuner.py:194-291; candidate ranges in
// ..._masked_implicit_gemm_splitk.py:109-126 and ..._bwd_..._splitk.py:185-202, 254-271).  Here the
// choice is a static function of (floor(log2 N), Ci, Co): a table of measured entries for the shapes
// that were tuned on an MI355X, and a rule for everything else.
#include "fgx_common.h"

#include <algorithm>
#include <cmath>

namespace fgx {
namespace {

constexpr int kCUs = 256;

struct Entry {
    int pass_kind, dtype_bytes, log2n, ci, co;   // dtype_bytes: 2 or 4; 0 = any
    fgx_schedule s;
};

// Measured entries (MI355X).  Rows are matched exactly on (pass, element size, floor(log2 N), Ci, Co).
const Entry kTable[] = {
    // pass dtype log2n  Ci    Co    {rows, cols, slab_bytes, splitk, block_rows, stream}
    {0, 2, 19, 128, 128, {256, 128, 128, 1, 0, 1}},
    {1, 2, 19, 128, 128, {256, 128, 128, 1, 0, 1}},
    {2, 2, 19, 128, 128, {128, 128, 64, 1, 2048, 2}},
    {0, 2, 17, 256, 256, {128, 256, 128, 1, 0, 1}},
    {1, 2, 17, 256, 256, {128, 256, 128, 1, 0, 1}},
    {0, 2, 21, 32, 32, {256, 32, 64, 1, 0, 1}},
    {1, 2, 21, 32, 32, {256, 32, 64, 1, 0, 1}},
    {0, 2, 15, 1024, 1024, {256, 128, 128, 1, 0, 1}},
    {1, 2, 15, 1024, 1024, {256, 128, 128, 1, 0, 1}},
};

int floor_log2(size_t n) {
    int l = 0;
    while (n > 1) { n >>= 1; ++l; }
    return l;
}

int pick_cols(int c) { return c > 64 ? 128 : (c > 32 ? 64 : 32); }

size_t round_up(size_t x, size_t m) { return (x + m - 1) / m * m; }

// fp32: the matrix units take 32-bit operands at a sixteenth of the 16-bit rate, and six products of bf16 parts for one are not much faster,
// so a pass is bound by what is multiplied -- padding and idle CUs included -- before loads count.
//
// Weight gradient: 64 x 64 tiles, or 32 x 32 where those pad at least 28 % less (a 32 x 32 tile multiplies at about that
// much less: 64 160 voxels x 64 channels 0.169 against 0.122 ms), over voxel blocks short enough for about 2000 items of the
// larger tile: an item is (block, offset, tile), and with fewer the centre offset's items alone decide the time.
// Measured (ms; before: 128 x 128 tiles over blocks of 4096 rows and more):  96 channels, 38 720 voxels 0.513 -> 0.202;
// 155 096 voxels 1.08 -> 0.66;  128 channels, 3 840 voxels 0.275 -> 0.038;  166 232 voxels 0.81 -> 0.60;  64 channels,
// 15 192 voxels 0.096 -> 0.045;  16 channels, 669 288 voxels 0.75 -> 0.45.  From 1024 x 1024 channels on, where partial products
// must stay few and blocks are long, the 128 x 128 tile of the general rule is ahead (42 608 voxels: 9.5 ms against 10.3).
bool rule_wgrad_f32(size_t n, int Ci, int Co, int V, fgx_schedule* out) {
    if ((size_t)Ci * Co >= (size_t)1024 * 1024) return false;
    auto padded = [&](int t) { return (double)cdiv(Ci, t) * t * cdiv(Co, t) * t; };
    const int t = padded(32) < 0.72 * padded(64) ? 32 : 64;
    const double tiles = (double)cdiv(Ci, t) * cdiv(Co, t);
    const double ideal = (double)n * V * tiles / (t == 64 ? 2000.0 : 4000.0);
    size_t rows = V * tiles < 400 ? 512 : 1024;
    while (rows < 4096 && ideal > 1.42 * rows) rows *= 2;
    const double per_block = 4.0 * V * (double)Co * Ci;            // partial products stay below 256 MiB
    while ((double)cdiv(n ? n : 1, rows) * per_block > 268435456.0 && rows < ((size_t)1 << 29)) rows *= 2;
    if (n > rows) rows = round_up(cdiv(n, cdiv(n, rows)), 64);       // even blocks
    *out = fgx_schedule{t, t, 64, 1, (int)rows, 0};
    return true;
}

// Gather GEMM: what a CU multiplies, in columns of 256-row tiles and bytes of K in whole slabs, under each choice.
//   streaming kernel, three bf16 parts a value (csrc/split3.h), tiles of r x c: items per CU and what the launch waits for its
//   last and heaviest ones (`last`; `least` for a lone round, whose heaviest tile has half as many offsets again as the mean), at
//   a rate that falls with c: a fragment's parts are made once and multiplied c / 32 times; 7 us of its own;
//   tiled kernel, on the fp32 units, with K split until the pieces even out: a third of the rate, and 15 us of its own.
// Measured forward, us, 256 x 128 / 256 x 64 / 256 x 32 (64-byte slabs but for the first):  128 channels, 49 976 voxels 217 246
// 263;  77 064 287 315 343;  166 232 440 555 605;  406 920 938 1 205 1 365;  96 channels, 166 232 voxels 324 423 345;  192
// channels 1 135 1 187 1 312, 128 x 256 1 112;  48 channels 222 128 131, 64 channels 227 163 171.  256 x 64 on 64- and 128-byte slabs: 166 232
// voxels, into 64 columns, of 32 channels 99 92, 40 127 151, 64 162 152, 80 197 216, 96 232 217, 112 267 281, 128 302 283, 192 442 416; 49 976 voxels, 64 87
// 81, 128 162 150; 406 920, 64 342 320, 128 642 606.  32 channels, 77 064 voxels 89 64 43, tiled 51; 48, 36 936 voxels 79 (256 x 64) 68 (256 x 32), tiled 75,
// 20 330 75 54 66.  With what the fp32 units wanted (narrow tiles before padding) the products
// of three parts took 554 us under 128 channels at 166 977 voxels, on the fp32 units 681;  192 channels 1 301 and 1 378.
void rule_gemm_f32(size_t n, int K, int cols, int V, fgx_schedule* out) {
    const size_t row_bytes = (size_t)K * 4;
    const int slab = row_bytes % 128 == 0 ? 128 : 64;   // (of 64 columns: the longer ones are 6 to 8 % ahead where none is part empty)
    const double row_tiles = cdiv(n ? n : 1, 256);
    const int wide = cdiv(cols, 64) * 64;
    const bool narrow = cdiv(cols, 32) * 32 < wide;
    double best = row_tiles * (narrow ? cdiv(cols, 32) * 32 : wide) / kCUs / 0.33 * align_up(row_bytes, 64) + 15.0 * 446.0 * 27 / V;     // (446: of a microsecond)
    *out = fgx_schedule{narrow && n < 1024 ? 32 : 64, narrow ? 32 : 64, 64, 1, 0, 0};
    if (cdiv(cols, 128) * 128 == wide && row_bytes >= 1024 && cdiv(n ? n : 1, 128) * cdiv(cols, 128) >= 32) out->tile_rows = out->tile_cols = 128;
    {
        const size_t tiles = (size_t)cdiv(n ? n : 1, out->tile_rows) * cdiv(cols, out->tile_cols);
        const int steps = V * (int)cdiv(row_bytes, (size_t)64);
        int s = 1;
        while (tiles * s < (s < 8 ? 1500u : 300u) && s < 16 && 12 * s <= steps) s *= 2;
        out->splitk = s;
    }
    if (row_bytes < 64) return;
    struct Shape { int rows, cols, slab; double rate, last, least; };
    const Shape shapes[] = {{128, 256, 128, 1.04, 0.4, 1.45}, {256, 128, 128, 1.0, 0.6, 1.45}, {256, 64, slab, 0.79, 0.8, 1.75}, {256, 32, 64, 0.74, 1.4, 2.2}};
    for (const Shape& sh : shapes) {
        if (sh.slab > (int)align_up(row_bytes, 64) || (sh.cols == 256 && cols <= 128) || !stream_lds_fits(sh.rows, sh.cols, sh.slab, cols)) continue;
        const double items = (double)cdiv(n ? n : 1, sh.rows) * cdiv(cols, sh.cols) / kCUs;
        const double rounds = std::max(items + sh.last, sh.least);
        const double time = rounds * sh.cols * sh.rows / 256.0 / sh.rate * align_up(row_bytes, sh.slab) + 7.0 * 446.0 * 27 / V;
        if (time < best) {
            best = time;
            *out = fgx_schedule{sh.rows, sh.cols, sh.slab, 1, 0, 1};
        }
    }
}

// 16-bit gather GEMM where tiles of 256 rows leave CUs idle or fill them unevenly: streaming tiles of 64 and 128 rows, two workgroups to a CU but
// for 128 x 128.  A step of any tile takes a CU about as long as its loads do (34 bytes a cycle), so small tiles, which load more for a product, are behind
// once the chip is full, and ahead before: 64 x 64 goes through an item of one slab in 5.4 us, 256 x 128 in 15.  They also pad less.
// With items per CU x, slabs s: s (L^1.5 + (x P)^1.5)^(2/3), where L is what an item takes alone and P beside others (us; the tile of 256 rows: whole rounds).
// Measured forward, us, what was chosen before and now, 27 offsets:
//   channels        8 004 voxels   10 494       15 091      20 574      28 169      36 575      75 224      166 977
//    64 ->  64        18.6         20.3 16.3    23.1 16.3   24.7 17.1   27.9 18.2   24.7 19.8   28.8 24.4   45.9 37.6
//   128 -> 128        35.0 22.9    35.4 26.4    36.8 25.7   36.3 28.8   36.7 29.5   40.7 34.4   51.8        85.7
//   192 -> 192        43.1 33.6    62.1 34.1    49.3 40.6   48.8 44.6   54.8        71.4 64.0   105.9       198
//   256 -> 256        65.2 42.1    60.5 53.1    60.7        67.2        71.7        89.2        145.9       271
//   512 ->  64        54.7         60.5 56.3                100.8 56.6              165.9 75.9  156.0 135.1 300 276
//    64 -> 256        26.3 18.9    26.3 22.7                28.2                    33.0        46.5        83.1
// (where one figure stands, the tile stays; 64 -> 64 stays tiled below 24 576 voxels.)  The tiled kernel splits few rows well: under up to 64 columns, or rows of 512 bytes and more, it is level up
// to 10 000 voxels (8 004: 96 -> 64 21.0 22.3, 384 -> 96 43 47, 768 -> 128 64 83), otherwise up to 5 000 (4 947: 80 -> 80 21.0 22.7); and it wants no gather
// plan and no packed weight, 14 us of the host's time in a training pass on new coordinates, which little work does not bring in (64 -> 64 at 10 494 voxels
// gains 3.5 us a product, at 28 169 9.7).  A plan of another height than the neighboring layers' costs a new cache 6 to 13 us of the device, which the limits in n
// stand for as far as one layer can tell; a stack of unlike widths may pay it twice (32 -> 64 -> 128 at inference, 36 936 voxels 115 127; most gain, 20 330 113 102).
bool small_stream_tile(size_t n, int K, int cols, fgx_schedule* out) {
    const int slabs = (int)cdiv((size_t)K * 2, (size_t)128);
    if (K * 2 <= 64 || !stream_lds_fits(256, 128, 128, cols)) return false;
    // Up to 32 columns: 64 x 32 and 128 x 32.  Before, now:  64 -> 32 channels, 36 575 voxels 24.3 17.6, 75 224 25.8 21.8;  72 -> 24 166 977 69.8 55.2, 448 584
    // 148 130;  128 -> 32 20 574 25.4 20.2, 36 575 33.6 23.5, 75 224 54.4 34.2, 166 977 99.5 61.6;  256 -> 32 37.8 29.6, 53.5 34.8, 99.1 58.9, 185 116;
    // 512 -> 32 62 50, 95 66, 190 122, 352 245.  Not where a plan of this tile's own costs a new cache as much (20 574 voxels 72 -> 24 68.5 73.8, 128 -> 32 72.2
    // 72.4; 64 -> 32, whose input gradient has another, training on new coordinates, 73 461 voxels 216 212, 123 180 245 255) or more than the tile gains over
    // the 256 x 32 one, whose plan the wider layers of a stack share (65 ... 127 channels up to 131 072 voxels: 123 180 43.8 40.4, a plan 13).
    if (cols <= 32) {
        if (n > (slabs == 1 ? 98304u : K < 128 ? 524288u : 262144u) || (!out->stream && n < (K <= 96 ? 32768u : 20480u))) return false;
        if (slabs == 2 && out->stream && n < 131072) return false;
        *out = fgx_schedule{(slabs == 1 && n > 36864) || (slabs == 2 && K < 128 && n > 57344) ? 128 : 64, 32, 128, 1, 0, 1};
        return true;
    }
    // (rows of 128 bytes past 262 144 voxels: 277 018 62.5 56.2, 1 041 730 184 184; of two slabs past 131 072: the input gradient's plan is another, 96 -> 64,
    // training on new coordinates, 123 180 voxels 310 311, 244 211 459 465; 4 096 tiles are filled in one launch with their tables)
    if (n > (cols > 64 || slabs == 2 ? 131072u : slabs > 2 || K == 64 ? 262144u : 524288u) || (!out->stream && (n < (cols <= 64 || K >= 256 ? 10240u : 5120u) || n * slabs * cdiv(cols, 64) < 24576))) return false;
    auto take = [&](int rows, int wide) {
        *out = fgx_schedule{rows, wide, 128, 1, 0, 1};
        return true;
    };
    if (cols <= 64) {
        if (slabs >= 16 && n > 131072) return false;
        return take(slabs > 2 || n <= (slabs == 1 ? 36864u : 57344u) ? 64 : 128, 64);
    }
    // long rows under one tile of columns: 75 224 voxels, 384 -> 96 132 120, 768 -> 128 270 251
    if (cols <= 128 && K >= 384 && n >= 28672) return take(128, 128);
    if (cols > 192 && K >= 192 && n > 12288) return false;              // (the larger tiles fill the chip by then)
    const bool whole_chip = out->stream && out->tile_cols != 64;        // (256 x 128 and 128 x 256 tiles for at least half of the CUs)
    if (whole_chip && (cols > 128 || n > 40960)) return false;
    struct Shape { int rows, cols; double alone, beside; };
    const Shape shapes[] = {{64, 64, 5.4, 2.9}, {64, 128, 7.0, 3.7}, {128, 64, 7.45, 4.0}, {128, 128, 10.3, 6.5}};
    auto per_cu = [&](int rows, int wide) { return (double)cdiv(n, rows) * cdiv(cols, wide) / kCUs; };
    // (a tile that was chosen for its rounds: a whole one at the least, and most of one for each of its items)
    double best = 1e30;
    if (out->stream) best = 0.97 * (whole_chip ? 15.0 : 11.9) * std::max(1.0, 0.45 + 0.68 * per_cu(out->tile_rows, out->tile_cols));
    bool found = false;
    for (const Shape& sh : shapes) {
        const double time = std::pow(std::pow(sh.alone, 1.5) + std::pow(per_cu(sh.rows, sh.cols) * sh.beside, 1.5), 2.0 / 3.0);
        if (time < best) {
            best = time;
            found = take(sh.rows, sh.cols);
        }
    }
    return found;
}

void rule(int pass_kind, int es, size_t n, int Ci, int Co, int V, fgx_schedule* out) {
    if (es == 4 && pass_kind != 2) return rule_gemm_f32(n, pass_kind == 0 ? Ci : Co, pass_kind == 0 ? Co : Ci, V, out);
    if (es == 4 && rule_wgrad_f32(n, Ci, Co, V, out)) return;
    if (pass_kind == 2) {
        // wgrad: tiles over (Co, Ci) and voxel blocks; an item is (block, offset, tile), every item costs an exposed
        // epilogue and a partial product, and the fp32 partial products (blocks x V x Co x Ci) stay below 256 MiB.
        int t = pick_cols(Ci < Co ? Ci : Co);
        out->tile_rows = t;
        out->tile_cols = t;
        out->slab_bytes = 64;
        out->splitk = 1;
        // persistent streaming kernel: 16-bit types; measured ahead of the tiled kernel from a few hundred voxels on
        // (848 voxels: C = 32 0.024 -> 0.020 ms, C = 64 0.023 -> 0.020, C = 128 0.031 -> 0.020, C = 256 0.033 -> 0.023).
        // Under a weight of 512 x 512 channels and more it is ahead from the smallest layers on (C = 1024: 192 voxels 0.053 ->
        // 0.048 ms, 848 voxels 0.084 -> 0.072, 1 976 voxels 0.134 -> 0.115; C = 512: 1 976 voxels 0.055 -> 0.043).
        out->stream = (es == 2 && (n >= 512 || (n >= 128 && (size_t)Ci * Co >= (size_t)512 * 512))) ? 1 : 0;
        // A weight of one 64 x 64 or 128 x 128 tile (33 ... 128 channels on both sides): the sweep (stream = 2) --
        // every workgroup keeps two accumulators over an eighth of the voxels, block_rows is its sub-block size.
        // Measured 20 % to 30 % ahead of the block-major kernel from ten thousand voxels (C = 128: 0.051 against
        // 0.067 ms) to 2.7 million (1.32 against 1.70 ms), for C = 64, 96, 128, coordinates in scan order or shuffled.
        // 33 ... 64 channels on one side and 65 ... 128 on the other: the 128 x 128 tile, half of it empty, from 65 536 voxels and under kernels of more than
        // 8 offsets (the product alone, us: 64 -> 128, 166 977 voxels 107 and 84, 667 763 453 and 269; 38 407 45 and 44;  training with a fresh cache,
        // its plan included: 65 145 voxels 269 256, 166 789 405 389, 667 156 1130 997; 128 -> 64, 50 850 kept 115 117; under
        // 2 x 2 x 2, 180 000 outputs fresh 366 381).  The narrow end of the range gains as much, though more of the tile is empty, since the other kernel's two
        // 64 x 64 tiles pad as well (alone, and with cache and plan: 40 -> 72, 67 107 voxels 65 56, 199 185; 167 946 137 93, 299 242, in random order
        // 138 89, 317 258; 667 763 442 254, 636 489; 72 -> 64, 67 107 64 55, 194 183; 667 763 448 250, 650 482).
        const int wide = Ci > 64 || Co > 64 ? 128 : 64;
        // ... and 17 ... 32 channels on one side and 97 ... 128 on the other, four 32 x 32 tiles, from 131 072 voxels (32 -> 128, the product alone: 166 977
        // voxels 107 and 82, 667 763 380 and 250; training with a fresh cache: 125 569 voxels 384 358, 166 789 424 379, 667 156 1026 955;
        // 24 -> 72, three tiles: 125 569 voxels 310 316, 667 156 905 929;  24 -> 104, alone, and with cache and plan: 166 977 voxels 121 79, 291 230, in random
        // order 141 86, 331 253; 667 763 387 261, 575 482; 128 -> 24, 166 977 99 82, 268 229).
        const int narrow = Ci < Co ? Ci : Co, most = Ci < Co ? Co : Ci;
        const bool mixed = wide == 128 && V > 8 && (t == 64 ? n >= 65536 : t == 32 && narrow > 16 && most > 96 && n >= 131072);
        if (es == 2 && n >= 8192 && n <= ((size_t)1 << 24) && (t >= 64 || mixed) && V <= 2 * (kCUs / 8) && Ci <= wide && Co <= wide && (wide == t || mixed)) {
            out->tile_rows = out->tile_cols = wide;
            out->stream = 2;
            out->block_rows = 2048;
            return;
        }
        // 33 ... 64 channels on one side and over 192 on the other, or over 128 of many voxels: three and more 64 x 64 tiles.  The tiled kernel over short
        // blocks is ahead of the streaming one, whose workgroups walk one tile's pairs at a time (256 -> 64 channels, 38 720
        // voxels: 0.057 against 0.071 ms; 64 -> 160 channels, 228 816 voxels: 0.178 against 0.219).
        // ... and up to 32 channels on one side, in the same 64 x 64 tiles: of a row's 128 bytes a step's pairs ask for half as many lines a byte as in
        // 32 x 32 ones, which are asked for again by every tile (us, 32 x 32 streaming and this: 200 -> 32, 134 572 voxels 144 154, 166 977 183 174,
        // 294 092 343 268;  144 -> 32 96 124, 129 142, 241 213;  320 -> 24 166 179, 209 207, 374 330;  448 -> 32, 101 586 178 166, 294 092 560 433, 49 829
        // 106 108;  32 -> 640, 294 092 896 630).
        const bool lopsided = t == 32 && ((most > 384 && n >= 98304) || (most > 128 && n >= 196608));
        if (out->stream == 1 && ((t == 64 && (Ci > 192 || Co > 192 || ((Ci > 128 || Co > 128) && n >= 98304)) && n >= 12288) || lopsided)) {
            out->tile_rows = out->tile_cols = 64;
            out->stream = 0;
            size_t rows = n >= 98304 ? 4096 : 2048;
            const double per_block = 4.0 * V * (double)Co * Ci;
            while ((double)cdiv(n, rows) * per_block > 268435456.0 && rows < ((size_t)1 << 29)) rows *= 2;
            out->block_rows = (int)round_up(cdiv(n, cdiv(n, rows)), 64);
            return;
        }
        // Streaming kernel with balanced work lists (fgx_wgrad_item_lists): a launch takes as long as its most loaded
        // workgroup, and the lists even the loads out as far as the items allow -- the largest item is the centre
        // offset of a voxel block (one pair per row), the mean load is about 0.45 V pairs per voxel x tiles / CUs.
        // So: the largest tile shape whose items still fill the chip one and a half times with blocks of 4096 rows or
        // more, and as few blocks as keep a block's centre item below the mean load (CUs / (0.45 V x tiles) blocks).
        // Measured on shells with the lists (ms, best of the swept tile shapes and block counts):
        //   C = 256:  848 voxels 64 x 64 tiles 1 block 0.023 (tiled kernel 0.033);  3 840: 64 x 64, 1 block 0.035
        //             (256 x 128: 0.063);  15 192: 128 x 128, 4 blocks 0.059 (256 x 128, 4: 0.077);  64 160: 256 x 128,
        //             8 blocks 0.156, 11: 0.169 (16: 0.176);  166 232: 256 x 128, 11 blocks 0.295 (8: 0.337, 24: 0.329)
        //   C = 512:  3 840: 128 x 128, 1 block 0.054 (256 x 128: 0.072);  15 192: 256 x 128, 2 blocks 0.144, 3: 0.150
        //             (4: 0.162);  64 160: 256 x 128, 3 blocks 0.484 (5: 0.503, 8: 0.520)
        //   C = 1024: 3 840 ... 64 160 voxels: 256 x 128, 1 block (42 608 voxels: 0.957, 2 blocks 1.02, 4: 1.12)
        //   C = 32:   15 192: 8 blocks 0.026 (1: 0.040);  64 160: 11 blocks 0.030 (4: 0.046, 32: 0.040)
        // Tiles of 256 x 128 (or 128 x 256 where only Ci is wide) where they pad no more than 128 x 128 ones do: a step
        // then loads 48 KiB of rows for twice the products, and these shapes are bound by what the CUs can pull out
        // of L2.  Below about three thousand voxels the square tile's larger number of items counts for more.
        if (out->stream == 1) {
            struct Shape { int rows, cols; };
            Shape shapes[3];
            int ns = 0;
            if (t == 128) {
                if (n >= 3072 && Co > 128 && cdiv(Co, 256) * 256 == cdiv(Co, 128) * 128) shapes[ns++] = {256, 128};
                else if (n >= 3072 && Ci > 128 && cdiv(Ci, 256) * 256 == cdiv(Ci, 128) * 128) shapes[ns++] = {128, 256};
                shapes[ns++] = {128, 128};
                shapes[ns++] = {64, 64};
            } else {
                shapes[ns++] = {t, t};
            }
            size_t nb = 1, tiles = 1;
            int slices = 1;
            for (int i = 0; i < ns; ++i) {
                const bool last = i == ns - 1;
                slices = shapes[i].rows == 32 ? 4 : 1;           // the 32 x 32 tile splits a step's pairs over its four wavefronts
                tiles = (size_t)cdiv(Co, shapes[i].rows) * cdiv(Ci, shapes[i].cols);
                const size_t per_voxel = (size_t)V * 4 / 9 * (slices == 4 ? 2 : 1);
                const size_t wanted = cdiv((size_t)kCUs, (per_voxel ? per_voxel : 1) * tiles);
                const size_t shortest = slices == 4 ? 2048 : 4096;
                const size_t most = n > shortest ? cdiv(n, shortest) : 1;
                nb = wanted < most ? wanted : most;
                out->tile_rows = shapes[i].rows;
                out->tile_cols = shapes[i].cols;
                // How many items fill the chip: of 128 x 128 tiles a few more than CUs (324 items: 3 840 voxels, 256 -> 768 channels
                // 0.050 ms, 64 x 64 tiles 0.083; 848 voxels 0.031 and 0.038), of the larger ones half as many again.
                const bool square = shapes[i].rows == 128 && shapes[i].cols == 128;
                bool fills = (size_t)V * tiles * nb >= (square ? (size_t)kCUs * 5 / 4 : (size_t)kCUs * 3 / 2);
                if (square && !fills && n > 4096 && n <= 8192 && 10 * tiles * 4 <= (size_t)11 * cdiv(Co, 64) * cdiv(Ci, 64)) {
                    // ... in blocks of 1024 rows before smaller tiles, where they pad no more than those (5 816 voxels, 256 channels
                    // 0.051 -> 0.043 ms; 192 channels, padded to 256, 0.035 -> 0.045: not there)
                    const size_t most_short = cdiv(n, (size_t)1024), nb_short = wanted < most_short ? wanted : most_short;
                    if ((size_t)V * tiles * nb_short >= (size_t)kCUs * 5 / 4) {
                        nb = nb_short;
                        fills = true;
                    }
                }
                if (last && !fills) {
                    // nothing fills the chip: blocks down to 1024 rows (64 channels, 3 840 voxels: 0.020 -> 0.016 ms), 2048 where
                    // the tile splits its pairs over the wavefronts itself or two short blocks would be all (1 976 voxels,
                    // 64 -> 384 channels: 0.020 ms, one block 0.016)
                    const size_t least = (slices == 4 || n < 3072) ? 2048 : 1024;
                    const size_t most_short = n > least ? cdiv(n, least) : 1;
                    const size_t filling = cdiv((size_t)3 * kCUs, (size_t)2 * V * tiles);
                    nb = wanted < most_short ? wanted : most_short;
                    if (nb > filling) nb = filling;
                }
                if (last || fills) break;
            }
            // long blocks overflow an XCD's L2 when few tiles share their rows; partial products stay below 256 MiB
            // (nine tiles that pad, from 131 072 voxels on: blocks as of eight tiles while the lists take them, 16 at most; 272 channels, 166 977 voxels 717 -> 644 us,
            // 277 018 1 237 -> 1 052, 448 584 2 063 -> 1 758, blocks of 24 576 there 2 594;  320 channels 711 671, 1 214 1 142, 1 997 1 752.  Level or behind before,
            // 101 586 voxels 418 420 and 426 435, and where nothing is padded, 384 channels 653 665, 1 100 1 105)
            const bool pads = Ci % 128 != 0 || Co % 128 != 0;
            const size_t nine = !pads || n < 131072 ? 65536 : n <= 393216 ? 24576 : n <= 524288 ? 32768 : 65536;
            const size_t longest = tiles <= 4 ? 16384 : tiles <= 8 ? 24576 : tiles == 9 ? nine : 65536;
            if (nb < cdiv(n, longest)) nb = cdiv(n, longest);
            size_t max_blocks = (size_t)(268435456.0 / (4.0 * V * (double)Co * (double)Ci * slices));
            if (max_blocks < 1) max_blocks = 1;
            if (nb > max_blocks) nb = max_blocks;
            // The lists exist for up to 12 voxel blocks (16 when a block has several tiles per offset); beyond, the fixed
            // interleave runs (it keeps the offsets of a voxel block on one XCD, and with that many blocks it is balanced
            // well enough) on the blocks below.
            if (nb <= (tiles >= 2 ? 16u : 12u)) {
                size_t rows = round_up(cdiv(n, nb), 1024);
                if (rows > 0x40000000) rows = 0x40000000;
                out->block_rows = (int)rows;
                return;
            }
        }
        // Fixed interleave (the tiled kernel: fp32 or few voxels; the streaming kernel over more than 12 blocks): voxel
        // blocks of 4096 to 12288 rows -- as long as that still leaves about four items per CU: blocks beyond ~12K rows
        // overflow an XCD's L2 (measured at C = 128 ... 512: 12288 rows are 4 % to 11 % ahead of 4096 once there are enough
        // voxels; 16384 under 256-row tiles and for the 32 x 32 streaming tile, which writes four partial products per
        // block: 1 026 536 voxels at 32 channels, 16384 rows 0.161 ms, 32768 0.170, 65536 0.185).
        const int slices = (out->stream && out->tile_rows == 32) ? 4 : 1;
        const double per_block = 4.0 * V * (double)Co * (double)Ci * slices;
        size_t max_blocks = (size_t)(268435456.0 / per_block);
        if (max_blocks < 1) max_blocks = 1;
        const size_t tiles = (size_t)cdiv(Co, out->tile_rows) * cdiv(Ci, out->tile_cols);
        size_t blocks_wanted = cdiv((size_t)4 * kCUs, (size_t)V * tiles);
        if (blocks_wanted < 1) blocks_wanted = 1;
        size_t rows = round_up(cdiv(n ? n : 1, blocks_wanted), 1024);
        if (rows < (size_t)4096 * slices) rows = (size_t)4096 * slices;        // (32 x 32: 16384, its longest as well)
        const size_t longest = (out->tile_rows == 256 || out->tile_cols == 256 || slices == 4) ? 16384 : 12288;
        if (rows > longest) rows = longest;
        const size_t rows_mem = round_up((n + max_blocks - 1) / max_blocks, 1024);
        if (rows < rows_mem) rows = rows_mem;
        // even blocks: with a handful of them a short last block leaves its workgroups idle (two blocks of 12288 + 2904
        // rows: 0.86 ms, of 8192 + 7000: 0.62 ms at C = 1024)
        if (n > 0) rows = round_up(cdiv(n, cdiv(n, rows)), 1024);
        if (rows > 0x40000000) rows = 0x40000000;
        out->block_rows = (int)rows;
        return;
    }
    const int cols = pass_kind == 0 ? Co : Ci;
    const int K = pass_kind == 0 ? Ci : Co;
    const size_t row_bytes = (size_t)K * es;
    // Tiled kernel: 64 x 64 tiles (one of 32 columns where there are no more), 128 x 128 once splits of four go round with
    // those; K split until the CUs have one to three pieces each, as many as the tile's size leaves room for.  A piece's partial
    // sums are written and read again, so more than eight only of a long K.  (848 voxels: 8 splits against 16, C = 32 0.015 ->
    // 0.013 ms; C = 80 128 x 128 in 16 splits 0.022, these 0.016; 3 840 voxels, C = 128: 0.030 -> 0.026 in 4; 13 488 voxels,
    // C = 128: 128 x 128 in 4 0.042, 64 x 64 0.053; 15 192 voxels, 320 -> 16 channels in 2 0.060, in 4 0.044.)
    // A long K keeps the larger tile, which reads half as much per product: 256 channels and more
    // (848 voxels, 256 -> 768 channels: 0.042 ms, 64 x 64 0.062; 1 976 voxels, 256 channels: 0.034 and 0.038).
    out->tile_rows = (cols > 32 || n >= 1024) ? 64 : 32;
    out->tile_cols = cols > 32 ? 64 : 32;
    const bool long_k = row_bytes >= 512 && n >= 256;
    if (cols > 64 && (long_k || (size_t)cdiv(n, 128) * cdiv(cols, 128) >= (size_t)kCUs / 4)) out->tile_rows = out->tile_cols = 128;
    else if (cols > 32 && cols <= 64 && (size_t)cdiv(n, 128) >= 2 * (size_t)kCUs) out->tile_rows = 128;
    out->block_rows = 0;
    out->stream = 0;
    out->slab_bytes = 64;
    const size_t tiles = (size_t)cdiv(n ? n : 1, out->tile_rows) * cdiv(cols, out->tile_cols);
    int s = 1;
    const size_t steps = (size_t)V * cdiv(row_bytes, (size_t)64);
    for (; s < (steps >= 160 ? 16 : 8); s *= 2) {
        size_t pieces = cols <= 32 ? 700 : kCUs;
        // (input gradients on 128 x 128 tiles under a long K: two pieces for a CU rather than one and a half; 5 816 voxels, 256 channels in 4
        // splits 0.051 ms, in 8 0.045; 384 -> 256 0.067 and 0.057; not from 1.6 on: 13 488 voxels, 96 <- 320 0.059 and 0.064.  The forward
        // pass would gain as much -- 5 816 voxels, 256 channels 0.050 and 0.046, 1 976 voxels, 256 -> 768 0.051 and 0.047 -- and does
        // without it: another split rounds a forward sum differently, so that a ReLU behind it changes sides here and there, and
        // results stay those of the splits it has had.)
        if (pass_kind != 0 && out->tile_rows == 128 && out->tile_cols == 128 && steps >= 160) pieces = 400;
        if (out->tile_cols == 64 && (s < 4 ? steps >= 54 : (s < 8 && steps >= 320))) pieces = 450;
        if (tiles * s >= pieces) break;
    }
    out->splitk = s;
    // Persistent streaming kernel: rows of at least 64 bytes; 64-byte K-slabs for rows of one, 128-byte ones for longer rows: of 72 ... 127 bytes
    // one slab holds the row, what is past its end is not loaded, and an offset is one step instead of two (forward, 64- and 128-byte
    // slabs, us: 40 channels, 166 977 voxels 49.1 42.8, 407 279 94.5 88.9;  56 channels 58.3 47.3 and 117 104).
    // 16-bit rows of 128 ... 192 bytes (64 ... 96 channels) also take the 64-byte slabs while one column tile holds the outputs:
    // their rings leave room for two workgroups per CU, which is worth more than the longer pieces (measured forward, C = 64:
    // 143 616 / 252 392 / 577 592 / 1 026 536 voxels -5 / -22 / -7 / -12 %; C = 80 and 96: -2 ... -5 %) ... given two items per CU to keep both
    // workgroups busy (64 160 voxels, 251 items: 0.028 ms on 128-byte slabs, 0.031 on 64-byte ones).  Beyond 192 bytes they are four
    // steps for two (112 channels, 166 977 voxels 101 87, 407 279 217 199;  C = 128: 0.056 against 0.049 ms at 64 160 voxels).
    const bool short_slabs = row_bytes >= 128 && row_bytes <= 192 && cols <= 128 &&
                             (size_t)cdiv(n, 256) * cdiv(cols, cols > 64 ? 128 : 64) >= 2 * (size_t)kCUs;
    const int slab = (row_bytes > 64 && !short_slabs) ? 128 : 64;
    // The tile by what a CU multiplies and loads: whole items per CU, each its columns (of 256 rows) at the tile's rate.  One
    // tile of 128 rows x 256 columns gathers every row once for the same bytes per product as 256 x 128, and pads less;
    // 64-column tiles read a gathered row from L2 more often but even out a chip that larger ones fill 1.3 times or less than
    // half (measured forward: 42 608 voxels C = 192, 128 x 256 0.084 ms, 256 x 64 0.078; 8 624 voxels C = 384 0.131 ms in two
    // K splits, 0.096 on 256 x 64; 15 192 voxels C = 128 0.043 -> 0.039; 64 -> 160 channels at 228 816 voxels 256 x 128 on 64-byte
    // slabs 0.135, 128 x 256 0.104; 38 720 voxels C = 48 tiled 0.038, 256 x 64 0.027).
    // An item for half of the CUs is enough (15 192 voxels, 120 items: 384 -> 80 channels 0.087 ms, tiled 0.070; 160 -> 128
    // 0.052 and 0.044), for five eighths where the outputs are up to 32 columns, with little to multiply, and on rows of
    // 1 KiB, which the tiled kernel below splits well (1 976 voxels, C = 1024: 128 items 0.232 ms, tiled 0.166).
    // Up to 32 columns under rows of 256 bytes and more: from 320 000 voxels, where it is ahead with the tables of a fresh cache too (cache and
    // one layer, tiled 64 x 32 and 256 x 32: 128 -> 16 channels, 329 832 voxels 261 252 us, 1 053 495 970 891; 272 -> 32 484 456, 2 190 1 795;
    // 512 -> 16 723 696.  299 416 voxels: 512 -> 16 659 661, 128 -> 16 246 240;  166 789: 405 426 and 167 171.  With a kept cache
    // 1.1 to 1.4 times as fast from 320 000 on).  Not under few offsets, whose products do not pay for those tables: up to 3 (128 -> 32 channels, 350 457 and
    // 624 671 voxels, one layer at inference, fresh: 1 x 1 x 1 71 85 and 97 121, 3 x 1 x 1 94 103 and 135 151, where 2 x 2 x 2 has 461 433), and for input
    // gradients up to 8, of which a stride leaves one or two (2 x 2 x 2 under a stride of 2, 16 -> 128, training, fresh: 350 457 inputs 257 285,
    // 1 057 251 448 514; kept 96 95 and 232 202).
    const bool tables_pay = n >= 320000 && V > (pass_kind == 1 ? 8 : 3);
    struct Shape { int rows, cols, slab; double rate; };
    const Shape shapes[] = {{128, 256, 128, 1.0}, {256, 128, slab, 0.95}, {256, 64, slab, 0.6}, {256, 32, 64, 0.5}};
    double best = 0.0;
    for (const Shape& sh : shapes) {
        if (row_bytes < 64 || sh.slab > (int)align_up(row_bytes, 64)) continue;
        if (sh.cols == 256 ? cols <= 128 || slab != 128 : (sh.cols == 128 ? cols <= 64 : (sh.cols == 64 ? cols <= 32 : cols > 32 || (row_bytes >= 256 && !tables_pay)))) continue;
        // (from ~1900 output columns on the staged bias does not fit beside the rings of the 256 x 128 tile; the other shapes,
        // whose rings leave a little more room, are no help under a weight that wide)
        if (!stream_lds_fits(sh.rows, sh.cols, sh.slab, cols) || (cols > 128 && !stream_lds_fits(256, 128, slab, cols))) continue;
        const size_t items = (size_t)cdiv(n ? n : 1, sh.rows) * cdiv(cols, sh.cols);
        if (items < (size_t)kCUs * (sh.cols == 32 || row_bytes >= 1024 ? 5 : 4) / 8) continue;
        const double time = cdiv(items, (size_t)kCUs) * (sh.cols * sh.rows / 256.0 / sh.rate);
        if (best == 0.0 || time < best) {
            best = time;
            *out = fgx_schedule{sh.rows, sh.cols, sh.slab, 1, 0, 1};
        }
    }
    if (V > 8 && small_stream_tile(n, K, cols, out)) return;
    // 5 to 8 offsets: 64 x 128 where the products alone leave the chip idle in 256-row or 128 x 256 tiles (one layer at inference, us, kept coordinates, new ones:
    // 2 x 2 x 2 under a stride of 2, 256 -> 256 channels, 8 449 outputs 26 20, 92 82; 10 536 26 20, 94 84; 20 753 31 24, 95 87;  128 -> 128 20 753 17 14, 81 76;
    // 30 714 18 16, 86 78;  384 -> 512 10 536 42 34, 107 99.  1 x 2 x 3 256 -> 256 10 340 22 16, 91 81.  5 x 1 x 1 submanifold 13 572 20 17, 63 56).  Past this the larger
    // tiles fill the chip (33 900 128 -> 256 23.1 22.6, 89 93; 19 650 384 -> 512 36 37, 62 68).  Both directions take it or neither, by the fewer and the more of the
    // channels: a submanifold layer's input gradient reads the forward pass's plan, and a second plan costs more than the tile gains (training on new coordinates,
    // the forward pass alone on this tile, 5 x 1 x 1, 19 650 128 -> 128 182 189, 7 x 1 x 1 180 193; on both 181 178, 180 181; 128 -> 96, whose gradient kept its own, 182 204).
    const int least = std::min(Ci, Co), most = std::max(Ci, Co);
    if (V > 4 && V <= 8 && out->stream && least >= 128 && n * cdiv(most, 128) <= (most <= 128 ? 36864u : 49152u) && stream_lds_fits(256, 128, 128, most)) {
        *out = fgx_schedule{64, 128, 128, 1, 0, 1};
        return;
    }
    if (out->stream) return;
    // (not for an input gradient of a single tile of rows under a small weight: 192 voxels, 256 <- 768 channels 0.029 ms, 64 x 64 tiles 0.023)
    if (row_bytes >= 1024 && cols >= 128 && !(pass_kind != 0 && n < 256 && (size_t)K * cols < (size_t)512 * 512)) {
        // Too few tiles to stream and rows of 1 KiB or more (512 channels of a 16-bit type): a few hundred or thousand voxels
        // under a weight of tens of megabytes.  The tiled kernel on 256 x 128 tiles and 128-byte slabs, with as many K
        // splits as give every CU one workgroup, keeps more of the weight in flight than 128 x 128 tiles on 64-byte slabs
        // (measured forward, C = 1024: 192 voxels 0.048 -> 0.042 ms, 848 voxels 0.090 -> 0.084, 1 976 voxels 0.227 -> 0.138;
        // C = 512: 1 976 voxels 0.073 -> 0.054, 3 840 voxels 0.094 -> 0.085, 5 816 voxels 0.145 -> 0.133; at C = 256 the
        // smaller tiles are level).
        out->tile_rows = 256;
        out->tile_cols = 128;
        out->slab_bytes = 128;
        const size_t wide_items = (size_t)cdiv(n ? n : 1, 256) * cdiv(cols, 128);
        int sk = 1;
        while (wide_items * (size_t)sk * 2 <= (size_t)kCUs && sk < 32) sk *= 2;
        out->splitk = sk;
    }
}

}  // namespace
}  // namespace fgx

using namespace fgx;


// Weight gradient of few voxels, 16-bit types: the streaming kernel in one voxel block, which stores straight into the gradient, is
// ahead of the table's tiled kernel from the smallest layers on -- in 64 x 64 tiles, also where 32 x 32 ones would do (their four
// partial products want a reduction), in 128 x 128 ones under a weight of 512 x 512 channels and more.  Measured (us, table -> this):
// C = 16: 14 voxels 10.4 -> 5.6, 301 14.3 -> 7.0 (32 x 32 tiles: 9.6 and 10.2);  C = 64: 33 voxels 11.0 -> 5.6, 464 14.6 -> 8.3;
// C = 128: 14 voxels 15.2 -> 5.9, 464 22.0 -> 8.8;  C = 256: 91 voxels 17.1 -> 8.1, 464 22.9 -> 11.5;  C = 512: 33 voxels 18.7 -> 12.4
// (64 x 64: 14.1).  From 512 voxels on the table streams by itself.
extern "C" int fgx_wgrad_short_tile(int dtype, size_t n, int Ci, int Co) {
    if ((dtype != FGX_F16 && dtype != FGX_BF16) || n == 0 || n >= 512) return 0;
    return (size_t)Ci * Co >= (size_t)512 * 512 ? 128 : 64;
}

// fp32 weight gradient over the even split (fgx_conv_wgrad_split), in 96 x 96 tiles where they pad no more than 64 x 64 ones.  Its
// large tile multiplies at about twice the rate of the 32 x 32 one, which stays where it pads to less than half (32 channels,
// 49 829 voxels 0.048 ms, split 0.057;  32 -> 64 channels, half, 0.081 and 0.057, 448 584 voxels 0.400 and 0.347).  Two voxel blocks under few
// tiles, one otherwise: a block adds segments, and rows are read from L2 fast enough either way.
// Measured (us, tiled kernel on the fp32 units -> the split in three parts):  one 64 x 64 tile: 64 channels, 10 494 voxels 27 -> 28, 277 018 316 -> 224,
// 448 584 464 -> 354;  48 channels, 277 018 382 -> 225;  two: 112 -> 48 channels, 101 586 294 -> 169, 448 584 1 041 -> 690;  four: 128 channels, 101 586
// 390 -> 305, 166 977 595 -> 520, 448 584 1 533 -> 1 482, 635 497 2 161 -> 2 190;  25: 320 channels, 1 456 voxels 73 -> 55, 10 494 313 -> 232, 101 586 2 053 -> 1 981;  64: 512
// channels, 1 456 122 -> 112, 10 494 701 -> 553, 25 488 1 332 -> 1 196;  96 x 96: 96 channels, 2 581 39 -> 34, 667 763 2 330 -> 1 020.
// Sixteen tiles past 12 288 voxels, and four and more of 96 x 96 past 262 144, stay where they were.
extern "C" int fgx_wgrad_split_tile(size_t n, int Ci, int Co, int* block_rows) {
    if (n == 0 || Ci <= 0 || Co <= 0 || block_rows == nullptr || (size_t)Ci * Co >= (size_t)1024 * 1024) return 0;
    auto padded = [&](int t) { return (double)cdiv(Ci, t) * t * cdiv(Co, t) * t; };
    const int t = padded(96) <= padded(64) ? 96 : 64;
    const size_t tiles = (size_t)cdiv(Ci, t) * cdiv(Co, t), any = ~(size_t)0;
    const size_t least = t == 96 ? 2048 : tiles == 1 ? 4096 : tiles > 16 ? 1024 : 2048;
    const size_t most = t == 96 ? (tiles >= 4 ? 262144 : any) : tiles < 4 ? any : tiles < 16 ? 524288 : tiles == 16 ? 12288 : 131072;
    if (padded(32) <= 0.45 * padded(t) || n < least || n > most) return 0;
    *block_rows = (int)std::min(round_up(cdiv(n, (size_t)(tiles < 4 ? 2 : 1)), 64), (size_t)1 << 30);
    return t;
}

// The sweep multiplies row numbers with 24-bit multiplies and addresses both operands and the pair lists with 32-bit byte offsets.
extern "C" int fgx_wgrad_sweep_fits(size_t n, size_t n_in, int Ci, int Co, int elem_bytes, size_t n_pairs) {
    const double most = (double)0xFF000000u;
    return n > 0 && n <= ((size_t)1 << 24) && n_in <= ((size_t)1 << 24) && n_pairs > 0 && (double)n * Co * elem_bytes <= most &&
           (double)n_in * Ci * elem_bytes <= most && (double)n_pairs * 4 + 256 <= most;
}

extern "C" int fgx_wgrad_schedule(int dtype, size_t n, size_t n_in, uint32_t n_pairs, int Ci, int Co, int V, fgx_schedule* out) {
    const int rc = fgx_table_lookup(2, dtype, n, Ci, Co, V, out);
    if (rc != FGX_OK) return rc;
    int rows = 1024;
    if (dtype == FGX_F32) {
        const int tile = out->stream == 0 ? fgx_wgrad_split_tile(n, Ci, Co, &rows) : 0;
        if (tile != 0 && fgx_conv_wgrad_split_scratch_bytes(n, n_in, n_pairs, V, Ci, Co, tile, rows) > 0) *out = fgx_schedule{tile, tile, 64, 1, rows, 3};
    } else if (out->stream == 0) {
        if (const int tile = fgx_wgrad_short_tile(dtype, n, Ci, Co)) *out = fgx_schedule{tile, tile, 64, 1, rows, 1};
    } else if (out->stream == 2 && !fgx_wgrad_sweep_fits(n, n_in, Ci, Co, 2, n_pairs)) {       // very long operands, and empty pair lists
        out->stream = 1;
        out->block_rows = 12288;
    }
    return FGX_OK;
}

extern "C" int fgx_table_lookup(int pass_kind, int dtype, size_t n, int Ci, int Co, int V, fgx_schedule* out) {
    FGX_CHECK_ARG(out != nullptr, "fgx_table_lookup: null output");
    FGX_CHECK_ARG(pass_kind >= 0 && pass_kind <= 2, "fgx_table_lookup: pass_kind must be 0 (fwd), 1 (dgrad) or 2 (wgrad)");
    FGX_CHECK_ARG(dtype == FGX_F16 || dtype == FGX_BF16 || dtype == FGX_F32, "fgx_table_lookup: unknown dtype %d", dtype);
    FGX_CHECK_ARG(Ci > 0 && Co > 0 && V >= 1, "fgx_table_lookup: bad shape");
    const int es = dtype == FGX_F32 ? 4 : 2;
    const int l2 = floor_log2(n ? n : 1);
    for (const Entry& e : kTable) {
        if (e.pass_kind == pass_kind && (e.dtype_bytes == 0 || e.dtype_bytes == es) && e.log2n == l2 && e.ci == Ci && e.co == Co) {
            *out = e.s;
            if (pass_kind != 2 && out->stream && !stream_lds_fits(out->tile_rows, out->tile_cols, out->slab_bytes, pass_kind == 0 ? Co : Ci))
                break;      // (cannot happen for the shapes listed; the rule decides then)
            return FGX_OK;
        }
    }
    rule(pass_kind, es, n, Ci, Co, V, out);
    return FGX_OK;
}
