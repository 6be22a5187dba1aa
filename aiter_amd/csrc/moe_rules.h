// When the expert layer takes the kernels for many rows per expert (moe_prefill.hip).  Plain C++ (no HIP), so that the rule can
// be compiled and tested on the host.
#pragma once

#include <math.h>
#include <stdint.h>

namespace fp8bs {

constexpr int kTileRowsOfExpert = 128; // most rows of one expert in a tile

// The experts that the tokens' `pairs` = tokens x topk were routed to, of which `experts` are held here.  An expert-parallel
// rank sorts with all of them and holds a part; how many pairs are its own only the device knows, but the sorted arrays are
// sized for every expert's last block (pairs + all x unit - topk slots; padded: that in whole blocks).
inline int64_t routed_experts(int64_t pairs, int topk, int unit, int64_t padded, int experts)
{
    const int64_t all = (padded - pairs + topk + unit - 1) / unit;
    return all > experts ? all : experts;
}

// Tiles win where an expert has enough rows that the block-wise kernels' repeated passes over its weights cost more than a
// tile's padding -- fewer with a longer K of the second GEMM, where those kernels have nothing in flight while they multiply, and
// fewer on narrower layers, whose items are shorter -- and where there are enough items (a tile's 128 columns of the product;
// an expert's last tile is half full on average) for the chip.  Over 211
// layers (8 to 256 experts, 12 to 1024 rows each, dim 1024 to 7168, 150 of them drawn) this takes 1.2 % longer than the better of
// the two on average, 5 % and more in 20, 26 % at worst; with the first condition alone 3.8 %, 52 and 31 %.  us block by block / in tiles (experts, topk, dim, inter):
//   (256, 8, 3072, 128)  40 rows per expert (208 items): 128 / 130, 56 (240): 153 / 141, 128: 283 / 196
//   (256, 8, 7168, 256)  40 (416): 402 / 408, 52: 462 / 426, 64: 530 / 441, 256: 1652 / 900
//   (128, 8, 7168, 256)  48 (224): 228 / 257, 56 (240): 254 / 259, 64: 277 / 260, 96: 365 / 288
//   (32, 5, 4096, 256)   48 (56): 61 / 61, 64 (64): 76 / 62, 112: 92 / 64, 160: 119 / 68
//   (8, 2, 1024, 256)    384 (56): 43 / 40, 512 (72): 52 / 41, 1024: 72 / 49
//   (128, 8, 4096, 384)  40 (312): 168 / 188, 48 (336): 187 / 184, 128: 377 / 252
//   (256, 8, 2048, 512)  24 (704): 190 / 195, 32 (768): 219 / 212, 256: 1016 / 492
//   (64, 6, 7168, 512)   48 (224): 218 / 240, 64 (256): 267 / 247, 80: 298 / 248
//   (32, 8, 7168, 1024)  32 (192): 182 / 195, 48 (224): 212 / 186, 128: 394 / 261
//   (16, 4, 4096, 2048)  16 (160): 88 / 95, 24 (176): 116 / 100, 128: 257 / 140
//   (32 held of 256, 8, 7168, 2048)  2: 197 / 238, 16 (320): 301 / 286, 32 (384): 340 / 326, 256: 2004 / 865
//   (64 held of 256, 8, 4096, 1024)  16: 180 / 190, 32 (384): 210 / 190, 64: 321 / 227
// Below 48 items the line depends on how full the tiles are: an expert with a hundred rows or fewer has one ragged tile, and a chip
// that is a sixth full waits for the longest of them.  Time block by block over time in tiles, fewer than 112 rows: (322, 12
// experts, top-3, 6144, 384; 40 items) 0.84, (415, 16, 4, 4096, 256; 41) 0.92, (432, 8, 2, 3840, 512; 43) 0.92, (355, 24, 4, 2816, 256; 46)
// 0.96, (430, 12, 3, 4096, 384; 48) 1.10; more: (604, 12, 3, 2816, 256; 40) 0.94, (638, 12, 3, 6912, 256; 41) 1.10, (474, 16, 4, 5120, 256;
// 45) 1.17, (2362, 8, 2, 6144, 128; 40) 1.23.
// Three K blocks of the second GEMM (inter 384) take the ring there, and with 0.8 to 1.25 rounds of items need more rows to make up for
// it: (608, 96, 6, 4096; 229 items) 0.87, (618, 128, 8, 4096; 308) 0.94, (476, 112, 8, 3072; 257) 0.96, (380, 80, 8, 3072; 191) 1.21.
// (The average over 211 layers is from before these two.)
// `all`: the experts that the pairs are spread over, as routed_experts says.
inline bool tiles_win(int64_t pairs, int64_t all, int experts, int inter, int dim)
{
    const double rows  = (double)pairs / (double)all;
    const double items = (rows / kTileRowsOfExpert + 0.5) * experts * (inter / 128);
    const double least = inter <= 128 ? 80.0 : inter <= 256 ? 64.0 : inter <= 512 ? 40.0 : inter <= 1024 ? 28.0 : 24.0;
    if(rows >= least && items >= 80.0)
        return true;
    // fewer rows where the items fill the chip and are short
    const double filled = (items < 256.0 ? items : 256.0) / 256.0;
    const double fewest = rows >= 256.0 ? 40.0 : rows >= 112.0 ? 41.0 : 48.0;
    const double ring   = inter == 384 && items > 205.0 && items < 320.0 ? 1.2 : 1.0;
    return items >= fewest &&
           rows * pow(filled, 0.3) > 22.5 * ring * sqrt((dim > 1024 ? dim : 1024) / 1024.0) * pow(128.0 / (inter < 1024 ? inter : 1024), 0.2);
}

// Second GEMM with its rows in LDS: the parts that a tile's groups of 64 columns are cut into, one item each, of which the
// workgroup's waves take a group at a time.  More items fill 512 workgroups evenly and keep more requests in flight, but each
// brings the tile's rows into LDS.  us with 7, 4, 2 and 1 groups per wave (tokens, experts, topk, dim, inter; items with one):
//   (1000, 32, 5, 5120, 256)   1160: 39 / - / 24 / 22     (2500, 40, 6, 4352, 256)  2400: 64 / 58 / 54 / 46
//   (2795, 64, 6, 2816, 256)   1826: 59 / - / 41 / 36     (1184, 8, 2, 6400, 128)    500: 27 / 17 / 15 / 12
//   (5184, 256, 8, 2048, 256)  3616: 75 / 68 / 71 / 69    (3000, 128, 8, 4096, 128) 4000: 58 / 53 / 52 / 55
//   (2048, 256, 8, 7168, 256)  7170: 156 / - / 144 / 142  (4096, 256, 8, 4096, 256) 6140: 123 / 108 / 109 / 117
//   (8192, 256, 8, 3072, 128)  7680: 115 / 98 / 92 / 95   (8192, 256, 8, 7168, 256) 17920: 304 / - / 307 / 327
inline int down_col_splits(double rows_per_expert, int experts, int groups, int waves)
{
    const double tiles = (rows_per_expert / kTileRowsOfExpert + 0.5) * experts; // an expert's last one is half full on average
    auto splits = [&](int per_wave) { return groups <= per_wave * waves ? 1 : (groups + per_wave * waves - 1) / (per_wave * waves); };
    if(tiles * splits(1) <= 3800.0)
        return splits(1);
    if(tiles * splits(2) <= 5000.0)
        return splits(2);
    return groups <= 7 * waves ? 1 : groups / (7 * waves);
}

// Whether few tokens' rows, kept in fp32, go through memory to a kernel of their own for the per-token sum, where the kernel that owns
// 32 columns and sums in LDS would fit too.  That one walks every block of rows in each of its dim / 32 workgroups: a block's
// K block takes it 0.13 us, more than memory needs for all columns' weights below dim 5000, and a pair of token and expert
// 0.02 us; rows through memory cost a launch (with some margin 6.5 us), are written and read, and their weights arrive 6 % more slowly.
// Over 100 drawn layers (1 to 300 tokens, inter 128 and 256) this takes 0.5 % longer than the better of the two on average and 14 %
// at worst, where columns stay.  us in columns / through memory, sort excluded (tokens, experts, topk, dim, inter):
//   (140, 64, 6, 1536, 128)  47 / 35    (204, 64, 6, 3840, 128)  64 / 53    (29, 256, 8, 1024, 128)  47 / 30
//   (295, 128, 8, 4096, 256) 169 / 109  (18, 256, 8, 1280, 256)  48 / 38    (61, 256, 8, 3840, 256) 114 / 107
//   (16, 256, 8, 7168, 256)  89 / 94    (128, 256, 8, 7168, 256) 199 / 213  (66, 256, 8, 4864, 256) 131 / 133
//   (1, 256, 8, 1024, 256)   17 / 20    (3, 32, 5, 6400, 256)    24 / 26    (110, 256, 8, 5376, 256) 164 / 168
// and whole layers, whose rows take more than 32 MiB and wait in fp32 all the same:
//   (400, 256, 8, 2304, 128) 146 / 92   (554, 128, 8, 3840, 128) 160 / 121  (264, 256, 8, 4608, 256) 198 / 183
//   (270, 64, 6, 7168, 256)  127 / 128
// Measured from dim 1024 on; below, columns as long as they fit.
inline bool rows_beat_columns(int64_t pairs, int64_t all, int experts, int dim, int inter)
{
    if(dim < 1024)
        return false;
    const double rows = (double)pairs / (double)all, here = rows * experts, kblocks = inter / 128;
    const double blocks  = experts * (1.0 - exp(-rows)) + here / 32.0; // an even routing's, of up to 32 rows each
    const double weights = dim * 25.6e-6;                              // us per block and K block, at 5 TB/s
    const double in_columns = blocks * kblocks * (weights < 0.13 ? 0.13 - weights : 0.0) + here * 0.02;
    return in_columns > 6.5 + here * dim * 2.1e-6 + blocks * kblocks * weights * 0.06;
}

} // namespace fp8bs
