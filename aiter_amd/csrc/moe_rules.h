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
// tile's padding -- fewer with a longer K of the second GEMM, where those kernels have nothing in flight while they multiply --
// and where there are enough items (a tile's 128 columns of the product; an expert's last tile is half full on average) for
// the chip.  Over 1139 drawn layers (5 to 256 experts, 8 to 1200 rows each, dim 1024 to 7168) this takes 0.5 % longer than
// the better of the two on average, 5 % and more in 43 and 23 % at worst.  us block by block / in tiles (experts, topk, dim,
// inter):
//   (256, 8, 3072, 128)  64 rows per expert (256 items): 181 / 198, 80 (288): 215 / 206, 128: 299 / 236
//   (256, 8, 7168, 256)  48 (448): 468 / 490, 52: 494 / 479, 64: 553 / 515, 256: 1724 / 1044
//   (128, 8, 7168, 256)  64 (256): 294 / 319, 80 (288): 342 / 341, 96: 385 / 343
//   (32, 5, 4096, 256)   96 (80): 92 / 106, 112 (88): 109 / 108, 160: 137 / 113
//   (8, 2, 1024, 256)    640 (88): 72 / 75, 768 (104): 79 / 75, 1024: 88 / 77
//   (128, 8, 4096, 384)  48 (336): 208 / 214, 56 (360): 231 / 212, 128: 392 / 291
//   (256, 8, 2048, 512)  32 (768): 241 / 254, 40 (832): 273 / 255, 256: 1055 / 609
//   (64, 6, 7168, 512)   48 (224): 238 / 275, 64 (256): 283 / 291, 80: 328 / 296
//   (32, 8, 7168, 1024)  32 (192): 183 / 198, 48 (224): 207 / 192, 128: 414 / 291
//   (16, 4, 4096, 2048)  32 (192): 121 / 112, 128: 284 / 180
//   (32 held of 256, 8, 7168, 2048)  2: 245 / 273, 16 (320): 293 / 299, 32 (384): 396 / 319, 256: 1635 / 815
//   (64 held of 256, 8, 4096, 1024)  16: 187 / 219, 32 (384): 226 / 229, 64: 337 / 252
// `all`: the experts that the pairs are spread over, as routed_experts says.
inline bool tiles_win(int64_t pairs, int64_t all, int experts, int inter)
{
    const double rows  = (double)pairs / (double)all;
    const double items = (rows / kTileRowsOfExpert + 0.5) * experts * (inter / 128);
    const double least = inter <= 128 ? 80.0 : inter <= 256 ? 64.0 : inter <= 512 ? 40.0 : inter <= 1024 ? 28.0 : 24.0;
    return rows >= least && items >= 80.0;
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
// Measured from dim 1024 on; below, columns as long as they fit.
inline bool rows_beat_columns(int64_t pairs, int64_t all, int experts, int dim, int inter)
{
    if(dim < 1024)
        return false;
    const double rows = (double)pairs / (double)all, here = rows * experts, kblocks = inter / 128;
    const double blocks  = experts * (1.0 - exp(-rows)) + here / 32.0; // an even routing's, of up to 32 rows each
    const double weights = dim * 25.6e-6;                              // us per block and K block, at 5 TB/s
    const double in_columns = blocks * kblocks * (weights < 0.13 ? 0.13 - weights : 0.0) + here * 0.02;
    return in_columns > 6.5 + here * dim * 2e-6 + blocks * kblocks * weights * 0.06;
}

} // namespace fp8bs
