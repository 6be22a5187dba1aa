// Where the bands of weight rows of gemm_band.hip carry out a GEMM whose plan is one K range.  Plain arithmetic on sizes, so that it
// can be compiled and tested on the host.
#pragma once

#include <stdint.h>

namespace fp8bs {

constexpr int kBandRows = 256; // activation rows of a band's tile

// Weights that one workgroup reads, and that take more than half of the last-level cache, are read past the caches, which the rows
// then have for themselves (64 x 36864 x 7168: 50 us, 44 this way; 203 rows 74 and 71).
inline bool gemm_band_streams_weights(int64_t M, int64_t N, int64_t K)
{
    return M <= kBandRows && N * K >= (int64_t)128 << 20;
}

// The rows of weights per workgroup, 144 or 96, or 0 where what was chosen stays.  over_192: that is 256 x 192 tiles.  us of what was
// chosen / here.
//
// 144 where tiles of 128 rows take a second round of workgroups and these do not: over 149 drawn sizes 1 to 64 % ahead (75 x 34496 x 1920
// 28 / 17, 2044 x 4480 x 1024 18 / 15, 3841 x 2112 x 256 12.6 / 9.8) but for the exception below; where 128 fit one round as well, up
// to 24 % behind gemm_ring.hip's.  From 65 rows on: up to 64, one row of 64 x 64 tiles, two of them on a compute unit, reads the
// weights once as well (34 x 32960 x 512: 7.8 / 9.1).
//   Not in place of 192-row tiles that N is a multiple of, while it is none of 144, up to eight K blocks: those store whole tiles, and
//   the bands' gain per K block does not make up for the ragged one.  One to six K blocks 0 to 9 % behind (4096 x 2112 x 256 9.7 /
//   10.4, 1024 x 8256 x 256 9.3 / 10.3, 2048 x 4224 x 640 12.4 / 12.7), seven even (1280 x 6720 x 896 15.0 / 14.9), ten 3 to 13 % ahead
//   (2048 x 4224 x 1280 18.5 / 17.5).  Eight would be 2 to 9 % ahead (4096 x 2112 x 1024 16.3 / 15.9) and stay: that size is one that
//   callers are told takes 192-row tiles.  With N a multiple of both, bands are ahead at one K block (3840 x 2304 x 128 8.5 / 8.0).
//
// 96 for up to 256 rows and 40 K blocks or more where that covers two thirds of the chip, in place of tilings that read
// the weights more than once or cover less of it: 68 x 21632 x 5760 30.3 / 28.6, 151 x 17984 x 5504 41.4 / 37.4,
// 130 x 20480 x 6144 43.3 / 38.7, 100 x 24576 x 7168 44.9 / 39.4; with fewer K blocks 110 x 17984 x 2432 13.8 / 15.0, 256 x 16512 x
// 2560 19.0 / 22.0, on less of the chip 37 x 14464 x 2688 (151 workgroups) 11.2 / 13.7, for more rows 392 x 7872 x 6272 31 / 38.
//   Not where two columns of tiles of 128 weight rows are one round that fills the chip: 256 x 16384 x 8064 52 / 65, 64 x 16384 x 5120
//   21.7 / 25.8; 65 x 16400 x 5120 29.8 / 26.5.
//   From 25 rows on, or where the weights are read past the caches: 1 x 22480 x 5248 22.1 / 23.8, 8 x 22000 x 6016 26.4 / 27.7, 24 x
//   24576 x 5248 25.6 / 26.1; 28 x 19568 x 6784 30.6 / 29.8, 48 x 22784 x 5248 28.8 / 27.1; 1 x 24288 x 6400 31.2 / 30.3, 8 x 24576 x
//   7168 32.4 / 29.7.
inline int gemm_band_rows(int64_t M, int64_t N, int64_t K, bool over_192, int cus)
{
    const int64_t tiles_m = (M + kBandRows - 1) / kBandRows, kblocks = K / 128;
    auto tiles = [&](int rows) { return tiles_m * ((N + rows - 1) / rows); };
    if(M > 64 && tiles(128) > cus && tiles(144) <= cus)
        return over_192 && N % 192 == 0 && N % 144 != 0 && kblocks <= 8 ? 0 : 144;
    if(tiles_m == 1 && kblocks >= 40 && tiles(96) <= cus && tiles(96) * 3 >= cus * 2 && 2 * tiles(128) > cus &&
       (M > 24 || gemm_band_streams_weights(M, N, K)))
        return 96;
    return 0;
}

} // namespace fp8bs
