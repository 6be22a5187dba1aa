// Host check of where bands of weight rows carry out a GEMM (aiter_amd/csrc/gemm_rules.h).  Prints OK or the first failed expectation.
#include "../../aiter_amd/csrc/gemm_rules.h"

#include <cstdio>

#define EXPECT(cond)                                                                                                              \
    do                                                                                                                            \
    {                                                                                                                             \
        if(!(cond))                                                                                                               \
        {                                                                                                                         \
            std::printf("FAILED line %d: %s (m %d, n %d)\n", __LINE__, #cond, m, n);                                              \
            return 1;                                                                                                             \
        }                                                                                                                         \
    } while(0)

using namespace fp8bs;

int main()
{
    int  m = 0, n = 0;
    auto rows = [](int M, int N, int K, bool over_192 = false) { return gemm_band_rows(M, N, K, over_192, 256); };
    // 144: a second round of 128-row tiles, none of its own; from 65 rows on
    EXPECT(rows(203, 36864, 7168, true) == 144 && rows(65, 32772, 128) == 144 && rows(64, 32772, 128) == 0);
    EXPECT(rows(200, 32768, 1024) == 0 && rows(200, 32769, 1024) == 144 && rows(200, 36864, 1024) == 144 && rows(200, 36865, 1024) == 0);
    EXPECT(rows(257, 16400, 1152) == 144 && rows(512, 16384, 1152) == 0 && rows(2044, 4480, 8320) == 144 && rows(1000, 9216, 512) == 144);
    // not in place of 192-row tiles that fit exactly, up to eight K blocks, unless bands of 144 do, too
    for(int k = 128; k <= 1024; k += 128)
    {
        EXPECT(rows(4096, 2112, k, true) == 0 && rows(1024, 8256, k, true) == 0 && rows(256, 35904, k, true) == 0);
        EXPECT(rows(4096, 2112, k, false) == 144 && rows(3840, 2304, k, true) == 144 && rows(4096, 2096, k, true) == 144);
    }
    EXPECT(rows(4096, 2112, 1152, true) == 144 && rows(1024, 8256, 7168, true) == 144);
    // 96: two thirds of the chip up to all of it, 40 K blocks, one tile of rows
    for(m = 25; m <= 256; m += 33)
    {
        for(n = 16400; n <= 24576; n += 146 * 4)
            EXPECT(rows(m, n, 5120) == 96 && rows(m, n, 4992) == 0);
        EXPECT(rows(m, 24580, 5120) == 0 && rows(m + 256, 7000, 7168) == 0);
        // ... but where two columns of 128-row tiles are a round that fills the chip
        for(n = 16320; n <= 16384; n += 16)
            EXPECT(rows(m, n, 5120) == 0 && rows(m, n, 8064, m > 128) == 0);
    }
    // fewer rows: only with weights that are read past the caches
    for(m = 1; m <= 24; ++m)
        EXPECT(rows(m, 22480, 5248) == 0 && rows(m, 24576, 5376) == 0 && rows(m, 24576, 5504) == 96 && rows(m, 24288, 6400) == 96);
    EXPECT(gemm_band_streams_weights(256, 32768, 4096) && !gemm_band_streams_weights(256, 32767, 4096) && !gemm_band_streams_weights(257, 32768, 4096));
    std::printf("OK\n");
    return 0;
}
