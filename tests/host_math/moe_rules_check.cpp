// Host check of the rule by which the expert layer takes its kernels for many rows per expert (aiter_amd/csrc/moe_rules.h).
// Prints OK or the first failed expectation.
#include "../../aiter_amd/csrc/moe_rules.h"

#include <cstdio>
#include <initializer_list>

#define EXPECT(cond)                                                                             \
    do                                                                                           \
    {                                                                                            \
        if(!(cond))                                                                              \
        {                                                                                        \
            std::printf("FAILED line %d: %s (tokens %d, experts %d)\n", __LINE__, #cond, m, e);  \
            return 1;                                                                            \
        }                                                                                        \
    } while(0)

using namespace fp8bs;

// a layer of the widest dim that was measured
static bool tiles_win(int64_t pairs, int64_t all, int held, int inter) { return fp8bs::tiles_win(pairs, all, held, inter, 7168); }

// slots as the sort's arrays are sized, in whole blocks
static int64_t padded(int64_t pairs, int topk, int unit, int all) { return (pairs + (int64_t)all * unit - topk) / unit * unit; }

int main()
{
    int m = 0, e = 0;
    for(int unit : {32, 64, 128})
        for(int topk : {1, 2, 5, 8})
            for(m = 1; m < 9000; m += 37)
                for(int all : {8, 33, 256, 1000})
                    for(int held : {1, all / 8, all / 2, all})
                    {
                        const int64_t pairs = (int64_t)m * topk, p = padded(pairs, topk, unit, all);
                        e = held;
                        EXPECT(routed_experts(pairs, topk, unit, p, e) == all);
                        // arrays that say less than the weights: the experts held are the least there are
                        EXPECT(routed_experts(pairs, topk, unit, pairs / unit * unit, 1000) == 1000);
                        // a rank that holds a part of the experts sees the rows per expert of the whole: no more tiles than
                        // with all of them, whatever its own part
                        for(int inter : {128, 256, 512, 2048})
                            if(tiles_win(pairs, all, e, inter))
                                EXPECT(tiles_win(pairs, all, all, inter));
                    }
    // 32 of 256 experts held: a decode batch of 64 tokens has two rows per expert, not sixteen
    e = 32;
    for(m = 1; m <= 512; ++m)
        EXPECT(!tiles_win((int64_t)m * 8, routed_experts((int64_t)m * 8, 8, 32, padded((int64_t)m * 8, 8, 32, 256), e), e, 2048));
    m = 8192;
    EXPECT(tiles_win((int64_t)m * 8, 256, e, 256) && tiles_win((int64_t)m * 8, 256, 256, 256));
    // parts of the second GEMM's columns: at least one, never more than the workgroup's waves have groups for
    for(e = 1; e <= 512; e += 7)
        for(m = 1; m <= 4096; m = m * 2 + 1) // rows per expert
            for(int groups = 4; groups <= 256; groups += 4)
            {
                const int splits = down_col_splits(m, e, groups, 4);
                EXPECT(splits >= 1 && splits * 4 <= groups);
            }
    // Few tokens: rows through memory where a narrow layer leaves the column kernel few workgroups, columns for the rest.  A rank that
    // holds a part of the experts counts its own pairs
    m = 140, e = 64;
    EXPECT(rows_beat_columns(140 * 6, 64, 64, 1536, 128) && !rows_beat_columns(140 * 6, 64, 64, 512, 128));
    EXPECT(!rows_beat_columns(16 * 8, 256, 256, 7168, 256) && !rows_beat_columns(128 * 8, 256, 256, 7168, 256));
    EXPECT(!rows_beat_columns(5, 32, 32, 1024, 256) && !rows_beat_columns(140 * 6, 64, 4, 1536, 128));
    // the six layers whose bits test_fmoe_few_tokens_take_columns_or_rows compares: which side they are on
    EXPECT(rows_beat_columns(140 * 6, 64, 64, 1536, 128) && rows_beat_columns(29 * 8, 256, 256, 1024, 128) && rows_beat_columns(270 * 3, 5, 5, 1280, 256));
    EXPECT(!rows_beat_columns(140 * 6, 64, 64, 768, 128) && !rows_beat_columns(16 * 8, 64, 64, 5120, 256) && !rows_beat_columns(3 * 5, 32, 32, 1024, 256));
    // and the ones beyond 32 MiB of rows
    EXPECT(rows_beat_columns(540 * 8, 64, 64, 3584, 128) && rows_beat_columns(400 * 8, 256, 256, 3072, 128));
    // Tiles on both sides of where they were measured to win: (rows per expert, experts, dim, inter)
    auto tiles = [](int rows, int experts, int dim, int inter) { return fp8bs::tiles_win((int64_t)rows * experts, experts, experts, inter, dim); };
    struct
    {
        int experts, dim, inter, no, yes;
    } const lines[] = {
        {256, 3072, 128, 40, 56},  {256, 7168, 256, 40, 52},  {128, 7168, 256, 48, 56},  {32, 4096, 256, 48, 64}, {8, 1024, 256, 240, 384},
        {256, 2048, 512, 22, 32},  {16, 4096, 2048, 12, 24},  {64, 1536, 256, 26, 49},   {128, 1280, 128, 24, 36}, {64, 1024, 384, 18, 25},
        {32, 7168, 1024, 24, 48},  {128, 4096, 384, 38, 40},  {96, 4096, 384, 38, 40},   {80, 3072, 384, 34, 38},
        {16, 4096, 256, 104, 118}, {8, 3840, 512, 108, 117},  {12, 6144, 384, 95, 112},  {24, 2304, 256, 59, 64},  {8, 6144, 128, 560, 580},
    };
    for(auto& l : lines)
    {
        m = l.dim, e = l.experts;
        EXPECT(!tiles(l.no, l.experts, l.dim, l.inter) && tiles(l.yes, l.experts, l.dim, l.inter));
    }
    // a narrower layer takes tiles from no more rows than a wide one
    for(int inter : {128, 256, 512, 1024})
        for(e = 8; e <= 256; e *= 2)
            for(int rows = 8; rows <= 1024; rows += 8)
                for(m = 1024; m < 7168; m += 512)
                    EXPECT(tiles(rows, e, m, inter) || !tiles(rows, e, m + 512, inter));
    std::printf("OK\n");
    return 0;
}
