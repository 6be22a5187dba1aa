// Block-scale FP8 GEMM, up to 256 activation rows by a band of 96 or 144 weight rows per workgroup: one round of workgroups
// that covers the chip where 128-row tiles do not.
//
// Carries out, where it is faster (gemm_rules.h), what was chosen for other kernels with K in one range; the additions are the same,
// so the bits are too.  By name it takes any size that the prefill_* kernels take.
//
// Why bands of 144.  With 256 rows of weights per workgroup 36864 of them are 144 workgroups, with 192 they are 192, with 128
// a round and a fragment of one; with 144 they are 256, and a workgroup's K block is 18 KiB of weights beside the rows'.
//
// Why two rings.  The rows come from L2, the weights from memory, and a wave's loads are counted in the order they were issued: with
// fetching waves of its own (two and two) each operand waits for its own depth only, and has a ring of its own.  The rows keep three
// stages; the weights take what is left, up to six: bands of 144 four or more up to 208 rows (224 with scales that come K block by K
// block), three beyond, where both operands are two K blocks ahead, as in gemm_ring.h.  The gain over other tilings does not
// end there: 203, 224, 240 and 256 x 36864 x 7168 take 62.9, 64.1, 66.7 and 67.8 us, so most of it is the covered chip.
//
// Bound by, with few rows, the weights (64 x 36864 x 7168 by name: 45 us, 5.9 TB/s); beyond, by what a compute unit takes in and
// multiplies per K block.  us of 192-wide tiles or mid_128x128, K in one range / here, calls in a loop over several copies of the weights
// (among calls of other kinds 203 x 36864 x 7168 takes 104 / 72):
//   203 x 36864 x 7168 102 / 63   512 x 18432 x 7168 94 / 66   1024 x 9216 x 7168 87 / 64   75 x 34496 x 1920 26 / 17
//   86 x 35136 x 1152 18 / 13     288 x 17024 x 2816 39 / 25   2044 x 4480 x 1024 17 / 15   1439 x 5760 x 3072 34 / 28
// Taken out again: two stages of rows (203 x 36864 x 7168 81 us among other calls: a K block then waits for L2).
#include "gemm_ring.h"
#include "gemm_rules.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace fp8bs {

namespace {

constexpr int kMulWaves = 8, kFetchWaves = 4; // two that fetch weights, two that fetch rows and their scales
constexpr int kBandThreads = 64 * (kMulWaves + kFetchWaves);
static_assert(kBandRows == 32 * kMulWaves, "32 rows per multiplying wave");
constexpr int kXStages     = 3; // K blocks of rows in LDS

struct BandLayout // LDS, in bytes
{
    int rows;       // activation rows of a tile: a multiple of 16
    int w_stages;   // K blocks of weights
    int w_at, xs_at, total;
    int stream_w;   // weights are read past the caches
};

#define FP8BS_MFMA(P, A, B) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=&v"(P) : "v"(A), "v"(B))
#define FP8BS_FMA4(ACC, P, S)                                                              \
    do                                                                                     \
    {                                                                                      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[0]) : "v"((P)[0]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[1]) : "v"((P)[1]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[2]) : "v"((P)[2]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[3]) : "v"((P)[3]), "v"(S));      \
    } while(0)

// All but this wave's `n` youngest loads have landed.  The instruction takes its count as a constant.
__device__ __forceinline__ void wait_all_but_few(int n)
{
    switch(n)
    {
    case 18: asm volatile("s_waitcnt vmcnt(18)" ::: "memory"); break;
    case 17: asm volatile("s_waitcnt vmcnt(17)" ::: "memory"); break;
    case 16: asm volatile("s_waitcnt vmcnt(16)" ::: "memory"); break;
    case 15: asm volatile("s_waitcnt vmcnt(15)" ::: "memory"); break;
    case 14: asm volatile("s_waitcnt vmcnt(14)" ::: "memory"); break;
    case 13: asm volatile("s_waitcnt vmcnt(13)" ::: "memory"); break;
    case 12: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
    case 11: asm volatile("s_waitcnt vmcnt(11)" ::: "memory"); break;
    case 10: asm volatile("s_waitcnt vmcnt(10)" ::: "memory"); break;
    case 9: asm volatile("s_waitcnt vmcnt(9)" ::: "memory"); break;
    case 8: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
    case 7: asm volatile("s_waitcnt vmcnt(7)" ::: "memory"); break;
    case 6: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
    case 5: asm volatile("s_waitcnt vmcnt(5)" ::: "memory"); break;
    case 4: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
    case 3: asm volatile("s_waitcnt vmcnt(3)" ::: "memory"); break;
    case 2: asm volatile("s_waitcnt vmcnt(2)" ::: "memory"); break;
    case 1: asm volatile("s_waitcnt vmcnt(1)" ::: "memory"); break;
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    }
}
template <int STEP> // n: a multiple of STEP up to 4 STEP
__device__ __forceinline__ void wait_all_but(int n)
{
    if(n == 0)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    else if(n == STEP)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STEP) : "memory");
    else if(n == 2 * STEP)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * STEP) : "memory");
    else if(n == 3 * STEP)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(3 * STEP) : "memory");
    else
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * STEP) : "memory");
}

// NF: fragments of 16 weight rows per tile (6 or 9).  SHUF, XS4: as in gemm_ring.h.
template <In16 DT, bool SHUF, bool XS4, int NF>
__global__ __launch_bounds__(kBandThreads) void gemm_band_kernel(GemmKernelParams p, int tiles_m, int tiles_n, BandLayout lds)
{
    static_assert(NF % 3 == 0, "three buffers of weight fragments in rotation");
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    constexpr int      BN = 16 * NF;
    constexpr uint32_t kWStage = BN * 128;
    const lds_byte_ptr smem3 = (lds_byte_ptr)smem;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int n = p.kblocks;

    // each XCD takes a contiguous eighth of the tiles (workgroups go round robin over the XCDs), tiles of the same weights
    // next to each other
    const int total = tiles_m * tiles_n, xcd = blockIdx.x & 7;
    const int lo = (int)((int64_t)total * xcd / 8), hi = (int)((int64_t)total * (xcd + 1) / 8);
    const int tile = lo + ((int)blockIdx.x >> 3);
    if(tile >= hi)
        return;
    const int m0 = (tile % tiles_m) * kBandRows, n0 = (tile / tiles_m) * BN;
    const uint32_t x_stage = (uint32_t)lds.rows * 128u;

    if(wave >= kMulWaves)
    {
        const int f = wave - kMulWaves;
        __builtin_amdgcn_s_setprio(3); // a K block's loads leave before the multiplying waves take the issue slots (1-4 us of 73)
        if(f < 2)
        {
            // weights: 2 NF loads of 8 rows (1 KiB) per K block, every other one
            uint32_t goff[NF];
#pragma unroll
            for(int i = 0; i < NF; ++i)
            {
                const uint32_t u = 2u * i + f, r = 8u * u + ((uint32_t)lane >> 3), chunk = ((uint32_t)lane & 7u) ^ lds_swizzle(r);
                if constexpr(SHUF)
                    goff[i] = min(((uint32_t)n0 >> 4) + (u >> 1), ((uint32_t)p.N >> 4) - 1u) * 16u * (uint32_t)p.K + (u & 1u) * 1024u + (uint32_t)lane * 16u;
                else
                    goff[i] = min((uint32_t)n0 + r, (uint32_t)p.N - 1u) * (uint32_t)p.ldb + chunk * 16u;
            }
            const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem3) + (uint32_t)lds.w_at + (uint32_t)f * 1024u;
            uint32_t stage = 0;
            auto issue = [&](int kb) { // past the end the last block again, unused, so that every K block has its loads
                const uint8_t* src = p.wq + (size_t)min(kb, n - 1) * (SHUF ? 2048 : 128);
                if(lds.stream_w)
                {
#pragma unroll
                    for(int i = 0; i < NF; ++i)
                        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt"
                                     :
                                     : "s"(base + stage * kWStage + (uint32_t)i * 2048u), "v"(goff[i]), "s"(src)
                                     : "memory");
                }
                else
                {
#pragma unroll
                    for(int i = 0; i < NF; ++i)
                        ring_dma16(base + stage * kWStage + (uint32_t)i * 2048u, goff[i], src);
                }
                stage = stage + 1 == (uint32_t)lds.w_stages ? 0 : stage + 1;
            };
            for(int kb = 0; kb < lds.w_stages - 1; ++kb)
                issue(kb);
            const int young = NF * (lds.w_stages - 2);
            wait_all_but<NF>(young);
            __syncthreads();
            for(int kb = 0; kb < n; ++kb)
            {
                issue(kb + lds.w_stages - 1);
                wait_all_but<NF>(kb + 1 < n ? young : 0);
                __syncthreads();
            }
        }
        else
        {
            // rows: rows / 8 loads per K block, every other one, and the scales of rows / 2 rows
            const int      g = f - 2, loads = lds.rows / 16;
            uint32_t       goff[kBandRows / 16], xs_goff[kBandRows / 128];
#pragma unroll
            for(int i = 0; i < kBandRows / 16; ++i)
            {
                const uint32_t u = 2u * i + g, r = 8u * u + ((uint32_t)lane >> 3), chunk = ((uint32_t)lane & 7u) ^ lds_swizzle(r);
                goff[i] = min((uint32_t)m0 + r, (uint32_t)p.M - 1u) * (uint32_t)p.lda + chunk * 16u;
            }
#pragma unroll
            for(int i = 0; i < kBandRows / 128; ++i)
                xs_goff[i] = min((uint32_t)m0 + 64u * (2u * i + g) + (uint32_t)lane, (uint32_t)p.M - 1u) * (uint32_t)p.xs_m * 4u;
            const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem3);
            uint32_t stage = 0;
            int  count = 0; // loads of the youngest K block
            auto issue = [&](int kb) {
                count = 0;
                if(kb >= n)
                    return;
                const uint8_t* src = p.xq + (size_t)kb * 128;
#pragma unroll
                for(int i = 0; i < kBandRows / 16; ++i)
                    if(i < loads)
                        ring_dma16(base + stage * x_stage + (uint32_t)(2 * i + g) * 1024u, goff[i], src);
                count = loads;
#pragma unroll
                for(int i = 0; i < kBandRows / 128; ++i)
                    if(64 * (2 * i + g) < lds.rows)
                    {
                        if constexpr(XS4)
                        {
                            if((kb & 3) == 0)
                            {
                                ring_dma16(base + (uint32_t)lds.xs_at + (((uint32_t)kb >> 2 & 1u) * kBandRows + 64u * (2 * i + g)) * 16u,
                                           xs_goff[i] + (uint32_t)kb * 4u, (const uint8_t*)p.xs);
                                ++count;
                            }
                        }
                        else
                        {
                            ring_dma4(base + (uint32_t)lds.xs_at + ((uint32_t)(kb % 3) * kBandRows + 64u * (2 * i + g)) * 4u,
                                      xs_goff[i] + (uint32_t)kb * (uint32_t)p.xs_k * 4u, (const uint8_t*)p.xs);
                            ++count;
                        }
                    }
                stage = stage + 1 == (uint32_t)kXStages ? 0 : stage + 1;
            };
            issue(0);
            issue(1);
            wait_all_but_few(count);
            __syncthreads();
            for(int kb = 0; kb < n; ++kb)
            {
                issue(kb + kXStages - 1);
                wait_all_but_few(count);
                __syncthreads();
            }
        }
        return;
    }

    const int  l16 = lane & 15, kg = lane >> 4;
    const bool busy = m0 + wave * 32 < p.M;
    if(!busy)
    {
        for(int kb = 0; kb <= n; ++kb)
            __syncthreads();
        return;
    }
    const uint32_t sw      = lds_swizzle((uint32_t)l16);
    const uint32_t lo_off  = (uint32_t)l16 * 128u + (((2u * kg) ^ sw) << 4);
    const uint32_t hi_off  = (uint32_t)l16 * 128u + (((2u * kg + 1u) ^ sw) << 4);
    const uint32_t wlo_off = (uint32_t)lds.w_at + (SHUF ? (uint32_t)kg * 512u + (uint32_t)l16 * 16u : lo_off);
    const uint32_t whi_off = (uint32_t)lds.w_at + (SHUF ? (uint32_t)kg * 512u + (uint32_t)l16 * 16u + 256u : hi_off);
    const uint32_t xlo_off = (uint32_t)wave * 4096u + lo_off, xhi_off = (uint32_t)wave * 4096u + hi_off;
    uint32_t       w_on = 0, x_on = 0;
    auto frag = [&](uint32_t lo, uint32_t hi) -> i32x8 {
        const i32x4 a = *(lds_vec_ptr)(smem3 + lo);
        const i32x4 b = *(lds_vec_ptr)(smem3 + hi);
        return i32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    };
    auto read_w = [&](int i) { return frag(w_on + wlo_off + i * 2048u, w_on + whi_off + i * 2048u); };
    auto read_x = [&](int j) { return frag(x_on + xlo_off + j * 2048u, x_on + xhi_off + j * 2048u); };

    // w_scale: the band's rows lie in one or two blocks of 128; fragments from `split` on are the second one's
    const int    nblocks = (p.N + 127) / 128, nb = n0 >> 7;
    const int    split   = (128 - (n0 & 127)) >> 4;
    const float* ws_row  = p.ws + (size_t)min(nb, nblocks - 1) * n;
    const float* ws_row2 = p.ws + (size_t)min(nb + 1, nblocks - 1) * n;
    float        ws_vec[2] = {ring_ws_window(ws_row, n, 0, lane), ring_ws_window(ws_row2, n, 0, lane)};

    float acc[NF][2][4];
#pragma unroll
    for(int i = 0; i < NF; ++i)
#pragma unroll
        for(int q = 0; q < 8; ++q)
            acc[i][q >> 2][q & 3] = 0.f;
    f32x4 P[4];
    i32x8 bx[2][2], aw[3];
    float xsp[2] = {0.f, 0.f}, wsp[2] = {0.f, 0.f}; // scales of the previous K block
#pragma unroll
    for(int q = 0; q < 4; ++q)
    {
        P[q]             = f32x4{0.f, 0.f, 0.f, 0.f};
        bx[q >> 1][q & 1] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
        asm volatile("" : "+v"(bx[q >> 1][q & 1]));
    }
#pragma unroll
    for(int q = 0; q < 3; ++q)
    {
        aw[q] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
        asm volatile("" : "+v"(aw[q]));
    }
    asm volatile("s_nop 7" ::: "memory");
    const uint32_t xs_lds = (uint32_t)lds.xs_at + ((uint32_t)wave * 32u + (uint32_t)l16) * (XS4 ? 16u : 4u);

    __syncthreads(); // the first K block is in LDS
    // The instruction stream of gemm_ring.h with NF weight and two activation fragments: 2 NF slots per K block, a product
    // folded in two slots behind its MFMA, the last two fragments' tiles issued behind the barrier, while the next K block's
    // first fragments travel from LDS.  PAR: parity of the K block, i.e. which activation fragments are its own.
    auto kblock = [&](int kb, auto par) {
        constexpr int PAR = decltype(par)::value, BASE = PAR * ((2 * NF) & 3); // first product register
        aw[0]      = read_w(0);
        bx[PAR][0] = read_x(0);
        bx[PAR][1] = read_x(1);
        float xsv[2];
        const uint32_t xs_on = XS4 ? ((uint32_t)kb >> 2 & 1u) * (kBandRows * 16u) + ((uint32_t)kb & 3u) * 4u : (uint32_t)(kb % 3) * (kBandRows * 4u);
#pragma unroll
        for(int j = 0; j < 2; ++j)
            xsv[j] = *(lds_f32_ptr)(smem3 + xs_lds + xs_on + j * 16u * (XS4 ? 16u : 4u));
        if((kb & 63) == 0 && kb != 0)
        {
            ws_vec[0] = ring_ws_window(ws_row, n, kb, lane);
            ws_vec[1] = ring_ws_window(ws_row2, n, kb, lane);
            asm volatile("" : "+v"(ws_vec[0]), "+v"(ws_vec[1])); // waited for here, and not in every K block
        }
        float wsc[2];
#pragma unroll
        for(int g = 0; g < 2; ++g)
            wsc[g] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ws_vec[g]), kb & 63));
#pragma unroll
        for(int q = 0; q < 2 * NF; ++q)
        {
            if(q < 4) // tile (NF - 2 + q / 2, q % 2) of the previous K block
                FP8BS_MFMA(P[(BASE + q) & 3], aw[(NF - 2 + q / 2) % 3], bx[1 - PAR][q & 1]);
            else // tile (q / 2 - 2, q % 2) of this one
                FP8BS_MFMA(P[(BASE + q) & 3], aw[(q / 2 - 2) % 3], bx[PAR][q & 1]);
            if((q & 1) && (q - 1) / 2 + 1 < NF) // the buffer that this slot was the last to read
                aw[(q / 2 + 1) % 3] = read_w(q / 2 + 1);
            const int i = q < 6 ? NF - 3 + q / 2 : q / 2 - 3; // fragment of the product issued two slots ago
            const float s = (q < 6 ? xsp[q & 1] : xsv[q & 1]) * (i < split ? (q < 6 ? wsp[0] : wsc[0]) : (q < 6 ? wsp[1] : wsc[1]));
            FP8BS_FMA4(acc[i][q & 1], P[(BASE + q + 2) & 3], s);
        }
        xsp[0] = xsv[0];
        xsp[1] = xsv[1];
        wsp[0] = wsc[0];
        wsp[1] = wsc[1];
        w_on = w_on + kWStage == (uint32_t)lds.w_stages * kWStage ? 0u : w_on + kWStage;
        x_on = x_on == (kXStages - 1u) * x_stage ? 0u : x_on + x_stage;
        __syncthreads();
    };
    int kb = 0;
    for(; kb + 1 < n; kb += 2)
    {
        kblock(kb, std::integral_constant<int, 0>{});
        kblock(kb + 1, std::integral_constant<int, 1>{});
    }
    // the last two fragments' tiles of the last K block, then the two products in flight
    auto drain = [&](auto par) {
        constexpr int PAR = decltype(par)::value, BASE = PAR * ((2 * NF) & 3);
#pragma unroll
        for(int q = 0; q < 6; ++q)
        {
            if(q < 4)
                FP8BS_MFMA(P[(BASE + q) & 3], aw[(NF - 2 + q / 2) % 3], bx[1 - PAR][q & 1]);
            if(q == 4)
                asm volatile("s_nop 15\n s_nop 15\n s_nop 15" ::: "memory"); // >= 11 wait states after the last MFMA
            const int i = NF - 3 + q / 2;
            FP8BS_FMA4(acc[i][q & 1], P[(BASE + q + 2) & 3], (xsp[q & 1] * (i < split ? wsp[0] : wsp[1])));
        }
    };
    if(kb < n)
    {
        kblock(kb, std::integral_constant<int, 0>{});
        drain(std::integral_constant<int, 1>{});
    }
    else
        drain(std::integral_constant<int, 0>{});

    // (behind the last barrier every load has landed and every read is done: the LDS is free)
    constexpr uint32_t kPitch = BN * 2 + 16;
    static_assert(kMulWaves * 32 * kPitch <= 160 * 1024, "LDS");
    const uint32_t ebase = (uint32_t)wave * (32u * kPitch);
    typedef u32x2 __attribute__((address_space(3)))*       lds_u2_ptr;
    typedef const u32x4 __attribute__((address_space(3)))* lds_u4_ptr;
#pragma unroll
    for(int j = 0; j < 2; ++j)
#pragma unroll
        for(int i = 0; i < NF; ++i)
            *(lds_u2_ptr)(smem3 + ebase + (uint32_t)(j * 16 + l16) * kPitch + (uint32_t)(i * 16 + kg * 4) * 2u) =
                u32x2{pack2<DT>(acc[i][j][0], acc[i][j][1]), pack2<DT>(acc[i][j][2], acc[i][j][3])};
    constexpr int kRowLanes = 2 * NF, kRowsPer = 64 / kRowLanes; // lanes that store a row; rows per instruction
    const int  rl = lane / kRowLanes, col = (lane - rl * kRowLanes) * 8;
    const int  nn = n0 + col;
    const bool vec_ok = (p.N & 7) == 0 && ((uintptr_t)p.out & 15) == 0 && nn + 8 <= p.N;
#pragma unroll
    for(int c = 0; c < (32 + kRowsPer - 1) / kRowsPer; ++c)
    {
        const int row = c * kRowsPer + rl, m = m0 + wave * 32 + row;
        if(rl >= kRowsPer || row >= 32 || m >= p.M)
            continue;
        const u32x4 v   = *(lds_u4_ptr)(smem3 + ebase + (uint32_t)row * kPitch + (uint32_t)col * 2u);
        uint16_t*   dst = p.out + (size_t)m * p.N + nn;
        if(vec_ok)
            *(u32x4*)dst = v;
        else
        {
#pragma unroll
            for(int r = 0; r < 8; ++r)
                if(nn + r < p.N)
                    dst[r] = (uint16_t)((v[r >> 1] >> ((r & 1) * 16)) & 0xffffu);
        }
    }
}
#undef FP8BS_MFMA
#undef FP8BS_FMA4

constexpr int kLds = 160 * 1024;
constexpr int scale_bytes(bool xs4) { return xs4 ? 2 * kBandRows * 16 : 3 * kBandRows * 4; }
constexpr int weight_stages(int rows, int nf, bool xs4)
{
    return std::min(6, (kLds - kXStages * rows * 128 - scale_bytes(xs4)) / (16 * nf * 128));
}
// The waits count w_stages - 2 K blocks of the youngest loads, at most four: three to six stages, fewest with the most rows
static_assert(weight_stages(kBandRows, 9, true) == 3 && weight_stages(kBandRows, 9, false) == 3 && weight_stages(kBandRows, 6, true) == 4 &&
              weight_stages(208, 9, true) == 4 && weight_stages(224, 9, true) == 3 && weight_stages(224, 9, false) == 4 &&
              weight_stages(240, 9, false) == 3 && weight_stages(16, 9, true) == 6, "stages of weights");

BandLayout band_layout(const GemmKernelParams& p, int nf, bool xs4)
{
    BandLayout l{};
    l.rows     = std::min((p.M + 15) & ~15, kBandRows);
    const int scales = scale_bytes(xs4), stage = 16 * nf * 128;
    l.w_stages = weight_stages(l.rows, nf, xs4);
    l.w_at     = kXStages * l.rows * 128;
    l.xs_at    = l.w_at + l.w_stages * stage;
    l.total    = std::max(l.xs_at + scales, kMulWaves * 32 * (16 * nf * 2 + 16));
    l.stream_w = gemm_band_streams_weights(p.M, p.N, p.K);
    return l;
}

template <int NF>
auto band_kernel(bool shuffled, bool xs4, bool bf)
{
    return shuffled ? (bf ? gemm_band_kernel<In16::bf16, true, false, NF> : gemm_band_kernel<In16::fp16, true, false, NF>)
           : xs4    ? (bf ? gemm_band_kernel<In16::bf16, false, true, NF> : gemm_band_kernel<In16::fp16, false, true, NF>)
                    : (bf ? gemm_band_kernel<In16::bf16, false, false, NF> : gemm_band_kernel<In16::fp16, false, false, NF>);
}

} // namespace

// band: 96 or 144 weight rows per workgroup.  Operands as gemm_prefill_supports says.
hipError_t launch_gemm_band(const GemmKernelParams& p, In16 out_dtype, const LaunchCtx& ctx, int band)
{
    int        device = 0;
    hipError_t e      = hipGetDevice(&device);
    if(e != hipSuccess)
        return e;
    const int  tiles_m = (p.M + kBandRows - 1) / kBandRows, tiles_n = (p.N + band - 1) / band;
    const bool xs4 = !p.w_shuffled && p.xs_k == 1 && p.xs_m == p.kblocks && (p.kblocks & 3) == 0 && ((uintptr_t)p.xs & 15) == 0;
    const bool bf  = out_dtype == In16::bf16;
    auto kernel = band == 96 ? band_kernel<6>(p.w_shuffled, xs4, bf) : band_kernel<9>(p.w_shuffled, xs4, bf);
    const BandLayout l = band_layout(p, band / 16, xs4);
    // the opt-in to more than 64 KiB of LDS, per device and instantiation, once (racing first calls repeat it)
    constexpr int kMaxDevices = 64;
    static std::atomic<bool> ready[kMaxDevices][12];
    const int inst = (p.w_shuffled ? 2 : xs4 ? 4 : 0) + (bf ? 0 : 1) + (band == 96 ? 6 : 0);
    if(device < 0 || device >= kMaxDevices || !ready[device][inst])
    {
        if((e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024)) != hipSuccess)
            return e;
        if(device >= 0 && device < kMaxDevices)
            ready[device][inst] = true;
    }
    const int grid = (tiles_m * tiles_n + 7) & ~7;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kBandThreads), (size_t)l.total, ctx.stream, p, tiles_m, tiles_n, l);
    return hipGetLastError();
}

} // namespace fp8bs
