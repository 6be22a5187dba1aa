// The multiply loop shared by the kernels whose workgroup tile is 128 x 256 or 256 x 128: eight waves multiply, with a
// 64 (n) x 64 (m) block of the tile each; four more bring both operand slabs in by direct global->LDS loads, into a ring
// of three stages.
//
// Why waves that only fetch.  A wave that issues a load is held at the issue while the memory pipeline's queue is full
// (48 KiB are 768 cycles of it per K block), and with it the MFMAs behind: with the loads dealt out over the multiplying
// waves a K block took the sum of the two, 2000 cycles of which the matrix pipes were busy for 1024.
//
// Why three stages.  A K block of such a tile is 1024 matrix cycles per SIMD, 0.45-0.55 us; a slab load takes 1-2 us
// from the last-level cache or HBM while every compute unit asks.  With two stages the loads of K block kb + 1 have
// one K block of time to arrive and set the pace; with three they have two.  A stage is 48 KiB, so a tile of this
// size is the largest for which three fit the 160 KiB.
//
// Bound by, per K block of a compute unit: 48 KiB taken in, 128 KiB of fragments out of LDS (1024 cycles at 128
// bytes a cycle, beside 384 for what the loads write), 128 MFMAs (1024 cycles per SIMD).
#pragma once

#include "gemm_common.h"

namespace fp8bs {

typedef uint8_t __attribute__((address_space(3)))*              lds_byte_ptr;
typedef const volatile i32x4 __attribute__((address_space(3)))* lds_vec_ptr;
typedef const volatile float __attribute__((address_space(3)))* lds_f32_ptr;

constexpr int kRingStages = 3, kRingFrags = 4;   // weight (and activation) fragments per multiplying wave
constexpr int kRingMulWaves = 8, kRingFetchWaves = 4;
constexpr int kRingMulThreads = 64 * kRingMulWaves, kRingThreads = 64 * (kRingMulWaves + kRingFetchWaves);

// WN: waves along n (2 or 4); the tile is 64 WN (n) x 64 (8 / WN) (m)
template <int WN>
struct RingTile
{
    static constexpr int kWM = 8 / WN, kBN = WN * 64, kBM = kWM * 64;
    static constexpr int kSlabBytes  = (kBM + kBN) * 128;       // weight rows, then activation rows: 48 KiB
    static constexpr int kStageBytes = kSlabBytes + kBM * 4;    // + the K block's x_scale of the tile's rows
    static constexpr int kWindows    = kRingStages * kStageBytes; // two windows of four K blocks of x_scale (XS4)
    static constexpr int kWindowBytes = kBM * 16;
    static constexpr int kLoads      = (kBM + kBN) / 32;        // slab loads per fetching wave and stage: 8 rows each
    static constexpr int kWLoads     = kBN / 32;
    static constexpr size_t lds_bytes(bool xs4) { return (size_t)kWindows + (xs4 ? 2 * kWindowBytes : 0); }
};

// Where a tile's operands come from: filled by the kernel; the per-lane offsets by the fetching waves, the w_scale rows by
// the multiplying ones.
template <int WN>
struct RingSource
{
    const uint8_t* wq;                      // uniform bases; a load reads base + goff + kb * (bytes per K block)
    const uint8_t* xq;
    const uint8_t* xs;
    uint32_t       goff[RingTile<WN>::kLoads];
    uint32_t       xs_goff;                 // fetching waves 0 .. kWM - 1: this lane's row of x_scale
    uint32_t       xs_step;                 // bytes between two K blocks of x_scale (not XS4)
    const float*   ws_row[2];               // w_scale of weight fragments 0, 1 and of 2, 3 (SG = 2), [kblocks]
    int            kblocks;
};

// One LDS-direct load: lane l's 16 (4) bytes land at M0 + 16 l (4 l).  From asm: the compiler models the builtin as a
// flat access that may touch LDS and from then on waits for every outstanding LDS read in full.  The loads are
// invisible to its wait counts; their consumers sit behind the explicit waits below and a barrier.
__device__ __forceinline__ void ring_dma16(uint32_t lds_dst, uint32_t voff, const uint8_t* sbase)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_dst), "v"(voff), "s"(sbase) : "memory");
}
__device__ __forceinline__ void ring_dma4(uint32_t lds_dst, uint32_t voff, const uint8_t* sbase)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(lds_dst), "v"(voff), "s"(sbase) : "memory");
}

// The stage row that lane `lane` of fetching wave f brings in with load i, and the 16-byte chunk of that row's K block: a
// load fills 8 rows (1 KiB) of the stage, lane l its chunk l, i.e. row 8 u + l / 8, stored chunk l % 8, which holds the row's
// logical chunk (l % 8) ^ lds_swizzle(row).  (Shuffled weights are copied as they lie: half of tile u / 2's K block.)
struct RingUnit
{
    uint32_t u, row, chunk;
};
__device__ __forceinline__ RingUnit ring_unit(int i, int f, int lane)
{
    const uint32_t u = (uint32_t)(kRingFetchWaves * i + f), r = 8u * u + ((uint32_t)lane >> 3);
    return RingUnit{u, r, ((uint32_t)lane & 7u) ^ lds_swizzle(r)};
}

// The fetching waves' half of a tile: K blocks kb_lo .. kb_hi - 1 (kb_hi > kb_lo) into the ring.  f: 0 .. 3.
//
// SHUF: weights pre-shuffled (16,16); a 16-row tile's K block is 2 KiB in fragment order and is copied as it lies.
// XS4: x_scale rows are 16-byte aligned and come four K blocks per load (see gemm_prefill.hip for what that saves).
//
// Both halves pass the same barriers: one when K block kb_lo is in LDS, one per K block, after which the next one is, and
// the stage just multiplied is free.  At the last one every load has landed and every read is done: the LDS is free.  The
// caller has a barrier between the last use of the LDS and this call.
template <int WN, bool SHUF, bool XS4>
__device__ __forceinline__ void ring_fetch(lds_byte_ptr smem3, const RingSource<WN>& src, int f, int kb_lo, int kb_hi)
{
    using T = RingTile<WN>;
    const bool xs_wave = f < T::kWM; // waves that fetch x_scale, 64 rows each
    auto issue_slabs = [&](int kb, uint32_t stage) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem3 + stage + f * 1024));
#pragma unroll
        for(int u = 0; u < T::kLoads; ++u)
        {
            const size_t koff = (size_t)kb * (u < T::kWLoads && SHUF ? 2048 : 128);
            ring_dma16(dst + (uint32_t)u * (kRingFetchWaves * 1024u), src.goff[u], (u < T::kWLoads ? src.wq : src.xq) + koff);
        }
    };
    // x_scale of K block kb, with its stage: every K block, or (XS4) where kb opens a window of four; `real`: kb is not
    // the last block fetched again
    auto fetches_xs = [&](int kb, bool real) { return xs_wave && (!XS4 || ((kb & 3) == 0 && real)); };
    auto issue_xs = [&](int kb, uint32_t stage) {
        if constexpr(XS4)
            ring_dma16(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem3 + T::kWindows + ((kb >> 2) & 1) * T::kWindowBytes + f * 1024)),
                       src.xs_goff + (uint32_t)(kb & ~3) * 4u, src.xs);
        else
            ring_dma4(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem3 + stage + T::kSlabBytes + f * 256)),
                      src.xs_goff + (uint32_t)kb * src.xs_step, src.xs);
    };
    // all but the youngest stage's loads of this wave have landed; `xs`: that stage's loads include one of x_scale
    auto wait_but_youngest = [&](bool xs) {
        static_assert(T::kLoads == 12, "the waits count a stage's loads");
        if(xs)
            asm volatile("s_waitcnt vmcnt(13)" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    };
    const int k1 = min(kb_lo + 1, kb_hi - 1);
    issue_slabs(kb_lo, 0);
    if(xs_wave)
        issue_xs(kb_lo, 0);
    issue_slabs(k1, T::kStageBytes);
    bool xs = fetches_xs(k1, k1 != kb_lo);
    if(xs)
        issue_xs(k1, T::kStageBytes);
    wait_but_youngest(xs);
    __syncthreads();
    uint32_t stage2 = 2 * T::kStageBytes; // of K block kb + 2
    for(int kb = kb_lo; kb < kb_hi; ++kb)
    {
        const int kn = min(kb + 2, kb_hi - 1); // at the end the last block is fetched again, unused
        issue_slabs(kn, stage2);
        xs = fetches_xs(kn, kn == kb + 2);
        if(xs)
            issue_xs(kn, stage2);
        stage2 = stage2 == 2u * T::kStageBytes ? 0u : stage2 + (uint32_t)T::kStageBytes;
        if(kb + 1 < kb_hi)
            wait_but_youngest(xs);
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
}

// The multiplying waves' half: acc[i][j] += this wave's share, weight fragment i, activation fragment j.  wave: 0 .. 7.
//
// SG: w_scale blocks per wave (fragments 0, 1 and 2, 3 may belong to different 128-row blocks).
// busy: false for a wave whose rows are all padding: it multiplies nothing.
// kb_start: the first K block that the fetching waves bring in; a tile's blocks may be multiplied in several calls that
// follow one another (kb_lo > kb_start continues where the call before stopped), for sums of their own.
template <int WN, bool SHUF, bool XS4, int SG>
__device__ __forceinline__ void ring_multiply(lds_byte_ptr smem3, const RingSource<WN>& src, int wave, int lane, int kb_lo,
                                              int kb_hi, bool busy, float (&acc)[kRingFrags][4][4], int kb_start)
{
    using T = RingTile<WN>;
    if(!busy)
    {
        for(int kb = kb_lo + (kb_lo > kb_start ? 1 : 0); kb <= kb_hi; ++kb)
            __syncthreads();
        return;
    }
    const int l16 = lane & 15, kg = lane >> 4;
    const int wn = wave % WN, wm = wave / WN;
    const uint32_t sw      = lds_swizzle((uint32_t)l16);
    const uint32_t lo_off  = (uint32_t)l16 * 128u + (((2u * kg) ^ sw) << 4);
    const uint32_t hi_off  = (uint32_t)l16 * 128u + (((2u * kg + 1u) ^ sw) << 4);
    const uint32_t wlo_off = SHUF ? (uint32_t)kg * 512u + (uint32_t)l16 * 16u : lo_off;
    const uint32_t whi_off = SHUF ? wlo_off + 256u : hi_off;
    const uint32_t w_base  = (uint32_t)wn * (64u * 128u);
    const uint32_t x_base  = (uint32_t)T::kBN * 128u + (uint32_t)wm * (64u * 128u);

    auto frag = [&](uint32_t lo, uint32_t hi) -> i32x8 {
        const i32x4 a = *(lds_vec_ptr)(smem3 + lo);
        const i32x4 b = *(lds_vec_ptr)(smem3 + hi);
        return i32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    };
    auto read_w = [&](uint32_t stage, int i) { return frag(stage + w_base + wlo_off + i * 2048u, stage + w_base + whi_off + i * 2048u); };
    auto read_x = [&](uint32_t stage, int j) { return frag(stage + x_base + lo_off + j * 2048u, stage + x_base + hi_off + j * 2048u); };

    // w_scale for 64 consecutive K blocks in one VGPR (lane = K block), picked with v_readlane: a scalar load in the
    // loop would share the LGKM counter with the LDS reads
    auto load_ws_window = [&](const float* row, int kb0) -> float {
        const int k = kb0 + lane;
        return row[k < src.kblocks ? k : src.kblocks - 1];
    };
    float ws_vec[SG];
#pragma unroll
    for(int g = 0; g < SG; ++g)
        ws_vec[g] = load_ws_window(src.ws_row[g], kb_lo & ~63);
    if(kb_lo == kb_start)
        __syncthreads();

#define FP8BS_MFMA(P, A, B) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=&v"(P) : "v"(A), "v"(B))
#define FP8BS_FMA4(ACC, P, S)                                                              \
    do                                                                                     \
    {                                                                                      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[0]) : "v"((P)[0]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[1]) : "v"((P)[1]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[2]) : "v"((P)[2]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[3]) : "v"((P)[3]), "v"(S));      \
    } while(0)

    uint32_t stage = (uint32_t)((kb_lo - kb_start) % kRingStages) * T::kStageBytes; // of K block kb

    // The instruction stream is that of gemm_prefill.hip with four weight fragments: 16 MFMA slots per K block, the FMAs
    // that fold a product into the accumulators two slots behind its MFMA; the tiles of fragments 2 and 3 are issued
    // behind the barrier, while the next K block's first fragments travel from LDS.  Where those notes speak of zero
    // fragments for the first K block's predecessor and the wait states ahead of the first MFMA, the same holds here.
    f32x4 P[4];
    i32x8 bx[4], aw[4];
#pragma unroll
    for(int q = 0; q < 4; ++q)
    {
        P[q]  = f32x4{0.f, 0.f, 0.f, 0.f};
        bx[q] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
        aw[q] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
    float scp[SG][4]; // x_scale * w_scale of the previous K block
#pragma unroll
    for(int g = 0; g < SG; ++g)
#pragma unroll
        for(int j = 0; j < 4; ++j)
            scp[g][j] = 0.f;
#pragma unroll
    for(int q = 0; q < 4; ++q)
        asm volatile("" : "+v"(bx[q]), "+v"(aw[q]));
    asm volatile("s_nop 7" ::: "memory");

    // LDS address of this lane's x_scale for m tile 0; tile j sits 64 (XS4: 256) bytes further
    const uint32_t xs_lds = XS4 ? (uint32_t)T::kWindows + ((uint32_t)wm * 64u + (uint32_t)l16) * 16u
                                : (uint32_t)T::kSlabBytes + ((uint32_t)wm * 64u + (uint32_t)l16) * 4u;
    auto xs_window_addr = [&](int kb) -> uint32_t { return (uint32_t)(((kb >> 2) & 1) * T::kWindowBytes + (kb & 3) * 4) + xs_lds; };
    uint32_t xs_addr = XS4 ? xs_window_addr(kb_lo) : 0u;

    for(int kb = kb_lo; kb < kb_hi; ++kb)
    {
        if((kb & 63) == 0 && kb != kb_lo)
        {
#pragma unroll
            for(int g = 0; g < SG; ++g)
                ws_vec[g] = load_ws_window(src.ws_row[g], kb);
        }
        float wsc[SG];
#pragma unroll
        for(int g = 0; g < SG; ++g)
            wsc[g] = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ws_vec[g]), kb & 63));

        aw[0] = read_w(stage, 0);
        float sc[SG][4];
#pragma unroll
        for(int j = 0; j < 4; ++j)
        {
            const float xsv = XS4 ? *(lds_f32_ptr)(smem3 + xs_addr + j * 256) : *(lds_f32_ptr)(smem3 + stage + xs_lds + j * 64);
#pragma unroll
            for(int g = 0; g < SG; ++g)
                sc[g][j] = xsv * wsc[g];
        }
#pragma unroll
        for(int q = 0; q < 16; ++q)
        {
            if(q == 2)
                aw[1] = read_w(stage, 1);
            if(q < 8) // deferred tile (2 + (q & 1), q >> 1) of the previous K block
                FP8BS_MFMA(P[q & 3], aw[2 + (q & 1)], bx[q >> 1]);
            else // tile ((q - 8) >> 2, (q - 8) & 3) of this one
                FP8BS_MFMA(P[q & 3], aw[(q - 8) >> 2], bx[(q - 8) & 3]);
            // LDS reads that the slot just issued has made room for
            if(q < 8 && (q & 1))
                bx[q >> 1] = read_x(stage, q >> 1);
            if(q == 6)
                aw[2] = read_w(stage, 2);
            if(q == 7)
                aw[3] = read_w(stage, 3);
            if(XS4 && q == 8)
            {
                xs_addr = xs_window_addr(kb + 1);
                asm volatile("" : "+v"(xs_addr)); // here, between two slots
            }
            // fold in the product issued two slots ago
            if(q < 2)
                FP8BS_FMA4(acc[1][2 + q], P[2 + q], scp[0][2 + q]);
            else if(q < 10)
                FP8BS_FMA4(acc[2 + ((q - 2) & 1)][(q - 2) >> 1], P[(q - 2) & 3], scp[SG - 1][(q - 2) >> 1]);
            else
                FP8BS_FMA4(acc[(q - 10) >> 2][(q - 10) & 3], P[(q - 2) & 3], sc[0][(q - 10) & 3]);
        }
#pragma unroll
        for(int g = 0; g < SG; ++g)
#pragma unroll
            for(int j = 0; j < 4; ++j)
                scp[g][j] = sc[g][j];
        stage = stage == 2u * T::kStageBytes ? 0u : stage + (uint32_t)T::kStageBytes;
        // (every fragment of this K block is in registers, or on its way there: the barrier waits for outstanding LDS
        // reads) K block kb + 1 is in LDS behind it
        __syncthreads();
    }
    // the 8 deferred tiles of the last K block, then the two products in flight
#pragma unroll
    for(int q = 0; q < 8; ++q)
    {
        FP8BS_MFMA(P[q & 3], aw[2 + (q & 1)], bx[q >> 1]);
        if(q < 2)
            FP8BS_FMA4(acc[1][2 + q], P[2 + q], scp[0][2 + q]);
        else
            FP8BS_FMA4(acc[2 + ((q - 2) & 1)][(q - 2) >> 1], P[(q - 2) & 3], scp[SG - 1][(q - 2) >> 1]);
    }
    asm volatile("s_nop 15\n s_nop 15\n s_nop 15" ::: "memory"); // >= 11 wait states after the last MFMA
    FP8BS_FMA4(acc[2][3], P[2], scp[SG - 1][3]);
    FP8BS_FMA4(acc[3][3], P[3], scp[SG - 1][3]);
#undef FP8BS_MFMA
#undef FP8BS_FMA4
}

} // namespace fp8bs
