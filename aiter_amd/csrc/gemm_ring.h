// The multiply loop shared by the kernels whose workgroup tile is 256 x 128: eight waves multiply, with a 64 (n) x 64 (m) block
// of the tile each; four more bring both operand slabs in by direct global->LDS loads, into a ring of three stages.
//
// Why waves that only fetch.  A wave that issues a load is held at the issue while the memory pipeline's queue is full
// (48 KiB are 768 cycles of it per K block), and with it the MFMAs behind: with the loads dealt out over the multiplying
// waves a K block took the sum of the two, 2000 cycles of which the matrix pipes were busy for 1024.
//
// Why three stages of a 256 x 128 tile.  A K block of it is 1024 matrix cycles per SIMD, 0.45-0.55 us; a slab load takes
// 1-2 us from the last-level cache or HBM while every compute unit asks.  With two stages the loads of K block kb + 1 have
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

constexpr int kRingMulWaves = 8, kRingFetchWaves = 4;
constexpr int kRingMulThreads = 64 * kRingMulWaves, kRingThreads = 64 * (kRingMulWaves + kRingFetchWaves);

// WN: waves along n (2 or 4); the tile is 64 WN (n) x 64 (8 / WN) (m).
template <int WN>
struct RingTile
{
    static constexpr int kWN = WN, kFrags = 4, kStages = 3; // fragments of 16 weight rows per multiplying wave
    static constexpr int kWM = 8 / WN, kBN = WN * 64, kBM = kWM * 64;
    static constexpr int kSlabBytes  = (kBM + kBN) * 128;       // weight rows, then activation rows: 48 KiB
    static constexpr int kStageBytes = kSlabBytes + kBM * 4;    // + the K block's x_scale of the tile's rows
    static constexpr int kWindows    = kStages * kStageBytes;   // two windows of four K blocks of x_scale (XS4)
    static constexpr int kWindowBytes = kBM * 16;
    static constexpr int kLoads      = (kBM + kBN) / 32;        // slab loads per fetching wave and stage: 8 rows each
    static constexpr int kWLoads     = kBN / 32;
    static constexpr size_t lds_bytes(bool xs4) { return (size_t)kWindows + (xs4 ? 2 * kWindowBytes : 0); }
};

// Where a tile's operands come from: filled by the kernel; the per-lane offsets by the fetching waves, the w_scale rows by
// the multiplying ones.
template <class T>
struct RingSource
{
    const uint8_t* wq;                      // uniform bases; a load reads base + goff + kb * (bytes per K block)
    const uint8_t* xq;
    const uint8_t* xs;
    uint32_t       goff[T::kLoads];
    uint32_t       xs_goff;                 // fetching waves 0 .. kWM - 1: this lane's row of x_scale
    uint32_t       xs_step;                 // bytes between two K blocks of x_scale (not XS4)
    const float*   ws_row;                  // w_scale of the tile's columns of this wave, [kblocks]
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

// The fetching waves' half of a tile: its K blocks into the ring.  f: 0 .. 3.
//
// SHUF: weights pre-shuffled (16,16); a 16-row tile's K block is 2 KiB in fragment order and is copied as it lies.
// XS4: x_scale rows are 16-byte aligned and come four K blocks per load (see gemm_prefill.hip for what that saves).
//
// Both halves pass the same barriers: one when the first K block is in LDS, one per K block, after which the next one is, and
// the stage just multiplied is free.  At the last one every load has landed and every read is done: the LDS is free.  The
// caller has a barrier between the last use of the LDS and this call.
template <class T, bool SHUF, bool XS4>
__device__ __forceinline__ void ring_fetch(lds_byte_ptr smem3, const RingSource<T>& src, int f)
{
    constexpr int S = T::kStages;
    const bool xs_wave = f < T::kWM; // waves that fetch x_scale, 64 rows each
    const int  n = src.kblocks;
    auto issue_slabs = [&](int kb, uint32_t stage) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem3 + stage + f * 1024));
#pragma unroll
        for(int u = 0; u < T::kLoads; ++u)
        {
            const size_t koff = (size_t)kb * (u < T::kWLoads && SHUF ? 2048 : 128);
            ring_dma16(dst + (uint32_t)u * (kRingFetchWaves * 1024u), src.goff[u], (u < T::kWLoads ? src.wq : src.xq) + koff);
        }
    };
    auto issue_xs = [&](int kb, uint32_t stage) {
        if constexpr(XS4)
            ring_dma16(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem3 + T::kWindows + ((kb >> 2) & 1) * T::kWindowBytes + f * 1024)),
                       src.xs_goff + (uint32_t)(kb & ~3) * 4u, src.xs);
        else
            ring_dma4(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem3 + stage + T::kSlabBytes + f * 256)),
                      src.xs_goff + (uint32_t)kb * src.xs_step, src.xs);
    };
    // K block kb into `stage`; past the end the last block again, unused, so that every stage has its loads.  x_scale comes
    // with each of them, or (XS4) with the one that opens a window of four.
    bool with_xs = false; // whether this wave's loads of the youngest stage include one of x_scale
    auto issue = [&](int kb, uint32_t stage) {
        const int at = min(kb, n - 1);
        issue_slabs(at, stage);
        with_xs = xs_wave && (!XS4 || ((at & 3) == 0 && at == kb));
        if(with_xs)
            issue_xs(at, stage);
    };
    auto wait_but_youngest = [&] { // all but the youngest stage's loads of this wave have landed
        static_assert(T::kLoads == 12 && S == 3, "the waits count the loads of a stage");
        if(with_xs)
            asm volatile("s_waitcnt vmcnt(13)" ::: "memory");
        else
            asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    };
#pragma unroll
    for(int s = 0; s < S - 1; ++s)
        issue(s, (uint32_t)s * T::kStageBytes);
    wait_but_youngest();
    __syncthreads();
    uint32_t stage = (S - 1) * T::kStageBytes; // of K block kb + S - 1
    for(int kb = 0; kb < n; ++kb)
    {
        issue(kb + S - 1, stage);
        stage = stage == (S - 1u) * T::kStageBytes ? 0u : stage + (uint32_t)T::kStageBytes;
        if(kb + 1 < n)
            wait_but_youngest();
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }
}

// w_scale for 64 consecutive K blocks from kb0 (a multiple of 64) on in one VGPR, lane = K block: picked with
// v_readlane, because a scalar load in the loop would share the LGKM counter with the LDS reads
__device__ __forceinline__ float ring_ws_window(const float* row, int kblocks, int kb0, int lane)
{
    return row[min(kb0 + lane, kblocks - 1)];
}

// The multiplying waves' half: acc[i][j] += this wave's share, weight fragment i, activation fragment j.  wave: 0 .. 7.
//
// lo, hi: K blocks.  A tile's K blocks may be multiplied in several calls that follow one another (lo > 0 continues where the
// call before stopped), for sums of their own.
// ws_vec: ring_ws_window of the window that `lo` lies in; handed on from call to call.
// busy: false for a wave whose rows are all padding: it multiplies nothing.
template <class T, bool SHUF, bool XS4>
__device__ __forceinline__ void ring_multiply(lds_byte_ptr smem3, const RingSource<T>& src, int wave, int lane, int lo, int hi,
                                              bool busy, float& ws_vec, float (&acc)[T::kFrags][4][4])
{
    constexpr int NF = T::kFrags, H = NF / 2, D = 4 * H; // fragments H .. NF - 1 are deferred: D tiles
    if(!busy)
    {
        for(int kb = lo + (lo > 0 ? 1 : 0); kb <= hi; ++kb)
            __syncthreads();
        return;
    }
    const int l16 = lane & 15, kg = lane >> 4;
    const int wn = wave % T::kWN, wm = wave / T::kWN;
    const uint32_t sw      = lds_swizzle((uint32_t)l16);
    const uint32_t lo_off  = (uint32_t)l16 * 128u + (((2u * kg) ^ sw) << 4);
    const uint32_t hi_off  = (uint32_t)l16 * 128u + (((2u * kg + 1u) ^ sw) << 4);
    const uint32_t wlo_off = SHUF ? (uint32_t)kg * 512u + (uint32_t)l16 * 16u : lo_off;
    const uint32_t whi_off = SHUF ? wlo_off + 256u : hi_off;
    const uint32_t w_base  = (uint32_t)wn * (16u * NF * 128u);
    const uint32_t x_base  = (uint32_t)T::kBN * 128u + (uint32_t)wm * (64u * 128u);

    auto frag = [&](uint32_t lo, uint32_t hi) -> i32x8 {
        const i32x4 a = *(lds_vec_ptr)(smem3 + lo);
        const i32x4 b = *(lds_vec_ptr)(smem3 + hi);
        return i32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    };
    auto read_w = [&](uint32_t stage, int i) { return frag(stage + w_base + wlo_off + i * 2048u, stage + w_base + whi_off + i * 2048u); };
    auto read_x = [&](uint32_t stage, int j) { return frag(stage + x_base + lo_off + j * 2048u, stage + x_base + hi_off + j * 2048u); };

    if(lo == 0)
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

    uint32_t stage = (uint32_t)(lo % T::kStages) * T::kStageBytes; // of K block kb

    // The instruction stream is that of gemm_prefill.hip with four weight fragments: 4 NF MFMA slots per K block, the FMAs
    // that fold a product into the accumulators two slots behind its MFMA; the tiles of the upper half of the fragments are
    // issued behind the barrier, while the next K block's first fragments travel from LDS.  Where those notes speak of zero
    // fragments for the first K block's predecessor and the wait states ahead of the first MFMA, the same holds here.
    f32x4 P[4];
    i32x8 bx[4], aw[NF];
#pragma unroll
    for(int q = 0; q < 4; ++q)
    {
        P[q]  = f32x4{0.f, 0.f, 0.f, 0.f};
        bx[q] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for(int q = 0; q < NF; ++q)
        aw[q] = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
    float scp[4]; // x_scale * w_scale of the previous K block
#pragma unroll
    for(int j = 0; j < 4; ++j)
        scp[j] = 0.f;
#pragma unroll
    for(int q = 0; q < 4; ++q)
        asm volatile("" : "+v"(bx[q]));
#pragma unroll
    for(int q = 0; q < NF; ++q)
        asm volatile("" : "+v"(aw[q]));
    asm volatile("s_nop 7" ::: "memory");

    // LDS address of this lane's x_scale for m tile 0; tile j sits 64 (XS4: 256) bytes further
    const uint32_t xs_lds = XS4 ? (uint32_t)T::kWindows + ((uint32_t)wm * 64u + (uint32_t)l16) * 16u
                                : (uint32_t)T::kSlabBytes + ((uint32_t)wm * 64u + (uint32_t)l16) * 4u;
    auto xs_window_addr = [&](int kb) -> uint32_t { return (uint32_t)(((kb >> 2) & 1) * T::kWindowBytes + (kb & 3) * 4) + xs_lds; };
    uint32_t xs_addr = XS4 ? xs_window_addr(lo) : 0u;

    for(int kb = lo; kb < hi; ++kb)
    {
        if((kb & 63) == 0 && kb != 0)
            ws_vec = ring_ws_window(src.ws_row, src.kblocks, kb, lane);
        const float wsc = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ws_vec), kb & 63));

        aw[0] = read_w(stage, 0);
        float sc[4];
#pragma unroll
        for(int j = 0; j < 4; ++j)
        {
            const float xsv = XS4 ? *(lds_f32_ptr)(smem3 + xs_addr + j * 256) : *(lds_f32_ptr)(smem3 + stage + xs_lds + j * 64);
            sc[j]           = xsv * wsc;
        }
#pragma unroll
        for(int q = 0; q < 4 * NF; ++q)
        {
            if(q == 2)
                aw[1] = read_w(stage, 1);
            if(q < D) // deferred tile (H + q % H, q / H) of the previous K block
                FP8BS_MFMA(P[q & 3], aw[H + q % H], bx[q / H]);
            else // tile ((q - D) >> 2, (q - D) & 3) of this one
                FP8BS_MFMA(P[q & 3], aw[(q - D) >> 2], bx[(q - D) & 3]);
            // LDS reads that the slot just issued has made room for
            if(q < D && q % H == H - 1)
                bx[q / H] = read_x(stage, q / H);
            if(q < D && q >= D - H)
                aw[q - D + NF] = read_w(stage, q - D + NF);
            if(XS4 && q == D)
            {
                xs_addr = xs_window_addr(kb + 1);
                asm volatile("" : "+v"(xs_addr)); // here, between two slots
            }
            // fold in the product issued two slots ago
            if(q < 2)
                FP8BS_FMA4(acc[H - 1][2 + q], P[2 + q], scp[2 + q]);
            else if(q < D + 2)
                FP8BS_FMA4(acc[H + (q - 2) % H][(q - 2) / H], P[(q - 2) & 3], scp[(q - 2) / H]);
            else
                FP8BS_FMA4(acc[(q - 2 - D) >> 2][(q - 2 - D) & 3], P[(q - 2) & 3], sc[(q - 2 - D) & 3]);
        }
#pragma unroll
        for(int j = 0; j < 4; ++j)
            scp[j] = sc[j];
        stage = stage == (T::kStages - 1u) * T::kStageBytes ? 0u : stage + (uint32_t)T::kStageBytes;
        // (every fragment of this K block is in registers, or on its way there: the barrier waits for outstanding LDS
        // reads) the next one is in LDS behind it
        __syncthreads();
    }
    // the deferred tiles of the last K block, then the two products in flight
#pragma unroll
    for(int q = 0; q < D; ++q)
    {
        FP8BS_MFMA(P[q & 3], aw[H + q % H], bx[q / H]);
        if(q < 2)
            FP8BS_FMA4(acc[H - 1][2 + q], P[2 + q], scp[2 + q]);
        else
            FP8BS_FMA4(acc[H + (q - 2) % H][(q - 2) / H], P[(q - 2) & 3], scp[(q - 2) / H]);
    }
    asm volatile("s_nop 15\n s_nop 15\n s_nop 15" ::: "memory"); // >= 11 wait states after the last MFMA
#pragma unroll
    for(int q = D; q < D + 2; ++q)
        FP8BS_FMA4(acc[H + (q - 2) % H][(q - 2) / H], P[(q - 2) & 3], scp[(q - 2) / H]);
#undef FP8BS_MFMA
#undef FP8BS_FMA4
}

} // namespace fp8bs
