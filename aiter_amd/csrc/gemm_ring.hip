// Block-scale FP8 GEMM on 256 x 128 tiles: the three-stage ring of gemm_ring.h, four waves that fetch, eight that multiply.
//
// Carries out, where it is faster and 256 x 128 tiles fill at most one round of workgroups, what was chosen for other
// kernels: plans of gemm_prefill.hip with one or two K ranges, and mid_* tilings with one; the additions are the plan's, so the
// bits are too.
//
// Bound by what a compute unit takes in: 48 KiB per K block, 0.75 us with few workgroups, 0.9 us with 256 (13 TB/s out of L2
// over the chip; the matrix pipes need 0.45).  The two-stage tiles of gemm_prefill.hip wait for each K block's loads
// instead (1.2-1.8 us).  us there / here: 3001 x 2112 x 2048 24.1 / 19.3, 2048 x 4096 x 3584 39.8 / 33.8,
// 3000 x 2560 x 5120 59.5 / 43.1; two ranges: 3001 x 2112 x 7168 70 / 53, 2048 x 4096 x 7168 75 / 63,
// 300 x 16384 x 7168 78 / 55.  With more than one round the 256 x 256 tile, 64 KiB for twice the products, is ahead again
// (4096^3: 64 / 68).
#include "gemm_ring.h"

#include <algorithm>
#include <atomic>

namespace fp8bs {

namespace {

constexpr int      WN           = 2;             // waves along n: 256 (m) x 128 (n)
constexpr int      kGroupN      = 8;             // columns of tiles that consecutive workgroups of an XCD sweep together
constexpr uint32_t kOutPitch    = 144;           // bytes per row of a wave's 64 x 64 output block in LDS
constexpr size_t   kParkedBytes = 16 * 512 * 16; // a workgroup's tile in fp32

// FOLD: the K blocks from fold_kb on (0 < fold_kb < kblocks) are summed apart from those before, and the two sums are added:
// what two workgroups with a range each would do.

template <In16 DT, bool SHUF, bool XS4, bool FOLD>
__global__ __launch_bounds__(kRingThreads) void gemm_ring_kernel(GemmKernelParams p, int tiles_m, int tiles_n, int fold_kb, float* parked)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    using T = RingTile<WN>;
    const lds_byte_ptr smem3 = (lds_byte_ptr)smem;

    // each XCD takes a contiguous eighth of the tiles (workgroups go round robin over the XCDs): neighbours share slabs in its L2
    const int total    = tiles_m * tiles_n;
    const int xcd      = blockIdx.x & 7;
    const int tile_end = (int)((int64_t)total * (xcd + 1) / 8);
    for(int tile = (int)((int64_t)total * xcd / 8) + ((int)blockIdx.x >> 3); tile < tile_end; tile += (int)gridDim.x >> 3)
    {
        int t = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
        const int l16 = lane & 15, kg = lane >> 4;
        const int wn = wave % WN, wm = wave / WN;

        const int group  = tile / (kGroupN * tiles_m);
        const int within = tile - group * (kGroupN * tiles_m);
        const int gn     = min(kGroupN, tiles_n - group * kGroupN);
        const int tm     = within / gn;
        const int tn     = group * kGroupN + (within - tm * gn);
        const int m0 = tm * T::kBM, n0 = tn * T::kBN;

        RingSource<T> src;
        src.wq      = p.wq;
        src.xq      = p.xq;
        src.xs      = (const uint8_t*)p.xs;
        src.kblocks = p.kblocks;
        src.xs_step = (uint32_t)p.xs_k * 4u;
        if(wave >= kRingMulWaves)
        {
            const int f = wave - kRingMulWaves;
#pragma unroll
            for(int i = 0; i < T::kLoads; ++i)
            {
                const RingUnit v = ring_unit(i, f, lane);
                if(i < T::kWLoads && SHUF)
                {
                    const uint32_t w16 = min(((uint32_t)n0 >> 4) + (v.u >> 1), ((uint32_t)p.N >> 4) - 1u);
                    src.goff[i]        = w16 * 16u * (uint32_t)p.K + (v.u & 1u) * 1024u + (uint32_t)lane * 16u;
                }
                else if(i < T::kWLoads)
                    src.goff[i] = min((uint32_t)n0 + v.row, (uint32_t)p.N - 1u) * (uint32_t)p.ldb + v.chunk * 16u;
                else
                    src.goff[i] = min((uint32_t)m0 + v.row - (uint32_t)T::kBN, (uint32_t)p.M - 1u) * (uint32_t)p.lda + v.chunk * 16u;
            }
            src.xs_goff = min((uint32_t)m0 + 64u * (uint32_t)(f % T::kWM) + (uint32_t)lane, (uint32_t)p.M - 1u) * (uint32_t)p.xs_m * 4u;
            ring_fetch<T, SHUF, XS4>(smem3, src, f);
            __syncthreads();
            continue;
        }
        float          acc[T::kFrags][4][4];
        const uint32_t nb = min((uint32_t)(n0 + wn * 64) >> 7, (uint32_t)((p.N + 127) / 128 - 1));
        src.ws_row = p.ws + (size_t)nb * p.kblocks;
        const bool busy = m0 + wm * 64 < p.M && n0 + wn * 64 < p.N;
        float      ws_vec = ring_ws_window(src.ws_row, p.kblocks, 0, lane);
        auto zero = [&] {
#pragma unroll
            for(int q = 0; q < 16; ++q)
#pragma unroll
                for(int r = 0; r < 4; ++r)
                    acc[q >> 2][q & 3][r] = 0.f;
        };
        zero();
        if constexpr(FOLD)
        {
            // The second of two ranges of K blocks starts a sum of its own.  There are no 64 registers for the first
            // one's: it waits in memory, each thread reads back what it wrote (5 us of 63 at 2048 x 4096 x 7168).
            const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
                (uint8_t*)parked + (size_t)blockIdx.x * kParkedBytes, 0, (int)kParkedBytes, 0x00020000);
            const int at = t * 4;
            ring_multiply<T, SHUF, XS4>(smem3, src, wave, lane, 0, fold_kb, busy, ws_vec, acc);
#pragma unroll
            for(int q = 0; q < 64; ++q)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[q >> 4][(q >> 2) & 3][q & 3]), rsrc, at, q * 2048, 0);
            zero();
            ring_multiply<T, SHUF, XS4>(smem3, src, wave, lane, fold_kb, p.kblocks, busy, ws_vec, acc);
            // (all requested before the first is added: left to itself the compiler may wait for them one by one)
            float back[64];
#pragma unroll
            for(int q = 0; q < 64; ++q)
                back[q] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, at, q * 2048, 0));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for(int q = 0; q < 64; ++q)
                acc[q >> 4][(q >> 2) & 3][q & 3] = back[q] + acc[q >> 4][(q >> 2) & 3][q & 3];
        }
        else
            ring_multiply<T, SHUF, XS4>(smem3, src, wave, lane, 0, p.kblocks, busy, ws_vec, acc);

        const uint32_t ebase = (uint32_t)wave * (64u * kOutPitch);
        typedef u32x2 __attribute__((address_space(3)))*       lds_u2_ptr;
        typedef const u32x4 __attribute__((address_space(3)))* lds_u4_ptr;
#pragma unroll
        for(int j = 0; j < 4; ++j)
#pragma unroll
            for(int i = 0; i < T::kFrags; ++i)
                *(lds_u2_ptr)(smem3 + ebase + (uint32_t)(j * 16 + l16) * kOutPitch + (uint32_t)(i * 16 + kg * 4) * 2u) =
                    u32x2{pack2<DT>(acc[i][j][0], acc[i][j][1]), pack2<DT>(acc[i][j][2], acc[i][j][3])};
        const int  col    = (lane & 7) * 8;
        const int  n      = n0 + wn * 64 + col;
        const bool vec_ok = (p.N & 7) == 0 && ((uintptr_t)p.out & 15) == 0 && n + 8 <= p.N;
#pragma unroll
        for(int c = 0; c < 8; ++c)
        {
            const int   row = c * 8 + (lane >> 3);
            const int   m   = m0 + wm * 64 + row;
            const u32x4 v   = *(lds_u4_ptr)(smem3 + ebase + (uint32_t)row * kOutPitch + (uint32_t)col * 2u);
            if(m >= p.M)
                continue;
            uint16_t* dst = p.out + (size_t)m * p.N + n;
            if(vec_ok)
                *(u32x4*)dst = v;
            else
            {
#pragma unroll
                for(int r = 0; r < 8; ++r)
                    if(n + r < p.N)
                        dst[r] = (uint16_t)((v[r >> 1] >> ((r & 1) * 16)) & 0xffffu);
            }
        }
        __syncthreads(); // the next tile's slabs land where the output was
    }
}

template <bool FOLD>
auto ring_kernel(bool shuffled, bool xs4, bool bf)
{
    return shuffled ? (bf ? gemm_ring_kernel<In16::bf16, true, false, FOLD> : gemm_ring_kernel<In16::fp16, true, false, FOLD>)
           : xs4    ? (bf ? gemm_ring_kernel<In16::bf16, false, true, FOLD> : gemm_ring_kernel<In16::fp16, false, true, FOLD>)
                    : (bf ? gemm_ring_kernel<In16::bf16, false, false, FOLD> : gemm_ring_kernel<In16::fp16, false, false, FOLD>);
}

} // namespace

hipError_t launch_gemm_ring(const GemmKernelParams& p, In16 out_dtype, const LaunchCtx& ctx, int fold_kb, int device, int cus)
{
    using T = RingTile<WN>;
    const int  tiles_m = (p.M + T::kBM - 1) / T::kBM, tiles_n = (p.N + T::kBN - 1) / T::kBN;
    const bool xs4 = !p.w_shuffled && p.xs_k == 1 && p.xs_m == p.kblocks && (p.kblocks & 3) == 0 && ((uintptr_t)p.xs & 15) == 0;
    const bool bf  = out_dtype == In16::bf16;
    const bool folds = fold_kb > 0 && fold_kb < p.kblocks;
    auto kernel = folds ? ring_kernel<true>(p.w_shuffled, xs4, bf) : ring_kernel<false>(p.w_shuffled, xs4, bf);
    const size_t smem = T::lds_bytes(xs4);
    // the opt-in to more than 64 KiB of LDS, per device and instantiation, once (racing first calls repeat it)
    constexpr int kMaxDevices = 64;
    static std::atomic<bool> ready[kMaxDevices][12];
    const int  inst = (p.w_shuffled ? 2 : xs4 ? 4 : 0) + (bf ? 0 : 1) + (folds ? 6 : 0);
    if(device < 0 || device >= kMaxDevices || !ready[device][inst])
    {
        const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
        if(e != hipSuccess)
            return e;
        if(device >= 0 && device < kMaxDevices)
            ready[device][inst] = true;
    }
    // one workgroup fills a compute unit; a multiple of 8, the same number on each XCD
    const int total = tiles_m * tiles_n, grid = std::min(std::max(cus, 8), total + 7) & ~7;
    void*      parked = nullptr;
    WorkspaceLock lock(folds);
    if(folds)
    {
        const hipError_t e = workspace_acquire(ctx, lock, WsKind::split_partial, (size_t)grid * kParkedBytes, false, &parked);
        if(e != hipSuccess)
            return e;
    }
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(kRingThreads), smem, ctx.stream, p, tiles_m, tiles_n, folds ? fold_kb : 0, (float*)parked);
    return hipGetLastError();
}

} // namespace fp8bs
