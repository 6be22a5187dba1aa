// Block-scale mixture of experts, many rows per expert: the two grouped GEMMs on 128-row tiles.
//
// DeepSeek-V3's routed experts (256, top-8, dim 7168, inter 256), the layer on 2048 / 4096 / 8192 tokens: 563 / 958 / 1764
// us block by block, 517 / 694 / 1038 in tiles, with the same bits.
//
// The kernels of moe_kernels.hip walk the sorted rows in blocks of 32 (or pairs of them) and stream an expert's weights
// once per block: right while the weights are what the layer reads, but with hundreds of rows per expert the same
// weights pass through the caches many times and the matrix pipes wait.  Here the sorted rows are cut into tiles of up
// to 128 rows of one expert, and
//   moe_prefill_gate_up  multiplies a tile by 128 gate and 128 up rows, 64 and 64 at a time, with the ring of gemm_ring.h,
//                        applies the activation, and quantises the product 1x128 in the same kernel;
//   moe_prefill_down     keeps a tile's activation rows in LDS (K = inter_dim of one or two K blocks) and streams the
//                        expert's down weights past them straight into operand registers; longer K takes the ring.
// The per-token sum is moe_kernels.hip's.
#include "gemm_ring.h"
#include "moe_launch.h"
#include "moe_rules.h"
#include "quant_stage.h"

#include <algorithm>
#include <atomic>

namespace fp8bs {

namespace {

constexpr int kTileBlocks = 4;                // sorted blocks of 32 rows per tile
constexpr int kTileRows   = 32 * kTileBlocks; // = RingTile<4>::kBM
static_assert(kTileRows == kTileRowsOfExpert, "the rule counts such tiles");

struct PrefillParams
{
    const uint8_t* xq;  // gate/up: tokens [M][lda]; down: [slots][K] by sorted slot
    const float*   xs;  // [rows of xq][xs_stride], 16-byte aligned rows
    const uint8_t* w;   // [experts][N][K], pre-shuffled (16,16) per expert
    const float*   wsc; // [experts][N/128][K/128]
    const int32_t* sorted_ids;
    const int32_t* tiles;  // [0] the number of tiles, then from [2] on {first block, blocks | expert << 8} each
    uint8_t*       hq;     // gate/up: codes of the activation product [slots][inter]
    float*         hs;     // and their scales [slots][hs_stride]
    void*          y;      // down: rows [slots][N], bf16 or fp32
    int64_t        lda;
    int32_t        M, K, N, inter, kblocks, xs_stride, hs_stride;
    int32_t        col_splits; // down from registers: parts a tile's columns are cut into
};

// The tiles of the sorted rows, by one workgroup, and the position of each (token, slot) pair (-1: none), by the others.
struct PrepParams
{
    const int32_t* sorted_ids;
    const int32_t* sorted_expert_ids;
    const int32_t* num_valid;
    int32_t*       tiles;
    int32_t*       where;
    int32_t        M, topk, experts, max_padded, expert_shift;
};
__global__ __launch_bounds__(1024) void moe_prefill_prep_kernel(PrepParams p)
{
    const int valid_rows = min(p.num_valid[0], p.max_padded);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    if(blockIdx.x > 0)
    {
        const int at = ((int)blockIdx.x - 1) * 1024 + t;
        if(at < valid_rows)
        {
            const int id = p.sorted_ids[at], token = id & 0xffffff, slot = (id >> 24) & 0xff;
            const int e  = p.sorted_expert_ids[(at >> 5) >> p.expert_shift];
            if(token < p.M && slot < p.topk) // (a block of an expert that is not held here has no tile, and its rows no sums)
                p.where[(size_t)token * p.topk + slot] = e >= 0 && e < p.experts ? at : -1;
        }
        return;
    }
    // A tile starts at every fourth block of an expert's run of blocks.  1024 blocks at a time: each wave's last run
    // start and its number of tiles are exchanged through LDS.
    __shared__ int last_start[16], wave_tiles[16];
    const int valid = (valid_rows + 31) / 32;
    int       carry_start = 0, carry_tiles = 0;
    for(int base = 0; base < valid; base += 1024)
    {
        const int  b  = base + t;
        const bool in = b < valid;
        const int  e  = in ? p.sorted_expert_ids[b >> p.expert_shift] : -1;
        const int  before = in && b > 0 ? p.sorted_expert_ids[(b - 1) >> p.expert_shift] : -2;
        const uint64_t starts = __ballot(in && e != before);
        if(lane == 63)
            last_start[wave] = starts ? base + wave * 64 + 63 - __builtin_clzll(starts) : -1;
        __syncthreads();
        int run = carry_start;
        for(int w = 0; w < wave; ++w)
            run = last_start[w] >= 0 ? last_start[w] : run;
        const uint64_t mine = starts & (~(uint64_t)0 >> (63 - lane));
        run                 = mine ? base + wave * 64 + 63 - __builtin_clzll(mine) : run;
        const bool     tile = in && e >= 0 && e < p.experts && ((b - run) & (kTileBlocks - 1)) == 0;
        const uint64_t tm   = __ballot(tile);
        if(lane == 0)
            wave_tiles[wave] = __popcll(tm);
        __syncthreads();
        int at = carry_tiles, all = carry_tiles;
        for(int w = 0; w < 16; ++w)
        {
            at += w < wave ? wave_tiles[w] : 0;
            all += wave_tiles[w];
            carry_start = last_start[w] >= 0 ? last_start[w] : carry_start;
        }
        carry_tiles = all;
        at += __popcll(tm & (((uint64_t)1 << lane) - 1));
        if(tile)
        {
            int n = 1;
            while(n < kTileBlocks && b + n < valid && p.sorted_expert_ids[(b + n) >> p.expert_shift] == e)
                ++n;
            p.tiles[2 + 2 * at]     = b;
            p.tiles[2 + 2 * at + 1] = n | e << 8;
        }
        __syncthreads();
    }
    if(t == 0)
        p.tiles[0] = carry_tiles;
}

// [K/128][M] scales, as the quantiser and the entry point have them, to rows of `stride` floats in the order in which the
// first GEMM takes its K blocks
__global__ __launch_bounds__(256) void moe_scale_rows_kernel(const float* __restrict__ in, float* __restrict__ out, int32_t M,
                                                             int32_t kblocks, int32_t stride)
{
    const int m = blockIdx.x * 256 + threadIdx.x, pos = blockIdx.y;
    if(m < M)
        out[(size_t)m * stride + pos] = in[(size_t)ring_kblock<kGateUpWaves>(pos, kblocks) * M + m];
}

// Items (tile, part of its columns) in tile order.  Each of the 8 XCDs takes a contiguous eighth of them, and its
// workgroups (they go round robin over the XCDs) take neighbouring items at the same time: the parts of a tile share its
// rows and the tiles of an expert share its weights in that XCD's L2.
struct Items
{
    int at, end, step;
};
__device__ __forceinline__ Items items_of_workgroup(int items)
{
    const int xcd = blockIdx.x & 7, lo = (int)((int64_t)items * xcd / 8), hi = (int)((int64_t)items * (xcd + 1) / 8);
    return Items{lo + ((int)blockIdx.x >> 3), hi, (int)gridDim.x >> 3};
}

template <int ACT> // 0 silu, 1 gelu (erf form)
__device__ __forceinline__ float prefill_activate(float g)
{
    return ACT == 0 ? g / (1.f + expf(-g)) : 0.5f * g * (1.f + erff(g * 0.70710678118654752f));
}

template <int NF>
__device__ __forceinline__ void zero_acc(float (&acc)[NF][4][4])
{
#pragma unroll
    for(int i = 0; i < NF; ++i)
#pragma unroll
        for(int j = 0; j < 4; ++j)
#pragma unroll
            for(int r = 0; r < 4; ++r)
                acc[i][j][r] = 0.f;
}

// First GEMM, activation and quantisation: item = (tile, 128 columns of the product), in two halves of 64 columns, each a
// 128 x 128 tile of the ring: its weight rows are 64 gate and 64 up rows, dealt out so that a wave holds 16 gate columns and
// the 16 up columns that belong to them, and the activation product is formed in registers.  It is rounded to bf16, as it
// would be stored, and a row's 128 columns -- one group of the quantiser -- meet in LDS: the first half's wait behind the
// ring while the second is multiplied, the second's land where the stages were.
//
// The sums are those of the block-wise kernel: kGateUpWaves chains of every kGateUpWaves-th K block, added one after the
// other.  An fp8 code of the product follows from a sum's last bits now and then, so that the order is part of the result, and
// one chain over all K blocks is the less precise of the two (against 64 bits 2.1125e-3, with eight 2.1115e-3).  That takes a second set of sums per wave, and with it half the
// columns per tile: 32 KiB taken in per K block where a 256 x 128 tile takes 48 for twice the products.  Bound by that
// intake: 8192 tokens (256 rows per expert) 445 us, where the block-wise kernel takes 826 and 256 x 128 tiles with one chain
// 345.  (No 256 x 128 tile holds both sets: 168 registers per wave of twelve; parked in memory they would add 256 KiB of
// intake per chain.)
constexpr uint32_t kHPitch = 144; // bytes per row of half a product (64 columns, bf16) in LDS
using GateUpTile = RingTile<4, 2>;
constexpr size_t kGateUpLds = GateUpTile::lds_bytes(true) + kTileRows * kHPitch;
static_assert(kGateUpLds <= 160 * 1024 && kTileRows * kHPitch <= GateUpTile::kWindows, "LDS");
template <int ACT>
__global__ __launch_bounds__(kRingThreads) void moe_prefill_gate_up_kernel(PrefillParams p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    using T = GateUpTile;
    constexpr int C = kGateUpWaves;
    static_assert(T::kBM == kTileRows, "a tile's rows");
    typedef u32x2 __attribute__((address_space(3)))*       lds_u2_ptr;
    typedef const u32x4 __attribute__((address_space(3)))* lds_u4_ptr;
    const lds_byte_ptr smem3 = (lds_byte_ptr)smem;
    auto h_lds = [&](int half) -> lds_byte_ptr { return smem3 + (half == 0 ? (uint32_t)T::lds_bytes(true) : 0u); };
    const int groups = p.inter / 128;
    Items     it     = items_of_workgroup(p.tiles[0] * groups);
    for(; it.at < it.end; it.at += it.step)
    {
        const int tile = it.at / groups, grp = it.at - tile * groups;
        const int first  = __builtin_amdgcn_readfirstlane(p.tiles[2 + 2 * tile]) * 32;
        const int info   = __builtin_amdgcn_readfirstlane(p.tiles[3 + 2 * tile]);
        const int rows   = (info & 0xff) * 32, expert = info >> 8;
        int       t      = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
        const int l16 = lane & 15, kg = lane >> 4;
        const int wn = wave & 3, wm = wave >> 2;

        // padding rows, and rows past the tile's blocks, are computed on some token and never read
        auto token_of = [&](int row) -> uint32_t {
            const int id = p.sorted_ids[first + min(row, rows - 1)] & 0xffffff;
            return (uint32_t)(id < p.M ? id : 0);
        };
        RingSource<T> src;
        src.wq      = p.w + (size_t)expert * (size_t)p.N * (size_t)p.K;
        src.xq      = p.xq;
        src.xs      = (const uint8_t*)p.xs;
        src.kblocks = p.kblocks;
        src.xs_step = 4u;
        if(wave >= kRingMulWaves)
        {
            const int f = wave - kRingMulWaves;
#pragma unroll
            for(int i = 0; i < T::kLoads; ++i)
            {
                const RingUnit v = ring_unit(i, f, lane);
                if(i < T::kWLoads)
                {
                    const uint32_t q   = v.u >> 1; // slab tile q: multiplying wave q / 2's gate (even) or up tile
                    const uint32_t col = (uint32_t)grp * 8u + (q >> 1) + ((q & 1u) ? (uint32_t)p.inter >> 4 : 0u);
                    src.goff[i]        = col * 16u * (uint32_t)p.K + (v.u & 1u) * 1024u + (uint32_t)lane * 16u;
                }
                else
                    src.goff[i] = token_of((int)v.row - T::kBN) * (uint32_t)p.lda + v.chunk * 16u;
            }
            src.xs_goff = token_of(64 * (f & 1) + lane) * (uint32_t)p.xs_stride * 4u;
            ring_fetch<T, true, true, C>(smem3, src, f);
#pragma unroll
            for(int i = 0; i < T::kWLoads; ++i)
                src.goff[i] += 64u * (uint32_t)p.K; // four tiles on: the other half of the columns
            ring_fetch<T, true, true, C>(smem3, src, f);
            __syncthreads();
            __syncthreads();
            continue;
        }
        src.ws_row[0] = p.wsc + ((size_t)expert * (p.N / 128) + grp) * p.kblocks;
        src.ws_row[1] = src.ws_row[0] + (size_t)groups * p.kblocks;

#pragma nounroll
        for(int half = 0; half < 2; ++half)
        {
            float acc[T::kFrags][4][4], sum[T::kFrags][4][4];
            float ws_vec[2] = {ring_ws_window<C>(src.ws_row[0], p.kblocks, 0, lane), ring_ws_window<C>(src.ws_row[1], p.kblocks, 0, lane)};
            zero_acc(sum);
            const int chains = min(p.kblocks, C);
#pragma nounroll
            for(int r = 0; r < chains; ++r)
            {
                zero_acc(acc);
                ring_multiply<T, true, true, 2, C>(smem3, src, wave, lane, ring_first_position<C>(r, p.kblocks),
                                                   ring_first_position<C>(r + 1, p.kblocks), wm * 64 < rows, ws_vec, acc);
#pragma unroll
                for(int q = 0; q < 16 * T::kFrags; ++q)
                    sum[q >> 4][(q >> 2) & 3][q & 3] += acc[q >> 4][(q >> 2) & 3][q & 3];
            }
            const lds_byte_ptr h_at = h_lds(half) + (uint32_t)(wm * 64 + l16) * kHPitch + (uint32_t)(wn * 16 + kg * 4) * 2u;
#pragma unroll
            for(int j = 0; j < 4; ++j)
            {
                float h[4];
#pragma unroll
                for(int r = 0; r < 4; ++r)
                    h[r] = prefill_activate<ACT>(sum[0][j][r]) * sum[1][j][r];
                *(lds_u2_ptr)(h_at + (uint32_t)j * 16u * kHPitch) =
                    u32x2{pack2<In16::bf16>(h[0], h[1]), pack2<In16::bf16>(h[2], h[3])};
            }
        }
        __syncthreads();
        // eight lanes per row, 16 columns each
#pragma unroll
        for(int u = 0; u < kTileRows * 8 / kRingMulThreads; ++u)
        {
            const int row = (u * kRingMulThreads + t) >> 3, part = t & 7;
            if(row >= rows) // (uniform over a row's eight lanes)
                continue;
            const lds_byte_ptr at = h_lds(part >> 2) + (uint32_t)row * kHPitch + (uint32_t)(part & 3) * 32u;
            const u32x4 lo = *(lds_u4_ptr)at;
            const u32x4 hi = *(lds_u4_ptr)(at + 16u);
            float       v[16], scale;
            unpack8<In16::bf16>(lo, v);
            unpack8<In16::bf16>(hi, v + 8);
            u32x4 codes;
            quant16<In16::bf16, 8>(lo, hi, v, codes, scale);
            *(u32x4*)(p.hq + (size_t)(first + row) * p.inter + grp * 128 + part * 16) = codes;
            if(part == 0)
                p.hs[(size_t)(first + row) * p.hs_stride + grp] = scale;
        }
        __syncthreads(); // the next item's slabs land where the product was
    }
}

// Second GEMM on the ring, for K of three and more K blocks: item = (tile, 256 columns).  F32: rows kept in fp32.
template <bool F32>
__global__ __launch_bounds__(kRingThreads) void moe_prefill_down_ring_kernel(PrefillParams p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    using T = RingTile<4>;
    constexpr uint32_t kSize = F32 ? 4 : 2, kPitch = 64 * kSize + 16; // bytes per row of a wave's 64 x 64 output block in LDS
    constexpr int      kLanes = 4 * kSize;                            // lanes that store a row of it, 16 bytes each
    static_assert(8 * 64 * kPitch <= T::kWindows, "LDS");
    const lds_byte_ptr smem3 = (lds_byte_ptr)smem;
    const int parts = p.N / T::kBN;
    Items     it    = items_of_workgroup(p.tiles[0] * parts);
    for(; it.at < it.end; it.at += it.step)
    {
        const int tile = it.at / parts, n0 = (it.at - tile * parts) * T::kBN;
        const int first = __builtin_amdgcn_readfirstlane(p.tiles[2 + 2 * tile]) * 32;
        const int info  = __builtin_amdgcn_readfirstlane(p.tiles[3 + 2 * tile]);
        const int rows  = (info & 0xff) * 32, expert = info >> 8;
        int       t     = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
        const int l16 = lane & 15, kg = lane >> 4;
        const int wn = wave & 3, wm = wave >> 2;
        RingSource<T> src;
        src.wq      = p.w + (size_t)expert * (size_t)p.N * (size_t)p.K;
        src.xq      = p.xq + (size_t)first * p.K;
        src.xs      = (const uint8_t*)(p.xs + (size_t)first * p.xs_stride);
        src.kblocks = p.kblocks;
        src.xs_step = 4u;
        if(wave >= kRingMulWaves)
        {
            const int f = wave - kRingMulWaves;
#pragma unroll
            for(int i = 0; i < T::kLoads; ++i)
            {
                const RingUnit v = ring_unit(i, f, lane);
                if(i < T::kWLoads)
                    src.goff[i] = (((uint32_t)n0 >> 4) + (v.u >> 1)) * 16u * (uint32_t)p.K + (v.u & 1u) * 1024u + (uint32_t)lane * 16u;
                else
                    src.goff[i] = min(v.row - (uint32_t)T::kBN, (uint32_t)rows - 1u) * (uint32_t)p.K + v.chunk * 16u;
            }
            src.xs_goff = min(64u * (f & 1) + lane, (uint32_t)rows - 1u) * (uint32_t)p.xs_stride * 4u;
            ring_fetch<T, true, true>(smem3, src, f);
            __syncthreads();
            continue;
        }
        src.ws_row[0] = src.ws_row[1] = p.wsc + ((size_t)expert * (p.N / 128) + (n0 + wn * 64) / 128) * p.kblocks;

        float acc[T::kFrags][4][4], ws_vec[1] = {ring_ws_window<0>(src.ws_row[0], p.kblocks, 0, lane)};
        zero_acc(acc);
        ring_multiply<T, true, true, 1>(smem3, src, wave, lane, 0, p.kblocks, wm * 64 < rows, ws_vec, acc);

        const uint32_t ebase = (uint32_t)wave * (64u * kPitch);
        typedef f32x4 __attribute__((address_space(3)))*       lds_f4_ptr;
        typedef u32x2 __attribute__((address_space(3)))*       lds_u2_ptr;
        typedef const u32x4 __attribute__((address_space(3)))* lds_u4_ptr;
#pragma unroll
        for(int j = 0; j < 4; ++j)
#pragma unroll
            for(int i = 0; i < T::kFrags; ++i)
            {
                const lds_byte_ptr at = smem3 + ebase + (uint32_t)(j * 16 + l16) * kPitch + (uint32_t)(i * 16 + kg * 4) * kSize;
                if constexpr(F32)
                    *(lds_f4_ptr)at = f32x4{acc[i][j][0], acc[i][j][1], acc[i][j][2], acc[i][j][3]};
                else
                    *(lds_u2_ptr)at = u32x2{pack2<In16::bf16>(acc[i][j][0], acc[i][j][1]), pack2<In16::bf16>(acc[i][j][2], acc[i][j][3])};
            }
        const int piece = lane % kLanes;
#pragma unroll
        for(int c = 0; c < kLanes; ++c)
        {
            const int   row = c * (64 / kLanes) + lane / kLanes;
            const u32x4 v   = *(lds_u4_ptr)(smem3 + ebase + (uint32_t)row * kPitch + (uint32_t)piece * 16u);
            if(wm * 64 + row < rows)
                *(u32x4*)((uint8_t*)p.y + ((size_t)(first + wm * 64 + row) * p.N + n0 + wn * 64) * kSize + piece * 16) = v;
        }
        __syncthreads();
    }
}

// Second GEMM for K of one or two K blocks: the tile's rows (K codes each) wait in LDS, and each wave walks groups of 64
// columns -- four 16-column weight tiles, loaded straight into operand registers by this wave alone -- with the next
// group requested while one is multiplied by the tile's rows, 16 at a time.  The 16 x 64 results leave through an LDS
// region of the wave's own as whole 128-byte lines.  Bound by memory: the rows written and the weights read; what it
// takes is requests in flight, 16 KiB per wave here.  8192 tokens: 295 us for 0.94 GB of rows and 0.47 GB of weights (4.8
// TB/s, a plain copy runs at 5.1); with the rows in registers and one weight tile ahead 367 us, block by block 583.
constexpr int      kDownWaves = 4;
constexpr uint32_t down_pitch(bool f32) { return f32 ? 272u : 144u; }
constexpr uint32_t down_x_bytes(int kb) { return (uint32_t)kb * kTileRows * 128u; }
constexpr uint32_t down_lds_bytes(int kb, bool f32) { return down_x_bytes(kb) + (uint32_t)kb * kTileRows * 4u + kDownWaves * 16u * down_pitch(f32); }

template <int KB, bool F32>
__global__ __launch_bounds__(64 * kDownWaves, 2) void moe_prefill_down_kernel(PrefillParams p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    constexpr uint32_t kSize = F32 ? 4 : 2, kPitch = down_pitch(F32);
    constexpr int      kLanes = 4 * kSize; // lanes that store 64 columns of a row, 16 bytes each
    typedef float __attribute__((address_space(3)))*       lds_float_ptr;
    typedef f32x4 __attribute__((address_space(3)))*       lds_f4_ptr;
    typedef u32x2 __attribute__((address_space(3)))*       lds_u2_ptr;
    typedef const u32x4 __attribute__((address_space(3)))* lds_u4_ptr;
    typedef const i32x4 __attribute__((address_space(3)))* lds_i4_ptr;
    const lds_byte_ptr smem3 = (lds_byte_ptr)smem;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6), l16 = lane & 15, kg = lane >> 4;
    const lds_byte_ptr  stage  = smem3 + down_x_bytes(KB) + KB * kTileRows * 4 + (uint32_t)wave * (16u * kPitch);
    const lds_float_ptr xs_lds = (lds_float_ptr)(smem3 + down_x_bytes(KB)); // [KB][rows]
    const uint32_t sw     = lds_swizzle((uint32_t)l16);
    const uint32_t lo_off = (uint32_t)l16 * 128u + (((2u * kg) ^ sw) << 4);
    const uint32_t hi_off = (uint32_t)l16 * 128u + (((2u * kg + 1u) ^ sw) << 4);
    const int groups = p.N / 64;
    Items     it     = items_of_workgroup(p.tiles[0] * p.col_splits);
    for(; it.at < it.end; it.at += it.step)
    {
        const int tile  = it.at / p.col_splits, part = it.at - tile * p.col_splits;
        const int first = __builtin_amdgcn_readfirstlane(p.tiles[2 + 2 * tile]) * 32;
        const int info  = __builtin_amdgcn_readfirstlane(p.tiles[3 + 2 * tile]);
        const int rows  = (info & 0xff) * 32, expert = info >> 8;
        int       grp = groups * part / p.col_splits + wave;
        const int grp_end = groups * (part + 1) / p.col_splits;

        const uint8_t* wexp = p.w + (size_t)expert * (size_t)p.N * (KB * 128) + kg * 512 + l16 * 16;
        const float*   wsr  = p.wsc + (size_t)expert * (p.N / 128) * KB;
        auto fetch = [&](int g, i32x8 (&w)[4][KB], float (&ws)[KB]) {
#pragma unroll
            for(int i = 0; i < 4; ++i)
#pragma unroll
                for(int kb = 0; kb < KB; ++kb)
                {
                    const i32x4* src = (const i32x4*)(wexp + ((size_t)(g * 4 + i) * KB + kb) * 2048);
                    const i32x4  lo = src[0], hi = src[16];
                    w[i][kb] = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                }
#pragma unroll
            for(int kb = 0; kb < KB; ++kb)
                ws[kb] = wsr[(size_t)(g >> 1) * KB + kb];
        };
        auto multiply = [&](int g, const i32x8 (&w)[4][KB], const float (&ws)[KB]) {
            for(int j = 0; j < rows / 16; ++j)
            {
                i32x8 x[KB];
                float sc[KB];
#pragma unroll
                for(int kb = 0; kb < KB; ++kb)
                {
                    const i32x4 lo = *(lds_i4_ptr)(smem3 + (uint32_t)(kb * kTileRows + j * 16) * 128u + lo_off);
                    const i32x4 hi = *(lds_i4_ptr)(smem3 + (uint32_t)(kb * kTileRows + j * 16) * 128u + hi_off);
                    x[kb]  = i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                    sc[kb] = xs_lds[kb * kTileRows + j * 16 + l16] * ws[kb];
                }
#pragma unroll
                for(int i = 0; i < 4; ++i)
                {
                    f32x4 acc = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for(int kb = 0; kb < KB; ++kb)
                    {
                        const f32x4 prod = mfma_16x16x128_fp8(w[i][kb], x[kb], f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
                        for(int c = 0; c < 4; ++c)
                            acc[c] = __builtin_fmaf(prod[c], sc[kb], acc[c]);
                    }
                    const lds_byte_ptr at = stage + (uint32_t)l16 * kPitch + (uint32_t)(i * 16 + kg * 4) * kSize;
                    if constexpr(F32)
                        *(lds_f4_ptr)at = acc;
                    else
                        *(lds_u2_ptr)at = u32x2{pack2<In16::bf16>(acc[0], acc[1]), pack2<In16::bf16>(acc[2], acc[3])};
                }
                // (a wave's LDS operations complete in the order they were issued)
#pragma unroll
                for(int h = 0; h < kLanes / 4; ++h)
                {
                    const int   row = h * (64 / kLanes) + lane / kLanes, c = lane % kLanes;
                    const u32x4 v   = *(lds_u4_ptr)(stage + (uint32_t)row * kPitch + (uint32_t)c * 16u);
                    *(u32x4*)((uint8_t*)p.y + ((size_t)(first + j * 16 + row) * p.N + g * 64) * kSize + c * 16) = v;
                }
            }
        };

        __syncthreads(); // the previous item's rows are no longer read
        for(int u = wave; u < rows / 8 * KB; u += kDownWaves)
        {
            const int      kb = u / (rows / 8), r8 = u - kb * (rows / 8);
            const uint32_t r  = (uint32_t)r8 * 8u + ((uint32_t)lane >> 3), c = ((uint32_t)lane & 7u) ^ lds_swizzle(r);
            ring_dma16(__builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(smem3 + (uint32_t)(kb * kTileRows + r8 * 8) * 128u)),
                       r * (KB * 128u) + kb * 128u + c * 16u, p.xq + (size_t)first * (KB * 128));
        }
        if(t < rows)
        {
#pragma unroll
            for(int kb = 0; kb < KB; ++kb)
                xs_lds[kb * kTileRows + t] = p.xs[(size_t)(first + t) * p.xs_stride + kb];
        }
        i32x8 wa[4][KB], wb[4][KB];
        float sa[KB], sb[KB];
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if(grp < grp_end)
            fetch(grp, wa, sa);
        for(; grp < grp_end; grp += 2 * kDownWaves)
        {
            const bool more = grp + kDownWaves < grp_end;
            if(more)
                fetch(grp + kDownWaves, wb, sb);
            multiply(grp, wa, sa);
            if(!more)
                break;
            if(grp + 2 * kDownWaves < grp_end)
                fetch(grp + 2 * kDownWaves, wa, sa);
            multiply(grp + kDownWaves, wb, sb);
        }
    }
}

size_t align_up(size_t v) { return (v + 255) & ~(size_t)255; }
int    row_floats(int kblocks) { return (kblocks + 3) & ~3; } // a row of scales that is read 16 bytes at a time
size_t tiles_bytes(const MoeArgs& a) { return align_up(((size_t)a.max_blocks + 1) * 8); }

hipError_t raise_lds(const void* kernel, size_t bytes, int device, std::atomic<bool> (&ready)[64])
{
    if(device >= 0 && device < 64 && ready[device])
        return hipSuccess;
    const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
    if(e == hipSuccess && device >= 0 && device < 64)
        ready[device] = true;
    return e;
}

} // namespace

bool moe_prefill_wanted(const MoeArgs& a)
{
    // arrays sorted in blocks of 32 or multiples; 32-bit byte offsets inside the token matrix, its scales and an expert
    const uint64_t lda = a.x16 ? (uint64_t)a.dim : (uint64_t)a.lda;
    if(a.block_rows != 32 || (uint64_t)a.M * lda >= (1ull << 32) || (uint64_t)a.M * row_floats(a.dim / 128) * 4 >= (1ull << 32) ||
       (uint64_t)2 * a.inter * a.dim >= (1ull << 32) || a.experts >= (1 << 23))
        return false;
    if(a.tiles128 >= 0)
        return a.tiles128 != 0;
    if(moe_down_by_columns(a)) // few tokens, whose sums never leave fp32
        return false;
    const int64_t pairs = (int64_t)a.M * a.topk;
    const int64_t all   = routed_experts(pairs, a.topk, a.block_rows << a.expert_shift, a.max_padded, a.experts);
    return tiles_win(pairs, all, a.experts, a.inter);
}

size_t moe_prefill_workspace_bytes(const MoeArgs& a)
{
    const size_t slots = (size_t)a.max_padded;
    size_t       b     = align_up(slots * a.inter) + align_up(slots * row_floats(a.inter / 128) * 4) + align_up(slots * a.dim * (moe_rows_in_f32(a) ? 4 : 2)) +
               align_up((size_t)a.M * a.topk * 4) + tiles_bytes(a) + align_up((size_t)a.M * row_floats(a.dim / 128) * 4);
    if(a.x16)
        b += align_up((size_t)a.M * a.dim) + align_up((size_t)a.M * (a.dim / 128) * 4);
    return b;
}

hipError_t launch_moe_prefill_gemms(const MoeArgs& a, hipStream_t stream, void* scratch, void** rows, int32_t** where)
{
    uint8_t*     ws    = (uint8_t*)scratch;
    auto         take  = [&](size_t bytes) { uint8_t* at = ws; ws += align_up(bytes); return at; };
    const size_t slots = (size_t)a.max_padded;
    uint8_t*  hq = take(slots * a.inter);
    float*    hs = (float*)take(slots * row_floats(a.inter / 128) * 4);
    const bool f32 = moe_rows_in_f32(a);
    void*     y  = take(slots * a.dim * (f32 ? 4 : 2));
    *where = (int32_t*)take((size_t)a.M * a.topk * 4);
    *rows  = y;
    int32_t* tiles = (int32_t*)take(tiles_bytes(a));
    float*   xs    = (float*)take((size_t)a.M * row_floats(a.dim / 128) * 4);
    hipError_t e;

    PrepParams pp{a.sorted_ids, a.sorted_expert_ids, a.num_valid, tiles, *where, a.M, a.topk, a.experts, a.max_padded, a.expert_shift};
    hipLaunchKernelGGL(moe_prefill_prep_kernel, dim3(1 + (a.max_padded + 1023) / 1024), dim3(1024), 0, stream, pp);

    const uint8_t* xq    = a.xq;
    const float*   xs_in = a.xs;
    int64_t        lda   = a.lda;
    if(a.x16)
    {
        uint8_t*  q = take((size_t)a.M * a.dim);
        float*    s = (float*)take((size_t)a.M * (a.dim / 128) * 4);
        QuantArgs qa{};
        qa.x                = a.x16;
        qa.y                = q;
        qa.scale            = s;
        qa.rows             = a.M;
        qa.groups_per_row   = a.dim / 128;
        qa.group            = 128;
        qa.num_rows_factor  = 1;
        qa.dtype            = a.x16_dtype;
        qa.transpose_scale  = true;
        if((e = launch_group_quant(qa, stream)) != hipSuccess)
            return e;
        xq    = q;
        xs_in = s;
        lda   = a.dim;
    }
    hipLaunchKernelGGL(moe_scale_rows_kernel, dim3((a.M + 255) / 256, a.dim / 128), dim3(256), 0, stream, xs_in, xs, a.M, a.dim / 128,
                       row_floats(a.dim / 128));

    static std::atomic<bool> ready[8][64];
    constexpr size_t kRingLds = RingTile<4>::lds_bytes(true);
    PrefillParams    g{};
    g.xq         = xq;
    g.xs         = xs;
    g.xs_stride  = row_floats(a.dim / 128);
    g.w          = a.w1;
    g.wsc        = a.w1_scale;
    g.sorted_ids = a.sorted_ids;
    g.tiles      = tiles;
    g.hq         = hq;
    g.hs         = hs;
    g.hs_stride  = row_floats(a.inter / 128);
    g.lda        = lda;
    g.M          = a.M;
    g.K          = a.dim;
    g.N          = 2 * a.inter;
    g.inter      = a.inter;
    g.kblocks    = a.dim / 128;
    auto gate_up = a.activation == 0 ? moe_prefill_gate_up_kernel<0> : moe_prefill_gate_up_kernel<1>;
    if((e = raise_lds((const void*)gate_up, kGateUpLds, a.device_id, ready[a.activation == 0 ? 0 : 1])) != hipSuccess)
        return e;
    hipLaunchKernelGGL(gate_up, dim3(256), dim3(kRingThreads), kGateUpLds, stream, g);

    PrefillParams d = g;
    d.xq        = hq;
    d.xs        = hs;
    d.xs_stride = g.hs_stride;
    d.w         = a.w2;
    d.wsc       = a.w2_scale;
    d.y         = y;
    d.K         = a.inter;
    d.N         = a.dim;
    d.kblocks   = a.inter / 128;
    d.lda       = a.inter;
    if(d.kblocks <= 2)
    {
        // each wave of an item walks about seven groups of columns: enough to amortise the tile's rows, and enough items
        d.col_splits = std::max(1, a.dim / 64 / (7 * kDownWaves));
        const size_t lds = down_lds_bytes(d.kblocks, f32);
        auto kernel = d.kblocks == 1 ? (f32 ? moe_prefill_down_kernel<1, true> : moe_prefill_down_kernel<1, false>)
                                     : (f32 ? moe_prefill_down_kernel<2, true> : moe_prefill_down_kernel<2, false>);
        if((e = raise_lds((const void*)kernel, lds, a.device_id, ready[(f32 ? 3 : 1) + d.kblocks])) != hipSuccess)
            return e;
        hipLaunchKernelGGL(kernel, dim3(512), dim3(64 * kDownWaves), lds, stream, d);
    }
    else
    {
        auto kernel = f32 ? moe_prefill_down_ring_kernel<true> : moe_prefill_down_ring_kernel<false>;
        if((e = raise_lds((const void*)kernel, kRingLds, a.device_id, ready[f32 ? 7 : 6])) != hipSuccess)
            return e;
        hipLaunchKernelGGL(kernel, dim3(256), dim3(kRingThreads), kRingLds, stream, d);
    }
    return hipGetLastError();
}

} // namespace fp8bs
