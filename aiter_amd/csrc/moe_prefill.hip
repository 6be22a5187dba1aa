// Block-scale mixture of experts, many rows per expert: the two grouped GEMMs on 128-row tiles.
//
// DeepSeek-V3's routed experts (256, top-8, dim 7168, inter 256), the layer on 2048 / 4096 / 8192 tokens: 563 / 958 / 1764
// us block by block, 464 / 610 / 926 in tiles, with the same bits.
//
// The kernels of moe_kernels.hip walk the sorted rows in blocks of 32 (or pairs of them) and stream an expert's weights
// once per block: right while the weights are what the layer reads, but with hundreds of rows per expert the same
// weights pass through the caches many times and the matrix pipes wait.  Here the sorted rows are cut into tiles of up
// to 128 rows of one expert, and
//   moe_prefill_gate_up  multiplies a tile by 128 gate and 128 up rows, applies the activation, and quantises the product
//                        1x128 in the same kernel;
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

// The order in which the first GEMM takes its K blocks: by their remainder modulo kGateUpWaves, ascending inside a remainder
// -- what that many waves with every so-many-th K block each add up, one wave's share after the other.  The scales of its
// rows are laid out in that order, weights and activations are not.
__device__ __forceinline__ int chain_kblock(int pos, int kblocks)
{
    constexpr int C = kGateUpWaves;
    const int q = kblocks / C, longer = (kblocks % C) * (q + 1); // the first kblocks % C remainders have one block more
    const bool in = pos < longer;
    const int  n = in ? q + 1 : max(q, 1), at = in ? pos : pos - longer;
    const int  r = at / n;
    return (in ? 0 : kblocks % C) + r + C * (at - r * n);
}
__device__ __forceinline__ int chain_start(int r, int kblocks) // where remainder r starts in it
{
    return r * (kblocks / kGateUpWaves) + min(r, kblocks % kGateUpWaves);
}

// [K/128][M] scales, as the quantiser and the entry point have them, to rows of `stride` floats in the order in which the
// first GEMM takes its K blocks
__global__ __launch_bounds__(256) void moe_scale_rows_kernel(const float* __restrict__ in, float* __restrict__ out, int32_t M,
                                                             int32_t kblocks, int32_t stride)
{
    const int m = blockIdx.x * 256 + threadIdx.x, pos = blockIdx.y;
    if(m < M)
        out[(size_t)m * stride + pos] = in[(size_t)chain_kblock(pos, kblocks) * M + m];
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

__device__ __forceinline__ void zero_acc(float (&acc)[4][4][4])
{
#pragma unroll
    for(int i = 0; i < 4; ++i)
#pragma unroll
        for(int j = 0; j < 4; ++j)
#pragma unroll
            for(int r = 0; r < 4; ++r)
                acc[i][j][r] = 0.f;
}

// First GEMM, activation and quantisation: item = (tile, 128 columns of the product): 128 rows by 128 gate and 128 up weight
// rows, dealt out over eight waves so that a wave holds 32 gate columns and the 32 up columns that belong to them (64 x 64
// of the tile), and the activation product is formed in registers.  It is rounded to bf16, as it would be stored, and a row's
// 128 columns -- one group of the quantiser -- meet in LDS.
//
// The sums are those of the block-wise kernel: kGateUpWaves chains of every kGateUpWaves-th K block, added one after the
// other.  An fp8 code of the product follows from a sum's last bits now and then, so that the order is part of the result, and
// one chain over all K blocks is the less precise of the two (against 64 bits 2.1125e-3, with eight 2.1115e-3).  That takes a
// second set of sums, 128 registers of sums per lane of a 256-column item: eight waves of 256 registers, which fetch what
// they multiply.  (Waves that only fetch leave twelve waves 168 registers each and the items half the columns: 32 KiB taken
// in per K block where these take 48 for twice the products.)  8192 tokens (256 rows per expert, dim 7168, inter 256): 435
// us with those, 374 with these; 2048 tokens, the layer: 509 and 469.
//
// Bound by what a compute unit can ask for and by its own rhythm: two K blocks are in flight while one is multiplied.  A K
// block takes 1.2 us with rows and weights from memory, 0.9 with both in L2, 0.8 without the loads, 0.67 without reading LDS
// either (a barrier per K block); the matrix pipes need 0.49 at this clock.  An item takes another 10 us: eight chains folded,
// the activation, the quantiser.  What did not change that: fewer scalar instructions around the barrier, the products in
// flight folded behind it, the next item's first K blocks under the activation (which stays: it costs nothing).
constexpr int      kGateUpThreads = 512, kGateUpStages = 3;
constexpr uint32_t kGateUpCols    = 256; // weight rows of an item: 16-row tiles 4 w .. 4 w + 3 are two gate and two up tiles of wave column w
constexpr uint32_t kGateUpWindow  = kTileRows * 16;     // LDS: two windows of four K blocks of the rows' scales, then the stages
constexpr uint32_t kGateUpRing    = 2 * kGateUpWindow;
constexpr uint32_t kGateUpX       = kGateUpCols * 128;  // a stage: weight rows, then the tile's rows, 128 bytes each
constexpr uint32_t kGateUpStage   = kGateUpX + kTileRows * 128;
constexpr uint32_t kGateUpRingEnd = kGateUpRing + kGateUpStages * kGateUpStage;
constexpr uint32_t kHPitch        = 272;                // bytes per row of the product (128 columns, bf16) in LDS
constexpr size_t   kGateUpLds     = kGateUpRingEnd;
static_assert(kGateUpLds <= 160 * 1024, "LDS");
static_assert(kTileRows * kHPitch <= kGateUpStage, "the product lies in one stage: the next item's first K blocks are landing in the others");
static_assert((kGateUpWaves & (kGateUpWaves - 1)) == 0, "remainders by a mask");

#define FP8BS_MFMA(P, A, B) asm volatile("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, 0" : "=&v"(P) : "v"(A), "v"(B))
#define FP8BS_FMA4(ACC, P, S)                                                              \
    do                                                                                     \
    {                                                                                      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[0]) : "v"((P)[0]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[1]) : "v"((P)[1]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[2]) : "v"((P)[2]), "v"(S));      \
        asm volatile("v_fmac_f32 %0, %1, %2" : "+v"((ACC)[3]) : "v"((P)[3]), "v"(S));      \
    } while(0)
// (from asm, so that they stay where they are written: moved, they keep two sets of registers alive)
#define FP8BS_ADD_AND_CLEAR(SUM, ACC) asm volatile("v_add_f32 %0, %0, %1\n\tv_mov_b32 %1, 0" : "+v"(SUM), "+v"(ACC))

template <int ACT>
__global__ __launch_bounds__(kGateUpThreads) void moe_prefill_gate_up_kernel(PrefillParams p)
{
    extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];
    constexpr int C = kGateUpWaves;
    typedef u32x2 __attribute__((address_space(3)))*       lds_u2_ptr;
    typedef const u32x4 __attribute__((address_space(3)))* lds_u4_ptr;
    const lds_byte_ptr smem3 = (lds_byte_ptr)smem;
    const int  groups = p.inter / 128, n = p.kblocks; // n is even, at least 2
    // This XCD's items, in rounds of one per workgroup.  What is left after the last full round is dealt out in halves or
    // quarters of a tile's rows if there are workgroups for them: a K block of 32 rows takes half the time of 128.
    const Items all  = items_of_workgroup(p.tiles[0] * groups);
    const int   lo   = all.at - ((int)blockIdx.x >> 3), step = all.step;
    const int   full = (all.end - lo) / step * step, left = all.end - lo - full;
    const int   cut  = left * 4 <= step ? 4 : left * 2 <= step ? 2 : 1;
    const int   end  = full + left * cut, begin = (int)blockIdx.x >> 3;
    if(begin >= end)
        return;
    const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int last = begin + (end - 1 - begin) / step * step;

    // An item is looked up three ahead (its tile), its rows' tokens two, and its first two K blocks are fetched while the
    // last two of the item before are multiplied, so that they arrive under that one's activation.
    struct Tile
    {
        int block, info, part, grp; // block, info: as in p.tiles, until `uniform` narrows them to the part
    };
    auto tile_of = [&](int at) -> Tile {
        at              = min(at, last);
        const int beyond = at - full;
        const int item  = lo + (beyond < 0 ? at : full + beyond / cut);
        const int32_t* e = p.tiles + 2 + 2 * (item / groups);
        return Tile{e[0], e[1], beyond < 0 ? -1 : beyond % cut, item % groups};
    };
    auto uniform = [&](Tile v) -> Tile {
        const int block = __builtin_amdgcn_readfirstlane(v.block), info = __builtin_amdgcn_readfirstlane(v.info);
        if(v.part < 0)
            return Tile{block, info, -1, v.grp};
        // (fewer blocks than parts: some parts are the same block, with the same results)
        const int n = info & 0xff, from = n * v.part / cut, to = max(from + 1, n * (v.part + 1) / cut);
        return Tile{block + from, (info & ~0xff) | (to - from), v.part, v.grp};
    };
    // padding rows, and rows past the tile's blocks, are computed on some token and never read
    auto id_of    = [&](Tile v, int row) -> int { return p.sorted_ids[v.block * 32 + min(row, (v.info & 0xff) * 32 - 1)]; };
    auto token_of = [&](int id) -> uint32_t { return (uint32_t)((id & 0xffffff) < p.M ? id & 0xffffff : 0); };
    // What this wave fetches of a K block: weight tiles 2 wave and 2 wave + 1 (as they lie: 2 KiB each in fragment order), 16
    // rows, and (waves 0 and 1, every fourth K block) 64 rows of the scales.
    struct Source
    {
        const uint8_t* w;
        uint32_t       x[2], xs;
    };
    auto row_of     = [&](int k) -> int { return wave * 16 + k * 8 + (lane >> 3); };
    auto weights_of = [&](Tile v) -> const uint8_t* {
        return p.w + (size_t)(v.info >> 8) * (size_t)p.N * (size_t)p.K +
               ((size_t)v.grp * 8 + (wave >> 1) * 2 + ((wave & 1) ? p.inter >> 4 : 0)) * 16 * (size_t)p.K;
    };
    auto rows_of = [&](Source& src, int id0, int id1, int ids) {
        src.x[0] = token_of(id0) * (uint32_t)p.lda + ((((uint32_t)lane & 7u) ^ lds_swizzle((uint32_t)row_of(0))) << 4);
        src.x[1] = token_of(id1) * (uint32_t)p.lda + ((((uint32_t)lane & 7u) ^ lds_swizzle((uint32_t)row_of(1))) << 4);
        src.xs   = token_of(ids) * (uint32_t)p.xs_stride * 4u;
    };
    const int xs_row = 64 * (wave & 1) + lane;
    Tile      tile = uniform(tile_of(begin)), tile1 = uniform(tile_of(begin + step)), tile2 = uniform(tile_of(begin + 2 * step));
    Source    src, after; // of the item being fetched and the one after it
    src.w   = weights_of(tile);
    after.w = weights_of(tile1);
    rows_of(src, id_of(tile, row_of(0)), id_of(tile, row_of(1)), id_of(tile, xs_row));
    rows_of(after, id_of(tile1, row_of(0)), id_of(tile1, row_of(1)), id_of(tile1, xs_row));
    // w_scale of the first 64 positions, lane = position; the up tiles' row lies behind the gate tiles'
    const size_t ws_up  = (size_t)groups * n;
    const int    ws_pos = chain_kblock(min(lane, n - 1), n);
    auto ws_row = [&](Tile v) -> const float* { return p.wsc + ((size_t)(v.info >> 8) * (p.N / 128) + v.grp) * n; };
    float ws_vec[2] = {ws_row(tile)[ws_pos], ws_row(tile)[ws_up + ws_pos]};

    const uint32_t lane16 = (uint32_t)lane * 16u;
    const uint32_t lds0   = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)smem3);
    const uint32_t wtile  = 16u * (uint32_t)p.K;
    uint32_t       walk   = 0; // K block fetched next, of position `ahead`
    int            ahead  = 0;
    uint32_t       fetch  = lds0 + kGateUpRing; // and its stage
    uint32_t       window = 0;                  // where the next window of scales lands
    const uint8_t* wnext  = src.w;
    const uint8_t* xnext  = p.xq;
    auto load = [&](int u) { // u: 0 .. 5
        if(u < 4)
            ring_dma16(fetch + (uint32_t)(wave * 4 + u) * 1024u, lane16, wnext + (u >> 1) * wtile + (u & 1) * 1024u);
        else
            ring_dma16(fetch + kGateUpX + (uint32_t)(wave * 2 + u - 4) * 1024u, src.x[u - 4], xnext);
    };
    // whether position `ahead` opens a window of scales that this wave fetches.  (n is even: the other window's last position
    // has been multiplied by then, also where `ahead` belongs to the next item.)
    auto opens   = [&] { return wave < 2 && (ahead & 3) == 0; };
    auto load_xs = [&] { ring_dma16(lds0 + window + (uint32_t)wave * 1024u, src.xs + (uint32_t)ahead * 4u, (const uint8_t*)p.xs); };
    auto advance = [&] { // to the next position, or the first of the next item (behind the last: of that one again, unused)
        window = (ahead & 3) == 0 ? window ^ kGateUpWindow : window;
        fetch  = fetch == lds0 + kGateUpRingEnd - kGateUpStage ? lds0 + kGateUpRing : fetch + kGateUpStage;
        walk   = walk + C < (uint32_t)n ? walk + C : (walk & (C - 1)) + 1;
        ++ahead;
        walk  = ahead == n ? 0 : walk;
        ahead = ahead == n ? 0 : ahead;
        wnext = src.w + (size_t)walk * 2048u;
        xnext = p.xq + (size_t)walk * 128u;
    };
    auto enter = [&] { // ahead of a position's loads
        if(ahead == 0)
        {
            src   = after;
            wnext = src.w;
        }
    };
#pragma unroll
    for(int s = 0; s < 2; ++s)
    {
#pragma unroll
        for(int u = 0; u < 6; ++u)
            load(u);
        if(s == 0 && opens())
            load_xs();
        advance();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    int      stage    = 0; // of the K block being multiplied
    uint32_t scales   = 0; // the window that the item's first scales lie in
    for(int at = begin; at < end; at += step)
    {
        const int rows = (tile.info & 0xff) * 32;
        int       t = threadIdx.x;
        asm volatile("" : "+v"(t));
        const int lane = t & 63, l16 = lane & 15, kg = lane >> 4;
        const int wn = wave & 3, wm = wave >> 2;
        auto h_stage = [&]() -> uint32_t { return kGateUpRing + (uint32_t)(stage == 0 ? kGateUpStages - 1 : stage - 1) * kGateUpStage; };
        int       id[3]; // requested behind the multiply loop: rows of the item after the next, the tile behind it, w_scale
        Tile      tile3;
        float     ws_new[2];
        auto request = [&] {
            id[0]     = id_of(tile2, row_of(0));
            id[1]     = id_of(tile2, row_of(1));
            id[2]     = id_of(tile2, xs_row);
            tile3     = tile_of(at + 3 * step);
            ws_new[0] = ws_row(tile1)[ws_pos];
            ws_new[1] = ws_row(tile1)[ws_up + ws_pos];
        };
        __syncthreads(); // the item's first two K blocks are in LDS, and the product of the one before is no longer read

        if(wm * 64 >= rows) // all padding: only fetches
        {
            for(int pos = 0; pos < n; ++pos)
            {
                const bool xs = opens();
                enter();
                if(xs)
                    load_xs();
#pragma unroll
                for(int u = 0; u < 6; ++u)
                    load(u);
                advance();
                stage = stage == kGateUpStages - 1 ? 0 : stage + 1;
                if(!xs)
                    asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
                asm volatile("s_waitcnt vmcnt(7)" ::: "memory");
                __syncthreads();
            }
            request();
        }
        else
        {
            float sum[4][4][4];
            zero_acc(sum);
            // addresses of this lane's fragments in the stage of the K block being multiplied, and of its rows' scales
            const uint32_t sw     = lds_swizzle((uint32_t)l16);
            const uint32_t on0    = (uint32_t)stage * kGateUpStage;
            const uint32_t x_row  = on0 + kGateUpRing + kGateUpX + (uint32_t)wm * 8192u + (uint32_t)l16 * 128u;
            uint32_t       w_at   = on0 + kGateUpRing + (uint32_t)wn * 8192u + (uint32_t)kg * 512u + (uint32_t)l16 * 16u;
            uint32_t       x_lo   = x_row + (((2u * kg) ^ sw) << 4), x_hi = x_row + (((2u * kg + 1u) ^ sw) << 4);
            const uint32_t xs_lds = ((uint32_t)wm * 64u + (uint32_t)l16) * 16u;
            uint32_t       xs_at  = xs_lds + scales;
            auto frag = [&](uint32_t lo, uint32_t hi) -> i32x8 {
                const i32x4 a = *(lds_vec_ptr)(smem3 + lo);
                const i32x4 b = *(lds_vec_ptr)(smem3 + hi);
                return i32x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
            };
            auto read_w = [&](int i) { return frag(w_at + i * 2048u, w_at + 256u + i * 2048u); };
            auto read_x = [&](int j) { return frag(x_lo + j * 2048u, x_hi + j * 2048u); };

            // The instruction stream of gemm_ring.h, with the next stage's loads between the slots
            float acc[4][4][4];
            zero_acc(acc);
            f32x4 P[4];
            i32x8 bx[4], aw[4];
            float scp[4];
#pragma unroll
            for(int q = 0; q < 4; ++q)
            {
                P[q]   = f32x4{0.f, 0.f, 0.f, 0.f};
                bx[q]  = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
                aw[q]  = i32x8{0, 0, 0, 0, 0, 0, 0, 0};
                scp[q] = 0.f;
            }
            float scg = 0.f, scg3 = 0.f; // the gate tiles' products in flight
#pragma unroll
            for(int q = 0; q < 4; ++q)
            {
                asm volatile("" : "+v"(bx[q]));
                asm volatile("" : "+v"(aw[q]));
            }

            int   chain_at = chain_start(1, n), chain = 1; // where the next chain starts
            float wsg = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ws_vec[0]), 0));
            float wsu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ws_vec[1]), 0));
            bool  xs  = opens();
            for(int pos = 0; pos < n; ++pos)
            {
                asm volatile("s_nop 1" ::: "memory");
                aw[0] = read_w(0);
                float xsv[4], sc[4], scu;
#pragma unroll
                for(int j = 0; j < 4; ++j)
                {
                    xsv[j] = *(lds_f32_ptr)(smem3 + xs_at + j * 256);
                }
#pragma unroll
                for(int q = 0; q < 16; ++q)
                {
                    if(q == 2)
                        aw[1] = read_w(1);
                    if(q < 8) // up tile (2 + q % 2, q / 2) of the previous K block
                        FP8BS_MFMA(P[q & 3], aw[2 + q % 2], bx[q / 2]);
                    else // gate tile ((q - 8) / 4, (q - 8) % 4) of this one
                        FP8BS_MFMA(P[q & 3], aw[(q - 8) >> 2], bx[(q - 8) & 3]);
                    if(q < 8 && (q & 1))
                        bx[q / 2] = read_x(q / 2);
                    if(q == 6 || q == 7)
                        aw[q - 4] = read_w(q - 4);
                    if(q == 0)
                        enter();
                    if((q & 1) && q < 12)
                        load(q >> 1);
                    if(q == 12 && xs)
                        load_xs();
                    if(q < 2)
                        FP8BS_FMA4(acc[1][2 + q], P[2 + q], (q == 0 ? scg : scg3));
                    else if(q < 10)
                        FP8BS_FMA4(acc[2 + q % 2][(q - 2) / 2], P[(q - 2) & 3], scp[(q - 2) / 2]);
                    else
                        FP8BS_FMA4(acc[(q - 10) >> 2][(q - 10) & 3], P[(q - 2) & 3], sc[(q - 10) & 3]);
                    if(q == 9)
                    {
                        if(pos == chain_at) // (every product of the chain before has been added)
                        {
#pragma unroll
                            for(int c = 0; c < 64; ++c)
                                FP8BS_ADD_AND_CLEAR(sum[c >> 4][(c >> 2) & 3][c & 3], acc[c >> 4][(c >> 2) & 3][c & 3]);
                            chain_at = chain_start(++chain, n);
                        }
#pragma unroll
                        for(int j = 0; j < 4; ++j)
                            sc[j] = xsv[j] * wsg;
                        scu = wsu;
                    }
                    // what the next K block starts with is worked out here, between the slots, and not between the barrier and its
                    // first reads, where nothing would be left to multiply
                    if(q == 13)
                    {
                        advance();
                        asm volatile("" : "+s"(fetch), "+s"(wnext), "+s"(xnext));
                        if(((pos + 1) & 63) == 0)
                        {
                            const float* const row = ws_row(tile);
                            const int kb = chain_kblock(min(pos + 1 + lane, n - 1), n);
                            ws_vec[0] = row[kb];
                            ws_vec[1] = row[ws_up + kb];
                            asm volatile("" : "+v"(ws_vec[0]), "+v"(ws_vec[1])); // waited for here, and not in every K block
                        }
                        wsg = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ws_vec[0]), (pos + 1) & 63));
                        wsu = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(ws_vec[1]), (pos + 1) & 63));
                        asm volatile("" : "+s"(wsg), "+s"(wsu));
                    }
                    if(q == 14)
                    {
                        stage = stage == kGateUpStages - 1 ? 0 : stage + 1;
                        const uint32_t on = stage == 0 ? -(kGateUpStages - 1) * kGateUpStage : kGateUpStage;
                        w_at += on;
                        x_lo += on;
                        x_hi += on;
                        xs_at = xs_lds + (scales ^ (((uint32_t)pos + 1) >> 2 & 1u) * kGateUpWindow) + (((uint32_t)pos + 1) & 3u) * 4u;
                        asm volatile("" : "+v"(w_at), "+v"(x_lo), "+v"(x_hi), "+v"(xs_at));
                    }
                }
                scg  = sc[2];
                scg3 = sc[3];
#pragma unroll
                for(int j = 0; j < 4; ++j)
                    scp[j] = xsv[j] * scu;
                // All but what was requested in this K block has landed, and (every fragment of this K block is in registers, or
                // on its way there: the barrier waits for outstanding LDS reads) behind the barrier the next one is in LDS.
                if(!xs)
                    asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
                asm volatile("s_waitcnt vmcnt(7)" ::: "memory");
                xs = opens();
                __syncthreads();
            }
            request();
            // the up tiles of the last K block, then the two products in flight
#pragma unroll
            for(int q = 0; q < 8; ++q)
            {
                FP8BS_MFMA(P[q & 3], aw[2 + q % 2], bx[q / 2]);
                if(q < 2)
                    FP8BS_FMA4(acc[1][2 + q], P[2 + q], (q == 0 ? scg : scg3));
                else
                    FP8BS_FMA4(acc[2 + q % 2][(q - 2) / 2], P[(q - 2) & 3], scp[(q - 2) / 2]);
            }
            asm volatile("s_nop 15\n s_nop 15\n s_nop 15" ::: "memory"); // >= 11 wait states after the last MFMA
            FP8BS_FMA4(acc[2][3], P[2], scp[3]);
            FP8BS_FMA4(acc[3][3], P[3], scp[3]);
#pragma unroll
            for(int c = 0; c < 64; ++c)
                sum[c >> 4][(c >> 2) & 3][c & 3] += acc[c >> 4][(c >> 2) & 3][c & 3];

            // the product lands in the stage of the last K block; the next item's first two are on their way to the others
            const lds_byte_ptr h_at = smem3 + h_stage() + (uint32_t)(wm * 64 + l16) * kHPitch + (uint32_t)(wn * 32 + kg * 4) * 2u;
#pragma unroll
            for(int i = 0; i < 2; ++i)
#pragma unroll
                for(int j = 0; j < 4; ++j)
                {
                    float h[4];
#pragma unroll
                    for(int r = 0; r < 4; ++r)
                        h[r] = prefill_activate<ACT>(sum[i][j][r]) * sum[2 + i][j][r];
                    *(lds_u2_ptr)(h_at + (uint32_t)j * 16u * kHPitch + i * 32u) =
                        u32x2{pack2<In16::bf16>(h[0], h[1]), pack2<In16::bf16>(h[2], h[3])};
                }
        }
        __syncthreads();
        // (ahead of the stores, which would be waited for as well: what was requested, and the next item's first K blocks)
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(id[0]), "+v"(id[1]), "+v"(id[2]), "+v"(ws_new[0]), "+v"(ws_new[1]), "+v"(tile3.block), "+v"(tile3.info)::"memory");
        // eight lanes per row, 16 columns each
#pragma unroll
        for(int u = 0; u < kTileRows * 8 / kGateUpThreads; ++u)
        {
            const int row = (u * kGateUpThreads + t) >> 3, part = t & 7;
            if(row >= rows) // (uniform over a row's eight lanes)
                continue;
            const lds_byte_ptr at_row = smem3 + h_stage() + (uint32_t)row * kHPitch + (uint32_t)part * 32u;
            const u32x4 lo = *(lds_u4_ptr)at_row;
            const u32x4 hi = *(lds_u4_ptr)(at_row + 16u);
            float       v[16], scale;
            unpack8<In16::bf16>(lo, v);
            unpack8<In16::bf16>(hi, v + 8);
            u32x4 codes;
            quant16<In16::bf16, 8>(lo, hi, v, codes, scale);
            const size_t slot = (size_t)tile.block * 32 + row;
            *(u32x4*)(p.hq + slot * p.inter + tile.grp * 128 + part * 16) = codes;
            if(part == 0)
                p.hs[slot * p.hs_stride + tile.grp] = scale;
        }
        rows_of(after, id[0], id[1], id[2]);
        after.w   = weights_of(tile2);
        tile      = tile1;
        tile1     = tile2;
        tile2     = uniform(tile3);
        ws_vec[0] = ws_new[0];
        ws_vec[1] = ws_new[1];
        scales ^= ((uint32_t)(n + 3) >> 2 & 1u) * kGateUpWindow;
    }
}
#undef FP8BS_MFMA
#undef FP8BS_FMA4
#undef FP8BS_ADD_AND_CLEAR

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
        src.ws_row = p.wsc + ((size_t)expert * (p.N / 128) + (n0 + wn * 64) / 128) * p.kblocks;

        float acc[T::kFrags][4][4], ws_vec = ring_ws_window(src.ws_row, p.kblocks, 0, lane);
        zero_acc(acc);
        ring_multiply<T, true, true>(smem3, src, wave, lane, 0, p.kblocks, wm * 64 < rows, ws_vec, acc);

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
    return tiles_win(pairs, all, a.experts, a.inter, a.dim);
}

size_t moe_prefill_workspace_bytes(const MoeArgs& a, bool rows_in_f32)
{
    const size_t slots = (size_t)a.max_padded;
    size_t       b     = align_up(slots * a.inter) + align_up(slots * row_floats(a.inter / 128) * 4) + align_up(slots * a.dim * (rows_in_f32 ? 4 : 2)) +
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
    hipLaunchKernelGGL(gate_up, dim3(256), dim3(kGateUpThreads), kGateUpLds, stream, g);

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
        const int64_t pairs = (int64_t)a.M * a.topk;
        const int64_t all   = routed_experts(pairs, a.topk, a.block_rows << a.expert_shift, a.max_padded, a.experts);
        d.col_splits        = down_col_splits((double)pairs / (double)all, a.experts, a.dim / 64, kDownWaves);
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
