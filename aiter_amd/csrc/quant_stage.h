// The 1 x G quant stage shared by the kernels that end in fp8 codes: 16-bit conversions, reductions over the lanes of
// a group, and the two encoders.
#pragma once

#include "fp8bs_launch.h"
#include "fp8bs_math.h"

namespace fp8bs {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------- 16-bit <-> fp32

template <In16 DT>
__device__ __forceinline__ void unpack8(const u32x4& c, float* v)
{
#pragma unroll
    for(int i = 0; i < 4; ++i)
    {
        if constexpr(DT == In16::bf16)
        {
            v[2 * i]     = __uint_as_float(c[i] << 16);
            v[2 * i + 1] = __uint_as_float(c[i] & 0xffff0000u);
        }
        else
        {
            const uint32_t w = c[i]; // copy first: bit_cast straight from a vector element misreads
            f16x2 h      = __builtin_bit_cast(f16x2, w);
            v[2 * i]     = (float)h.x;
            v[2 * i + 1] = (float)h.y;
        }
    }
}

// round to nearest even to the 16-bit type; returns the raw code
template <In16 DT>
__device__ __forceinline__ uint32_t round16(float f)
{
    if constexpr(DT == In16::bf16)
    {
        __bf16 b = (__bf16)f;
        return (uint32_t)__builtin_bit_cast(unsigned short, b);
    }
    else
    {
        _Float16 h = (_Float16)f;
        return (uint32_t)__builtin_bit_cast(unsigned short, h);
    }
}

template <In16 DT>
__device__ __forceinline__ float widen16(uint32_t code)
{
    if constexpr(DT == In16::bf16)
        return __uint_as_float(code << 16);
    else
        return (float)__builtin_bit_cast(_Float16, (unsigned short)code);
}

// two floats rounded to nearest even to the 16-bit type, a in the low half
template <In16 DT>
__device__ __forceinline__ uint32_t round16_pk(float a, float b)
{
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    if constexpr(DT == In16::bf16)
    {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
    }
    else
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, f16x2));
}

// Largest magnitude among 16 packed 16-bit floats, as its 15-bit pattern: for both 16-bit types the
// order of the patterns is the order of the magnitudes, with inf above every finite value and the
// NaNs above inf -- so a group that holds a NaN or an inf shows in its maximum, and nothing has to
// be tested element by element.
__device__ __forceinline__ uint32_t absmax_pk16(const u32x4& lo, const u32x4& hi)
{
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
    auto           mx = [](uint32_t a, uint32_t b) {
        return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
    };
    const uint32_t k = 0x7fff7fffu;
    const uint32_t a = mx(mx(mx(lo[0] & k, lo[1] & k), mx(lo[2] & k, lo[3] & k)),
                          mx(mx(hi[0] & k, hi[1] & k), mx(hi[2] & k, hi[3] & k)));
    return max(a & 0xffffu, a >> 16);
}

// ---------------------------------------------------------------- DPP reductions over a group

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_u32(uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}

constexpr int kDppXor1       = 0xB1;  // quad_perm [1,0,3,2]
constexpr int kDppXor2       = 0x4E;  // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141; // lane i <- lane 7-i inside each 8 lanes
constexpr int kDppRowMirror  = 0x140; // lane i <- lane 15-i inside each 16 lanes

// all-reduce max over LPG (1,2,4,8,16) adjacent lanes; every lane ends with the group's value
template <int LPG>
__device__ __forceinline__ float group_max_f32(float v)
{
    if constexpr(LPG >= 2)
        v = fmaxf(v, __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(v))));
    if constexpr(LPG >= 4)
        v = fmaxf(v, __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(v))));
    if constexpr(LPG >= 8)
        v = fmaxf(v, __uint_as_float(dpp_u32<kDppHalfMirror>(__float_as_uint(v))));
    if constexpr(LPG >= 16)
        v = fmaxf(v, __uint_as_float(dpp_u32<kDppRowMirror>(__float_as_uint(v))));
    return v;
}

template <int LPG>
__device__ __forceinline__ uint32_t group_max_u32(uint32_t v)
{
    if constexpr(LPG >= 2)
        v = max(v, dpp_u32<kDppXor1>(v));
    if constexpr(LPG >= 4)
        v = max(v, dpp_u32<kDppXor2>(v));
    if constexpr(LPG >= 8)
        v = max(v, dpp_u32<kDppHalfMirror>(v));
    if constexpr(LPG >= 16)
        v = max(v, dpp_u32<kDppRowMirror>(v));
    return v;
}

// sum of a double over the 64 lanes of a wave, same value in every lane.  DPP permutes inside
// each row of 16 lanes (no LDS traffic, unlike ds_bpermute-based shuffles), then the four row
// sums are read with v_readlane and added in a fixed order.
__device__ __forceinline__ double dpp_add_f64(double v, int which)
{
    uint32_t lo = (uint32_t)__double2loint(v), hi = (uint32_t)__double2hiint(v);
    uint32_t plo, phi;
    switch(which)
    {
    case 0: plo = dpp_u32<kDppXor1>(lo); phi = dpp_u32<kDppXor1>(hi); break;
    case 1: plo = dpp_u32<kDppXor2>(lo); phi = dpp_u32<kDppXor2>(hi); break;
    case 2: plo = dpp_u32<kDppHalfMirror>(lo); phi = dpp_u32<kDppHalfMirror>(hi); break;
    default: plo = dpp_u32<kDppRowMirror>(lo); phi = dpp_u32<kDppRowMirror>(hi); break;
    }
    return v + __hiloint2double((int)phi, (int)plo);
}

__device__ __forceinline__ double wave_sum_f64(double v)
{
    v = dpp_add_f64(v, 0);
    v = dpp_add_f64(v, 1);
    v = dpp_add_f64(v, 2);
    v = dpp_add_f64(v, 3); // every lane now holds the sum of its row of 16
    const uint32_t lo = (uint32_t)__double2loint(v), hi = (uint32_t)__double2hiint(v);
    double         r[4];
#pragma unroll
    for(int k = 0; k < 4; ++k)
        r[k] = __hiloint2double((int)__builtin_amdgcn_readlane(hi, 16 * k),
                                (int)__builtin_amdgcn_readlane(lo, 16 * k));
    return (r[0] + r[1]) + (r[2] + r[3]);
}

// ---------------------------------------------------------------- the quant stage
// v[16]: this lane's 16 consecutive elements of its group (already widened to fp32).
// codes: their 16 e4m3fn codes in memory order.  scale: the group's scale (same in all lanes).

// Rare path: group holds NaN/inf, is all zero, or its amax is so small or large that the
// scale or its reciprocal leaves the normal range.  Everything is done with IEEE divisions and
// the software conversion.  NaN/inf follow what the host division does in the torch reference:
// a NaN element keeps its own sign, other elements of a NaN group get the (positive) NaN of
// the scale; inf/inf is the default NaN, which has the sign bit set on x86.
// Inlined on purpose: an out-of-line call would give the kernel a private (scratch) segment,
// and waves that need scratch are dispatched far more slowly than the HBM stream can be fed.
__device__ __forceinline__ uint32_t absmax_bits16(const float (&v)[16])
{
    uint32_t mm = 0;
#pragma unroll
    for(int i = 0; i < 16; ++i)
        mm = max(mm, __float_as_uint(v[i]) & 0x7fffffffu);
    return mm; // as integers: NaN > inf > every finite magnitude
}

// mm: the group's largest |x| as an integer (absmax_bits16 reduced over the group)
__device__ __forceinline__ void encode16_slow(const float (&v)[16], uint32_t mm, u32x4& codes, float& scale)
{
    float s;
    if(mm > 0x7f800000u)
        s = __uint_as_float(mm | 0x00400000u);
    else
    {
        s = __uint_as_float(mm) / 448.0f;
        if(s == 0.0f)
            s = 1.0f;
    }
    uint32_t out[4] = {0, 0, 0, 0};
#pragma unroll
    for(int i = 0; i < 16; ++i)
    {
        uint32_t xb = __float_as_uint(v[i]);
        uint32_t xa = xb & 0x7fffffffu;
        uint32_t sg = (xb >> 24) & 0x80u;
        uint32_t c;
        if(mm > 0x7f800000u)
            c = (xa > 0x7f800000u) ? (sg | 0x7fu) : 0x7fu;
        else if(mm == 0x7f800000u)
            c = (xa == 0x7f800000u) ? 0xffu : sg;
        else
            c = f32_to_e4m3fn_sw(v[i] / s);
        out[i >> 2] |= c << (8 * (i & 3));
    }
    codes = u32x4{out[0], out[1], out[2], out[3]};
    scale = s;
}

// m: the group's amax, for which amax_allows_fast_path holds
__device__ __forceinline__ void encode16_fast(const float (&v)[16], float m, u32x4& codes, float& scale)
{
    const float s = amax_over_448(m); // = m / 448 as IEEE division gives it
    const float r = recip_in_range(s); // the correctly rounded reciprocal: s lies within 2^-89 .. 2^92 here
    uint32_t    out[4];
#pragma unroll
    for(int j = 0; j < 4; ++j)
    {
        int w = 0;
        w = __builtin_amdgcn_cvt_pk_fp8_f32(div_by_scale(v[4 * j], s, r), div_by_scale(v[4 * j + 1], s, r), w,
                                            false);
        w = __builtin_amdgcn_cvt_pk_fp8_f32(div_by_scale(v[4 * j + 2], s, r), div_by_scale(v[4 * j + 3], s, r),
                                            w, true);
        out[j] = (uint32_t)w;
    }
    codes = u32x4{out[0], out[1], out[2], out[3]};
    scale = s;
}

// lo, hi: the 16 values as packed 16-bit floats in memory order; v: the same values widened
template <In16 DT, int LPG>
__device__ __forceinline__ void quant16(const u32x4& lo, const u32x4& hi, const float (&v)[16], u32x4& codes,
                                        float& scale)
{
    const float m = widen16<DT>(group_max_u32<LPG>(absmax_pk16(lo, hi)));
    if(amax_allows_fast_path(__float_as_uint(m))) // false for inf and NaN, too
        encode16_fast(v, m, codes, scale);
    else
        encode16_slow(v, group_max_u32<LPG>(absmax_bits16(v)), codes, scale);
}

} // namespace fp8bs
