// split.hpp -- 32-bit values as pairs of halves for the f16 matrix cores.
//
// A value v scaled by a power of two into f16's range is held as hi + lo,
// hi = f16(v), lo = f16(v - hi), both rounded to nearest: off by at most 2^-23
// of |v| (2^-24.5 in the mean square; f32 itself holds v exactly), and by 2^-25
// where lo is subnormal.  pow2_scale puts the largest value of a row (or
// span) into [2^14, 2^15), so that floor is 2^-39 of it: a value less than
// 2^-16 of the largest has fewer bits.  A product of two such pairs as
// hi * hi + lo * hi + hi * lo leaves out lo * lo, at most 2^-22 of it.
// split8_part keeps lo 2^12 times larger for kernels that sum the lo halves
// apart: its floor is 2^-51.
#pragma once

#include "internal.hpp"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));
typedef float float2v __attribute__((ext_vector_type(2)));

// Eight f32 values as hi and lo halves (|v| < 65504).
__device__ __forceinline__ void split8(const float (&v)[8], half8 &hi, half8 &lo)
{
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const float2v p = {v[i], v[i + 1]};
        const half2v h = __builtin_convertvector(p, half2v);
        // v - hi, exact; as an fma it takes the half directly
        const float2v r = {__builtin_fmaf((float)h[0], -1.0f, v[i]), __builtin_fmaf((float)h[1], -1.0f, v[i + 1])};
        const half2v l = __builtin_convertvector(r, half2v);
        hi[i] = h[0];
        hi[i + 1] = h[1];
        lo[i] = l[0];
        lo[i + 1] = l[1];
    }
}

// The power of two that brings values below `bound` under 2^15, and its
// inverse (bound 0 or not finite: 1).  Exponents are clamped so that both
// stay normal.
__device__ __forceinline__ void pow2_scale(float bound, float &s, float &inv)
{
    int e = 15;
    if (bound > 0.0f && bound <= 3.402823466e38f) (void)frexpf(bound, &e); // bound < 2^e
    e = e < -100 ? -100 : e;
    s = ldexpf(1.0f, 15 - e);
    inv = ldexpf(1.0f, e - 15);
}

// One half of eight values x * s: hi (part 0) or 2^12 lo (part kLoApart), the
// same instructions for either, with s2 = s or s * kLoApart (a lane's part
// chosen by its constants: no lane forms both and drops one).
constexpr float kLoApart = 4096.0f;
__device__ __forceinline__ half8 split8_part(const float (&x)[8], float s, float s2, float part)
{
    half8 out;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        const float2v p = {x[i] * s, x[i + 1] * s};
        const half2v h = __builtin_convertvector(p, half2v);
        const float2v r = {__builtin_fmaf((float)h[0], -part, x[i] * s2),
                           __builtin_fmaf((float)h[1], -part, x[i + 1] * s2)};
        const half2v l = __builtin_convertvector(r, half2v);
        out[i] = l[0];
        out[i + 1] = l[1];
    }
    return out;
}

// Codes with a minimum: code * mul + add in f32 (one rounding), then split.
__device__ __forceinline__ void codes8(uint32_t q0, uint32_t q1, float mul, float add, half8 &hi, half8 &lo)
{
    float w[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = __builtin_fmaf(byte_f(i < 4 ? q0 : q1, i & 3), mul, add);
    split8(w, hi, lo);
}
// Biased codes: (code - BIAS) * m in pairs of halves.  The code minus its
// bias is a half exactly (0x64 over a byte is the half 1024 + byte); with
// m = mh + ml, hi = c * mh rounded, lo = (c * mh - hi), which an fma gives
// exactly, + c * ml.  2.5 instructions per weight against 7 through f32 (the
// decode is the longer half of a one-fragment tile's instructions).  The sum
// is c * m to 2^-22 of it, down to the floor above in m and in the sum (2^-25
// each); Q8_0's m is a half itself (ml = 0), so its weights are exact in blocks
// whose d is more than 2^-21 of the row's largest.
template <int BIAS>
__device__ __forceinline__ void biased8(uint32_t q0, uint32_t q1, float m, half8 &hi, half8 &lo)
{
    const _Float16 mh = (_Float16)m, ml = (_Float16)__builtin_fmaf((float)mh, -1.0f, m);
    const half2v mh2 = {mh, mh}, ml2 = {ml, ml}, bias = {(_Float16)(-1024.0f - BIAS), (_Float16)(-1024.0f - BIAS)};
    const uint32_t k = 0x64646464u, lo2 = 0x04010400u, hi2 = 0x04030402u;
    const uint32_t q[4] = {__builtin_amdgcn_perm(k, q0, lo2), __builtin_amdgcn_perm(k, q0, hi2),
                           __builtin_amdgcn_perm(k, q1, lo2), __builtin_amdgcn_perm(k, q1, hi2)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        half2v c;
        __builtin_memcpy(&c, &q[i], 4);
        c = c + bias;
        const half2v h = c * mh2;
        const half2v l = __builtin_elementwise_fma(c, ml2, __builtin_elementwise_fma(c, mh2, -h));
        hi[2 * i] = h[0];
        hi[2 * i + 1] = h[1];
        lo[2 * i] = l[0];
        lo[2 * i + 1] = l[1];
    }
}

// Eight codes minus BIAS as halves, exactly.
template <int BIAS> __device__ __forceinline__ void codes_minus(uint32_t q0, uint32_t q1, half8 &c8)
{
    const half2v bias = {(_Float16)(-1024.0f - BIAS), (_Float16)(-1024.0f - BIAS)};
    const uint32_t k = 0x64646464u, lo2 = 0x04010400u, hi2 = 0x04030402u;
    const uint32_t q[4] = {__builtin_amdgcn_perm(k, q0, lo2), __builtin_amdgcn_perm(k, q0, hi2),
                           __builtin_amdgcn_perm(k, q1, lo2), __builtin_amdgcn_perm(k, q1, hi2)};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        half2v c;
        __builtin_memcpy(&c, &q[i], 4);
        c = c + bias;
        c8[2 * i] = c[0];
        c8[2 * i + 1] = c[1];
    }
}

// One value as hi and lo operands that hold it in all eight places.
__device__ __forceinline__ void split_splat(float v, half8 &hi, half8 &lo)
{
    const _Float16 h = (_Float16)v, l = (_Float16)__builtin_fmaf((float)h, -1.0f, v);
    hi = half8{h, h, h, h, h, h, h, h};
    lo = half8{l, l, l, l, l, l, l, l};
}
