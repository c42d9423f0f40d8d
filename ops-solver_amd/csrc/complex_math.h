// Complex64 arithmetic shared by the complex kernels: pivot score, fused multiply-subtract and
// FP64-reciprocal scaling.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>
#include <cstdint>

namespace ops
{
namespace
{
__device__ inline uint32_t PivotScore(float2 v)
{
    const float r = fabsf(v.x), i = fabsf(v.y);
    float s = r + i;
    if (!(s >= 0.0f)) return 0u;
    if (s == 0.0f) return 1u;
    if (s > FLT_MAX)
    {
        s = r * 0.5f + i * 0.5f;
        return __float_as_uint(s) + 0x00800001u;
    }
    return __float_as_uint(s) + 1u;
}

__device__ inline float2 SubMul(float2 x, float2 a, float2 b)
{
    return make_float2(fmaf(a.y, b.y, fmaf(-a.x, b.x, x.x)), fmaf(-a.y, b.x, fmaf(-a.x, b.y, x.y)));
}

// 1/d in FP64 (exact enough that a * (1/d) rounds within one ulp of a / d).
__device__ inline double2 Recip64(float2 d)
{
    const double dr = d.x, di = d.y;
    const double den = dr * dr + di * di;
    const double inv = 1.0 / den;
    return make_double2(dr * inv, -di * inv);
}

__device__ inline float2 Mul64(float2 a, double2 r)
{
    const double ar = a.x, ai = a.y;
    return make_float2(static_cast<float>(ar * r.x - ai * r.y), static_cast<float>(ar * r.y + ai * r.x));
}

__device__ inline float2 Conj(float2 v, bool c) { return c ? make_float2(v.x, -v.y) : v; }
}  // namespace
}  // namespace ops
