// Solves with a unit-lower 64 x 64 block on the FP32 matrix cores (leaf.hip, gemm.hip). The block
// is prepared once as its solve form: the inverses of its four 16 x 16 diagonal blocks (without
// their ones) and, below them, -L; the solve substitutes from block to block, every sum of
// products formed from zero and added once (added up term by term onto B, whose entries are
// larger, it would round more). An inverse over all 64 columns would take as
// many products, but its error grows with |L| |inv(L)|: with multipliers of one sign and
// magnitude c like (1 + c)^63, where 16 columns give (1 + c)^15 and a substitution none (c = 0.3:
// |B - L U| / (|L| |U|) of 8e-2, 2e-7 and 1e-7). Blocks whose small inverses grow beyond
// kInverseGrowth (multipliers above 1, which a factorization without pivoting has, or all of one
// sign) and columns that are not finite are substituted outright: those solves are backward
// stable, and no infinity reaches the rows above its own.
// 128: 528 diagonal blocks each of Gaussian, uniform and small-integer matrices with partial
// pivoting have 46, 61 and 68 at most.
#pragma once
#include <hip/hip_runtime.h>

#include <cfloat>

#include "lanes.h"
#include "trtri64.h"

namespace ops
{
namespace
{
constexpr float kInverseGrowth = 128.0f;
// Element of the solve form (above the diagonal, otherwise zero) that is 1 where the block is to be
// substituted.
constexpr int kSubstituteFlag = 63 * 64;

// The solve form of a block by one workgroup of four waves. s_l: the block row-major in LDS, its
// strictly lower triangle with zeros elsewhere; the caller synchronizes before.
__device__ inline void SolveForm64(const float* s_l, float* __restrict__ form, int tid)
{
    const int lane = tid & 63, wave = tid >> 6;
    // Column 16 wave + k, row lane: below its diagonal block -L, above zero.
    if ((lane >> 4) != wave)
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            const int c = 16 * wave + k;
            if (c != 63 || lane != 0) form[c * 64 + lane] = (lane >> 4) > wave ? -s_l[lane * kInvStride + c] : 0.0f;
        }
    if (wave != 0) return;
    // Lane: column lane % 16 of diagonal block lane / 16, and its share of |L| |inv(L)|.
    const int b = lane & 48;
    float x[16], grow[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 16; ++i)
    {
        float v = i == (lane & 15) ? 1.0f : 0.0f;
        const float* const row = s_l + (b + i) * kInvStride + b;
#pragma unroll
        for (int k = 0; k < i; ++k)
        {
            v = fmaf(-row[k], x[k], v);
            grow[k & 3] = fmaf(fabsf(row[k]), fabsf(x[k]), grow[k & 3]);
        }
        x[i] = v;
        grow[3] += fabsf(v);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = i > (lane & 15) ? x[i] : 0.0f;
#pragma unroll
    for (int i = 0; i < 16; i += 4)
        *reinterpret_cast<float4*>(form + lane * 64 + b + i) = make_float4(x[i], x[i + 1], x[i + 2], x[i + 3]);
    const bool fine = (grow[0] + grow[1]) + (grow[2] + grow[3]) <= kInverseGrowth;
    const bool all = __all(fine);
    if (lane == 0) form[kSubstituteFlag] = all ? 0.0f : 1.0f;
}

// The solve form's operands of one lane: element (16 d + ui, 16 t + 4 uk + s) of block (d, t), d >= t,
// in the order of use.
struct SolveOperands
{
    float a[40];
    float substitute;
};
__device__ inline void LoadOperands(const float* __restrict__ form, int ui, int uk, SolveOperands& o)
{
#pragma unroll
    for (int t = 0, x = 0; t < 4; ++t)
#pragma unroll
        for (int d = t; d < 4; ++d)
#pragma unroll
            for (int s = 0; s < 4; ++s, ++x) o.a[x] = form[(16 * t + 4 * uk + s) * 64 + 16 * d + ui];
    o.substitute = form[kSubstituteFlag];
}

// U = inv(L) B for 16 columns by one wave: lane (ui, uk) holds rows 16 t + 4 uk + r of column ui in
// b[t][r], before and after. The product's result layout is the next one's operand layout if
// step s takes row 4 uk + s, so nothing moves between lanes. Returns whether every lane's block may
// be taken; if not, b holds nothing of use and the caller substitutes (SubstituteColumns).
__device__ inline bool SolveColumns(const SolveOperands& o, f32x4 (&b)[4])
{
    bool fine = o.substitute == 0.0f;
    f32x4 acc[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0, x = 0; t < 4; ++t)
    {
        if (t > 0) b[t] = b[t] + acc[t];
        f32x4 u = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s, ++x) u = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[x], b[t][s], u, 0, 0, 0);
        b[t] = b[t] + u;
#pragma unroll
        for (int d = t + 1; d < 4; ++d)
#pragma unroll
            for (int s = 0; s < 4; ++s, ++x) acc[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.a[x], b[t][s], acc[d], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) fine = fine && fabsf(b[t][r]) <= FLT_MAX;
    }
    return __all(fine);
}

// The same by substitution for 16 columns of one wave, lane: row. T: the block in memory, rows and
// columns from `size` on are the identity. Rarely taken; eight columns of T in flight together.
__device__ inline void SubstituteColumns(const float* __restrict__ T, int64_t ldt, int size, int lane, float (&v)[16])
{
#pragma unroll 1
    for (int k0 = 0; k0 < size; k0 += 8)
    {
        float l[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) l[e] = lane > k0 + e && lane < size ? T[(k0 + e) * ldt + lane] : 0.0f;
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int c = 0; c < 16; ++c)
            {
                const float x = ReadLane(v[c], k0 + e);
                v[c] = lane > k0 + e && lane < size ? fmaf(-l[e], x, v[c]) : v[c];
            }
    }
}
}  // namespace
}  // namespace ops
