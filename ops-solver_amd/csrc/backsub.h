// Back substitution of one small system from its stored U by one wave (vbatched.hip, vbrows.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ops
{
namespace
{
__device__ inline float Rl(float v, int lane)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Back substitution over the columns k of position segment S (64 S <= k < 64 S + 64, k < n),
// last to first, then the segments below. Lane l holds y at positions l + 64 i; column k of
// U (rows 0 .. 64 S + 63, slots 0..S) is read from the stored LU with a prefetch of D columns
// in registers. x_k = y_k * (1 / U_kk): the reciprocal depends only on U, so it stays off
// the dependent chain that runs through the y values.
template <int S, int RPL, int Q>
__device__ __attribute__((always_inline)) inline void BackSubSeg(const float* __restrict__ A, int n, int lane,
                                                                 float (&y)[Q][RPL])
{
    constexpr int D = 8;
    const int kLo = 64 * S;
    const int kHi = min(n, 64 * S + 64) - 1;
    float u[D][S + 1];
#pragma unroll
    for (int t = 0; t < D; ++t)
    {
        const int k = kHi - t;
#pragma unroll
        for (int i = 0; i <= S; ++i)
            u[t][i] = (k >= kLo && lane + 64 * i < n) ? A[static_cast<size_t>(k) * n + lane + 64 * i] : 0.0f;
    }
    for (int k0 = kHi; k0 >= kLo; k0 -= D)
    {
#pragma unroll
        for (int t = 0; t < D; ++t)
        {
            const int k = k0 - t;
            if (k >= kLo)
            {
                const int kl = k - kLo;
                const float r = 1.0f / Rl(u[t][S], kl);
#pragma unroll
                for (int q = 0; q < Q; ++q)
                {
                    const float x = Rl(y[q][S], kl) * r;
#pragma unroll
                    for (int i = 0; i < S; ++i) y[q][i] = fmaf(-u[t][i], x, y[q][i]);
                    y[q][S] = lane < kl ? fmaf(-u[t][S], x, y[q][S]) : (lane == kl ? x : y[q][S]);
                }
            }
            const int kn = k - D;
#pragma unroll
            for (int i = 0; i <= S; ++i)
                u[t][i] = (kn >= kLo && lane + 64 * i < n) ? A[static_cast<size_t>(kn) * n + lane + 64 * i] : 0.0f;
        }
    }
    if constexpr (S > 0) BackSubSeg<S - 1, RPL, Q>(A, n, lane, y);
}
}  // namespace
}  // namespace ops
