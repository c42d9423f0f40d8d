// How far the FP64 inverse of a 64 x 64 triangular block may be trusted in a solve (trs.hip, ctrs.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ops
{
namespace
{
// The factor of row i is (|E| |X| d)_i / d_i, d_i the largest entry of row i of E, for a block E and
// its inverse X: by so much may a solve with X exceed the backward error |E| |x| of a substitution, in
// units of X's own rounding. Entries |X_jk| d_k <= kSmallInverse bound it by 64^2 times that
// (|E_ij| <= d_i), so that it is computed for the odd block only.
constexpr double kInverseGrowth64 = 1 << 20;
constexpr double kSmallInverse = 1 << 8;
constexpr int kGrowthScratch = 10 * 64;  // doubles; d lies in the fifth 64
__device__ inline double* RowMaxima(double* s_g) { return s_g + 4 * 64; }

// By a workgroup of four waves. e: |E(lane, 16 wave + k)|, x(j): |X(lane, j)|; d in place. Returns the
// factor of row `lane`.
template <typename F>
__device__ inline double Growth64(const float (&e)[16], F x, double* s_g, int tid)
{
    const int lane = tid & 63, wave = tid >> 6;
    const double* const s_d = RowMaxima(s_g);
    double* const s_w = s_g + 5 * 64;
    double* const s_p = s_g + 6 * 64;
    double part = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) part = fma(x(16 * wave + k), s_d[16 * wave + k], part);
    s_p[tid] = part;
    __syncthreads();
    if (wave == 0) s_w[lane] = (s_p[lane] + s_p[64 + lane]) + (s_p[128 + lane] + s_p[192 + lane]);
    __syncthreads();
    part = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) part = fma(static_cast<double>(e[k]), s_w[16 * wave + k], part);
    s_g[tid] = part;
    __syncthreads();
    return ((s_g[lane] + s_g[64 + lane]) + (s_g[128 + lane] + s_g[192 + lane])) / s_d[lane];
}
}  // namespace
}  // namespace ops
