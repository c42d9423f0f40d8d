// Moves between a row per lane and MFMA accumulator layout (leaf.hip, cleaf.hip, cmatinv.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ops
{
namespace
{
// The upper 32 lanes of x and the lower 32 lanes of y change places.
__device__ inline void SwapHalves(float& x, float& y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    x = __uint_as_float(r[0]);
    y = __uint_as_float(r[1]);
}
__device__ inline void SwapHalves(int& x, int& y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(x), static_cast<unsigned>(y), false, false);
    x = static_cast<int>(r[0]);
    y = static_cast<int>(r[1]);
}

__device__ inline float ReadLane(float v, int lane)
{
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), lane));
}
}  // namespace
}  // namespace ops
