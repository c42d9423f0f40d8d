// Uneven batched LU solve, orders 65..256: one workgroup per matrix (vbrows.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ops
{
// waves (2, 3 or 4) per matrix, orders up to 64 waves; order: indices of the count matrices.
hipError_t VbRowsLaunch(int waves, int count, const int* order, const int* nArr, const long long* pivOff, int nrhs,
                        float* const* A, float* const* B, int* ipiv, int* info, hipStream_t stream);
}  // namespace ops
