// Chained complex triangular solves of up to kCTrsMaxRhs right-hand sides (ctrs.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace ops
{
constexpr int kCTrsMaxRhs = 2048;
// B <- op(A)^{-1} B, trans 0 / 1 / 2 = N / T / C, from packed LU factors with the interchanges
// ipiv (1-based, may be null; entries above their own row or out of range are none). info (may be
// null) receives kInfoWaitTimeout if a bounded wait gave up and is left alone otherwise.
size_t CTrsWorkspaceBytes(int n, int nrhs);
hipError_t CTrsSolve(int trans, int n, int nrhs, const float2* lu, int lda, const int* ipiv, float2* B, int ldb,
                     int* info, void* work, hipStream_t stream);
}  // namespace ops
