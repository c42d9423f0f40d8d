// Chained triangular solves of any number of right-hand sides (trs.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace ops
{
// B <- op(A)^{-1} B from packed LU factors (n x n, column-major), with the interchanges ipiv
// (1-based; may be null): three launches (preparation, two chained substitutions). info (may be
// null): set to 0, or to kInfoWaitTimeout if a bounded wait gave up. work: TrsWorkspaceBytes.
size_t TrsWorkspaceBytes(int n, int nrhs);
hipError_t TrsSolve(int trans, int n, int nrhs, const float* lu, int lda, const int* ipiv, float* B, int ldb, int* info,
                    void* work, hipStream_t stream);
}  // namespace ops
