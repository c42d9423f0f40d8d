// Chained triangular solves of any number of right-hand sides (trs.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace ops
{
// B <- op(A)^{-1} B from packed LU factors (n x n, column-major), with the interchanges ipiv
// (1-based; may be null): three launches (preparation, two chained substitutions). src == null:
// the right-hand sides are the identity (nrhs == n) and B only receives the result. info (may
// be null): set to 0, or to kInfoWaitTimeout if a bounded wait gave up. work: TrsWorkspaceBytes;
// pub (may be null): TrsPublicationBytes of memory used in place of that part of work.
size_t TrsPublicationBytes(int n, int nrhs);
size_t TrsWorkspaceBytes(int n, int nrhs, bool withPublication);
hipError_t TrsSolve(int trans, int n, int nrhs, const float* lu, int lda, const int* ipiv, const float* src, int lds,
                    float* B, int ldb, int* info, void* work, void* pub, hipStream_t stream);
}  // namespace ops
