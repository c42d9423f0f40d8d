// Panel leaves and panel launches of the complex LU (cleaf.hip); the real ones are in leaf.h.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace ops
{
// One leaf: columns [c0, c0 + wact) of rows [c0, m), inside the outer panel [j0, panelEnd).
struct CLeafArgs
{
    float2* A;
    int lda, m, j0, c0, wact, panelEnd;
    int pivoting;               // 0: the diagonal is the pivot
    int newPanel;               // c0 == j0: rowsrc starts as the identity
    int* ipiv;                  // may be null
    int* info;
    int* rowsrc;                // panel row sources (positions -> source rows)
    int* moves;                 // out: the leaf's moved rows, 128 (dst, src) pairs, dst < 0: none
    unsigned long long* slots;  // exchange words of the multi-workgroup leaves (kCLeafSlotWords)
    unsigned tagBase;           // tags tagBase .. tagBase + 63 are this leaf's
    int* err;                   // raised by a bounded wait that gave up
    unsigned spinLimit;
};
constexpr int kCLeafWidth = 64;
constexpr int kCLeafMaxGroups = 32;
constexpr int kCLeafSingleRows = 512;  // rows of the tallest one-workgroup leaf
constexpr int kCLeafMaxRows = 16384;
// Keys (2 parities x 32), candidates (x 16 words), pivot rows (2 x 8 x 144 words), arrivals.
constexpr int kCLeafValueWord = 2 * kCLeafMaxGroups;
constexpr int kCLeafRowWord = kCLeafValueWord + 2 * 16 * kCLeafMaxGroups;
constexpr int kCLeafRowStride = 2 * kCLeafWidth + 16;
constexpr int kCLeafArrivalWord = kCLeafRowWord + 2 * 8 * kCLeafRowStride;
constexpr int kCLeafSlotWords = kCLeafArrivalWord + kCLeafMaxGroups;
constexpr size_t kCFormBlock = 2 * 64 * 64;  // floats per diagonal block: real part, then imaginary part

hipError_t CLeafColumns(const CLeafArgs& a, bool spread, hipStream_t stream);
// The leaf's interchanges on the whole panel; the solve form of its unit-lower diagonal
// block to form (kCFormBlock floats: unitlower.h's, real parts, then imaginary parts); the top 64 rows of the
// panel columns right of it to ub (64 complex a column) instead of A.
hipError_t CLeafFinish(const CLeafArgs& a, float* form, float2* ub, hipStream_t stream);
// After CLeafFinish of a 64-column leaf: U = inv(L11) ub into A's top rows, and the update of the
// rows below, for the panel columns right of the leaf.
hipError_t CPanelUpdate(const CLeafArgs& a, const float* form, const float2* ub, hipStream_t stream);
// B <- L^{-1} B for the unit-lower K x K block T (K <= 512) and N columns, from the solve forms
// of T's 64 x 64 diagonal blocks.
hipError_t CTrsmLowerUnit(int K, int N, const float2* T, int ldt, const float* forms, float2* B, int ldb,
                          hipStream_t stream);
}  // namespace ops
