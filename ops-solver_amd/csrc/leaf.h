// Partial-pivoting panel leaves of the real LU (leaf.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace ops
{
// One leaf: columns [c0, c0 + wact) of rows [c0, m), inside the outer panel [j0, panelEnd).
struct LeafArgs
{
    float* A;
    int lda, m, j0, c0, wact, panelEnd;
    int pivoting;                // 0: the diagonal is the pivot
    int newPanel;                // c0 == j0: rowsrc starts as the identity
    int* ipiv;                   // may be null
    int* info;
    int* rowsrc;                 // panel row sources (positions -> source rows)
    int* moves;                  // out: the leaf's moved rows, 2 * kLeafMaxWidth (dst, src) pairs, dst < 0: none
    unsigned long long* slots;   // exchange words of the multi-workgroup leaves (kLeafSlotWords)
    unsigned tagBase;            // multi-workgroup leaves: tags tagBase .. tagBase + width - 1 are this leaf's
    int* err;                    // raised by a bounded wait that gave up
    unsigned spinLimit;
};

constexpr int kLeafMaxWidth = 64;    // columns of the widest leaf
constexpr int kLeafMaxGroups = 64;   // workgroups of one multi-workgroup leaf
constexpr int kLeafKeyWords = 2 * 9 * kLeafMaxGroups;
constexpr int kLeafRowStride = kLeafMaxWidth + 8;
constexpr int kLeafArrivalWord = kLeafKeyWords + 2 * 8 * kLeafRowStride;
constexpr int kLeafSlotWords = kLeafArrivalWord + kLeafMaxGroups;
constexpr int kLeafMoveInts = 4 * kLeafMaxWidth;

// Largest m - c0 a leaf of one workgroup takes, and its width there.
constexpr int kLeafSingleRows = 1024;
constexpr int kLeafMultiRows = 16384;

// The leaf leaves its rows where they started; LeafSwap, launched after it, applies its
// interchanges to every panel column [j0, panelEnd).
// One workgroup (m - c0 <= kLeafSingleRows, wact <= kLeafMaxWidth):
hipError_t LeafSingle(const LeafArgs& a, hipStream_t stream);
// Up to 64 workgroups (m - c0 <= kLeafMultiRows, wact <= kLeafMaxWidth):
hipError_t LeafMulti(const LeafArgs& a, bool cooperative, bool spread, hipStream_t stream);
hipError_t LeafSwap(const LeafArgs& a, hipStream_t stream);
// The same and, with it, the solve form (unitlower.h; 4096 floats, column-major) of the leaf's
// unit-lower diagonal block, padded with the identity; the top 64 rows of the panel columns right
// of the leaf go to ub (64 floats a column, 16-byte aligned) instead of A.
hipError_t LeafFinish(const LeafArgs& a, float* form, float* ub, hipStream_t stream);
// After LeafFinish of a 64-column leaf: U = inv(L11) ub into A's top rows and the update of the
// rows below, for the panel columns right of the leaf.
hipError_t PanelUpdate(const LeafArgs& a, const float* form, const float* ub, hipStream_t stream);
}  // namespace ops
