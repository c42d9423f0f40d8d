// Interchange sequence -> permutation, one lane per position (trs.hip, getri_blocked.hip).
#pragma once
#include <hip/hip_runtime.h>

namespace ops
{
namespace
{
// The source row of row i of P B: position i traced backward through the interchanges
// k <-> s_piv[k] (0-based, 16-byte aligned LDS array of n entries), k = n - 1 .. 0.
// plain: no entry points above its own row (LAPACK's pivots never do), so position i is first
// met by interchange i, and from there on only "x == pivot" can move it: half the steps on
// average and two instructions each. base: first position of the wave, a multiple of 64.
__device__ inline int TracePosition(const int* s_piv, int n, int i, int base, bool plain)
{
    int x = i;
    if (plain)
    {
        if (i < n) x = s_piv[i];
        for (int k = min(n, base + 64) - 1; k >= base && k >= 0; --k) x = k < i && s_piv[k] == x ? k : x;
#pragma unroll 1
        for (int k = base - 1; k >= 3; k -= 4)
        {
            const int4 v = *reinterpret_cast<const int4*>(s_piv + k - 3);  // k + 1 is a multiple of 64
            x = v.w == x ? k : x;
            x = v.z == x ? k - 1 : x;
            x = v.y == x ? k - 2 : x;
            x = v.x == x ? k - 3 : x;
        }
    }
    else
        for (int k = n - 1; k >= 0; --k)
        {
            const int v = s_piv[k];
            x = x == k ? v : (x == v ? k : x);
        }
    return x;
}
}  // namespace
}  // namespace ops
