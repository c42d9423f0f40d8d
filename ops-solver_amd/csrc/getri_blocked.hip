// Batched inverse from LU factors (getri_batched, orders 65..512): C = U^{-1} L^{-1} P, gfx950.
// Reference src/sgetri/real_lu_blocked_inverse_kernel.cpp:1115-1301 computes the same inverse
// blockwise per matrix; here every matrix of the batch moves through two launches together.
//   1. per matrix: the inverses of the 64 x 64 diagonal blocks of L and U (trtri64.h), the
//      permutation and the first zero pivot, one workgroup each;
//   2. per 32-column strip of C: the strip of P, then both block substitutions, in LDS.
// The two substitutions used to be a launch each over C in memory, behind a launch that wrote P
// (a serial interchange loop) and substitutions over whole blocks for the inverses.
#include <algorithm>
#include <climits>

#include "lu_kernels.h"
#include "permute.h"
#include "trtri64.h"

namespace ops
{
namespace
{
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kMaxOrder = 512;

// inv: per matrix nblk blocks of L, then nblk of U, column-major, identity beyond the matrix.
__global__ __launch_bounds__(256) void getri_prep_kernel(int n, const float* const* __restrict__ Aarr, int lda,
                                                         const int* __restrict__ piv, float* __restrict__ inv,
                                                         int* __restrict__ perm, int* __restrict__ info)
{
    __shared__ __align__(16) float s_l[64 * kInvStride], s_i[64 * kInvStride], s_t[32 * kInvStride];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int nblk = (n + 63) / 64, role = blockIdx.x, b = blockIdx.y;
    const float* const A = Aarr[b];
    if (role == 2 * nblk)
    {
        int* const s_piv = reinterpret_cast<int*>(s_l);
        int* const s_first = reinterpret_cast<int*>(s_t);
        if (tid == 0) *s_first = INT_MAX;
        bool plain = true;
        for (int k = tid; k < n; k += 256)
        {
            int v = piv != nullptr ? piv[static_cast<size_t>(b) * n + k] - 1 : k;
            if (v < 0 || v >= n) v = k;
            plain = plain && v >= k;
            s_piv[k] = v;
        }
        plain = __syncthreads_and(plain);
        for (int i = tid; i < kMaxOrder && i - lane < n; i += 256)
        {
            const int x = TracePosition(s_piv, n, i, i - lane, plain);
            if (i < n) perm[static_cast<size_t>(b) * n + i] = x;
        }
        for (int k = tid; k < n; k += 256)
            if (A[static_cast<size_t>(k) * lda + k] == 0.0f) atomicMin(s_first, k);
        __syncthreads();
        if (tid == 0) info[b] = *s_first == INT_MAX ? 0 : *s_first + 1;
        return;
    }
    const bool upper = role >= nblk;
    const int k0 = (upper ? role - nblk : role) * 64, kb = min(64, n - k0);
    const float* const T = A + static_cast<size_t>(k0) * lda + k0;
    // Lower: the block; upper: its transpose, whose inverse is transposed back.
#pragma unroll
    for (int k = 0; k < 16; ++k)
    {
        const int c = wave * 16 + k;
        const float v = lane < kb && c < kb ? T[static_cast<size_t>(c) * lda + lane] : (lane == c ? 1.0f : 0.0f);
        if (upper)
            s_l[c * kInvStride + lane] = lane <= c ? v : 0.0f;
        else
            s_l[lane * kInvStride + c] = lane > c ? v : 0.0f;
        s_i[lane * kInvStride + c] = 0.0f;
    }
    __syncthreads();
    if (upper)
        InvertLower64<false>(s_l, s_i, s_t, tid);
    else
        InvertLower64<true>(s_l, s_i, s_t, tid);
    float* const out = inv + (static_cast<size_t>(b) * 2 * nblk + role) * 4096;
#pragma unroll
    for (int k = 0; k < 16; ++k)
    {
        const int c = wave * 16 + k;
        out[c * 64 + lane] = upper ? s_i[c * kInvStride + lane] : s_i[lane * kInvStride + c];
    }
}

// One substitution over the strip in LDS (Xs: Kp rows of stride 33): per 64-row block, in
// ascending (lower) or descending (upper) order, X_b = inv(T_bb) B_b, then the unsolved rows
// -= T(rows, b) X_b, both on FP32 MFMA, the products formed transposed so that each
// accumulator lane holds one row.
template <bool UPPER>
__device__ inline void Substitute(int K, const float* __restrict__ T, int ldt, const float* __restrict__ Inv, float* Xs,
                                  int tid)
{
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), li = lane & 31, lk = lane >> 5, ui = lane & 15, uk = lane >> 4;
    const int nblk = (K + 63) / 64;
    float lf[32];
    // Operand fragments are loaded for a whole 32-row tile before its 32 products, the first tile
    // of a block before the block's own product.
    auto loadTile = [&](int k0, int k1, int r0)
    {
        // Rows and columns beyond the matrix repeat its last ones (their products are not used or
        // meet zero rows of X): no load is predicated.
        const float* const Lc = T + static_cast<size_t>(k0) * ldt + min(r0 + li, K - 1);
        const int last = k1 - k0 - 1;
#pragma unroll
        for (int t = 0; t < 32; ++t) lf[t] = Lc[static_cast<uint64_t>(min(2 * t + lk, last)) * static_cast<unsigned>(ldt)];
    };
    for (int q = 0; q < nblk; ++q)
    {
        const int b = UPPER ? nblk - 1 - q : q;
        const int k0 = b * 64, k1 = min(K, k0 + 64);
        const int rLo = UPPER ? 0 : k1, rHi = UPPER ? k0 : K;  // rows still to update
        // Wave: rows 16 wave .. + 15 of the block, both 16-column halves of the strip.
        float lb[16];
        const float* Lb = Inv + static_cast<size_t>(b) * 4096 + 16 * wave + ui;
#pragma unroll
        for (int t = 0; t < 16; ++t) lb[t] = Lb[(4 * t + uk) * 64];
        int r0 = rLo + wave * 32;
        if (r0 < rHi) loadTile(k0, k1, r0);
        f32x4 x[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
        for (int t = 0; t < 16; ++t)
        {
            if (UPPER ? t < 4 * wave : t >= 4 * (wave + 1)) continue;  // uniform: zeros of the triangle
#pragma unroll
            for (int h = 0; h < 2; ++h)
                x[h] = __builtin_amdgcn_mfma_f32_16x16x4f32(Xs[(k0 + 4 * t + uk) * 33 + 16 * h + ui], lb[t], x[h], 0, 0, 0);
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int r = 0; r < 4; ++r) Xs[(k0 + 16 * wave + ui) * 33 + 16 * h + 4 * uk + r] = x[h][r];
        __syncthreads();
        for (; r0 < rHi; r0 += 128)
        {
            f32x16 acc;
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll
            for (int t = 0; t < 32; ++t)
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(Xs[(k0 + 2 * t + lk) * 33 + li], lf[t], acc, 0, 0, 0);
            const int row = r0 + li;
            if (r0 + 128 < rHi) loadTile(k0, k1, r0 + 128);
            if (row < rHi)
#pragma unroll
                for (int v = 0; v < 16; ++v) Xs[row * 33 + (v & 3) + 8 * (v >> 2) + 4 * lk] -= acc[v];
        }
        __syncthreads();
    }
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4))) void getri_solve_kernel(int n, const float* const* __restrict__ Aarr, int lda,
                                                          const float* __restrict__ inv, const int* __restrict__ perm,
                                                          float* const* __restrict__ Carr, int ldc)
{
    extern __shared__ float Xs[];  // rows padded to whole blocks, stride 33
    const int tid = threadIdx.x, b = blockIdx.y;
    const int c0 = blockIdx.x * 32, nblk = (n + 63) / 64, Kp = nblk * 64;
    const int* const p = perm + static_cast<size_t>(b) * n;
    for (int r = tid >> 5; r < Kp; r += 8)
        Xs[r * 33 + (tid & 31)] = r < n && p[r] == c0 + (tid & 31) ? 1.0f : 0.0f;
    __syncthreads();
    const float* const Inv = inv + static_cast<size_t>(b) * 2 * nblk * 4096;
    Substitute<false>(n, Aarr[b], lda, Inv, Xs, tid);
    Substitute<true>(n, Aarr[b], lda, Inv + static_cast<size_t>(nblk) * 4096, Xs, tid);
    float* const C = Carr[b];
    const int lane = tid & 63, cols = min(32, n - c0);
    for (int c = tid >> 6; c < cols; c += 4)
        for (int r = lane; r < n; r += 64) C[static_cast<size_t>(c0 + c) * ldc + r] = Xs[r * 33 + c];
}
}  // namespace

size_t GetriBlockedBatchedWorkspaceBytes(int n, int batch)
{
    const size_t per = (static_cast<size_t>(2) * ((n + 63) / 64) * 4096 + n) * sizeof(float);
    return per * static_cast<size_t>(std::max(batch, 0));
}

hipError_t GetriBlockedBatched(int n, const float* const* Aarr, int lda, const int* piv, float* const* Carr, int ldc,
                               int* info, int batch, float* work, hipStream_t stream)
{
    if (n <= 0 || batch <= 0) return hipSuccess;
    if (n > kMaxOrder || batch > 65535) return hipErrorInvalidValue;
    const int nblk = (n + 63) / 64;
    int* perm = reinterpret_cast<int*>(work + static_cast<size_t>(batch) * 2 * nblk * 4096);
    hipLaunchKernelGGL(getri_prep_kernel, dim3(2 * nblk + 1, batch), dim3(256), 0, stream, n, Aarr, lda, piv, work, perm,
                       info);
    hipLaunchKernelGGL(getri_solve_kernel, dim3((n + 31) / 32, batch), dim3(256),
                       static_cast<size_t>(nblk) * 64 * 33 * sizeof(float), stream, n, Aarr, lda, work, perm, Carr, ldc);
    return hipGetLastError();
}
}  // namespace ops
