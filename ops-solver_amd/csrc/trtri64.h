// Inverse of a lower triangular 64 x 64 block in LDS by one workgroup of four waves: 16 x 16
// diagonal blocks by substitution (one lane per column), then two doublings
//   inv [P 0; Q R] = [P' 0; -R' Q P' R']
// by products on the FP32 matrix cores. Latency is all it costs: about 1.5 us where a
// substitution over the whole block takes 64 dependent steps.
#pragma once
#include <hip/hip_runtime.h>

namespace ops
{
namespace
{
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x4 __attribute__((ext_vector_type(4)));
constexpr int kInvStride = 68;  // row stride in LDS of the block and its inverse

// D (16 x 16 at d) = sign * A (16 x K at a) * B (K x 16 at b), row-major in LDS, one wave.
template <int K, typename T>
__device__ inline void Product16(const T* a, const T* b, T* d, T sign, int lane)
{
    const int i = lane & 15, k0 = lane >> 4;
    if constexpr (sizeof(T) == 4)
    {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < K; k += 4)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i * kInvStride + k + k0], b[(k + k0) * kInvStride + i], acc, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) d[(4 * k0 + r) * kInvStride + i] = sign * acc[r];
    }
    else
    {
        f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < K; k += 4)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i * kInvStride + k + k0], b[(k + k0) * kInvStride + i], acc, 0, 0, 0);
        // The FP64 result has row 4 r + lane / 16 in element r.
#pragma unroll
        for (int r = 0; r < 4; ++r) d[(4 * r + k0) * kInvStride + i] = sign * acc[r];
    }
}

// s_l: the block, row-major, its strictly upper part zero (UNIT: its diagonal is not read);
// s_i (64 rows): receives the inverse, its upper part must be zero on entry; s_t: 32 rows of
// scratch. The caller synchronizes before; the result is visible after the last barrier here.
template <bool UNIT, typename T>
__device__ inline void InvertLower64(const T* s_l, T* s_i, T* s_t, int tid)
{
    const int lane = tid & 63, wave = tid >> 6;
    if (wave == 0)
    {
        // Lane: column lane % 16 of diagonal block lane / 16.
        const int b = lane & 48;
        T x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            T v = i == (lane & 15) ? T(1) : T(0);
            const T* const row = s_l + (b + i) * kInvStride + b;
#pragma unroll
            for (int k = 0; k < i; ++k) v = fma(-row[k], x[k], v);
            x[i] = UNIT ? v : v / row[i];
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) s_i[(b + i) * kInvStride + lane] = x[i];
    }
    __syncthreads();
    if (wave < 2)
        Product16<16>(s_l + (32 * wave + 16) * kInvStride + 32 * wave, s_i + 32 * wave * kInvStride + 32 * wave,
                      s_t + 16 * wave * kInvStride, T(1), lane);
    __syncthreads();
    if (wave < 2)
        Product16<16>(s_i + (32 * wave + 16) * kInvStride + 32 * wave + 16, s_t + 16 * wave * kInvStride,
                      s_i + (32 * wave + 16) * kInvStride + 32 * wave, T(-1), lane);
    __syncthreads();
    const int qr = 16 * (wave >> 1), qc = 16 * (wave & 1);
    Product16<32>(s_l + (32 + qr) * kInvStride, s_i + qc, s_t + qr * kInvStride + qc, T(1), lane);
    __syncthreads();
    Product16<32>(s_i + (32 + qr) * kInvStride + 32, s_t + qc, s_i + (32 + qr) * kInvStride + qc, T(-1), lane);
    __syncthreads();
}
}  // namespace
}  // namespace ops
