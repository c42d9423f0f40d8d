// Batched complex inverses of orders 33..64, gfx950: in-place Gauss-Jordan with implicit pivoting
// (the derivation is in batched.hip, the small orders in complex.hip), eight columns at a time.
#include <climits>

#include "complex_math.h"
#include "internal.h"
#include "lanes.h"
#include "wave.h"

namespace ops
{
namespace
{
typedef float f32x16 __attribute__((ext_vector_type(16)));

// One wave per matrix. The 64 columns lie as a ring in MFMA accumulator layout (cur, then nxt;
// real and imaginary tiles apart); the first eight are taken out one row per lane and go through
// their eight steps; the other 56 receive them as one rank-8 update of four real products (the
// pivot rows first brought to the state they have at their own step, by substitution); then the
// ring turns by eight. Against a row of 64 columns per lane, updated and read from LDS step by
// step: an eighth of the vector multiplications and no row through LDS per step.
// Bound by the chain of a step (score, FP64 reciprocal, eight columns), two waves a SIMD:
// 4096 matrices of order 64 432 us a call before, 225 us now (the host's pointer checks included).
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void cmatinv_rows_kernel(
    int n, const float2* const* __restrict__ Aarr, const float2* __restrict__ Abase, int64_t lda, int64_t strideA,
    float2* const* __restrict__ Carr, float2* __restrict__ Cbase, int64_t ldc, int64_t strideC, int* __restrict__ info)
{
    constexpr int US = 72;
    __shared__ __align__(16) float s_ur[8][US], s_ui[8][US];
    __shared__ __align__(16) float2 s_l[8][8];
    __shared__ int s_inv[64];
    const int lane = threadIdx.x, mat = blockIdx.x;
    const float2* const A = Aarr ? Aarr[mat] : Abase + mat * strideA;
    float2* const C = Carr ? Carr[mat] : Cbase + mat * strideC;
    const bool valid = lane < n;
    f32x16 curR[2], curI[2], nxtR[2], nxtI[2];
    {
        // Columns beyond n repeat the last one: no step pivots on them and none is stored.
        const float2* src = A + (valid ? lane : 0);
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            float2 x[32];
#pragma unroll
            for (int c = 0; c < 32; ++c)
            {
                x[c] = *src;
                src += 32 * h + c + 1 < n ? lda : 0;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    float2 lo = x[8 * k + r], hi = x[8 * k + 4 + r];
                    if (!valid) lo = hi = make_float2(0.0f, 0.0f);
                    SwapHalves(lo.x, hi.x);
                    SwapHalves(lo.y, hi.y);
                    (h == 0 ? curR : nxtR)[0][4 * k + r] = lo.x;
                    (h == 0 ? curI : nxtI)[0][4 * k + r] = lo.y;
                    (h == 0 ? curR : nxtR)[1][4 * k + r] = hi.x;
                    (h == 0 ? curI : nxtI)[1][4 * k + r] = hi.y;
                }
        }
    }
    int pos = valid ? lane : -1;
    int zeroCol = 0;
    double2 sigma = make_double2(1.0, 0.0);
    int steps = 0;  // ring turns, in columns
    for (; steps < n; steps += 8)
    {
        float2 v[8], lm[8];
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            v[r] = make_float2(curR[0][r], curI[0][r]);
            v[4 + r] = make_float2(curR[1][r], curI[1][r]);
            SwapHalves(v[r].x, v[4 + r].x);
            SwapHalves(v[r].y, v[4 + r].y);
        }
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
        {
            lm[jj] = make_float2(0.0f, 0.0f);
            const int k = steps + jj;
            if (k >= n) continue;  // uniform
            // Score class: 0 for rows already used, else PivotScore + 1.
            const bool cand = pos >= k;
            unsigned bh = __float_as_uint(fabsf(v[jj].x) + fabsf(v[jj].y)) + 2u;
            if (__builtin_expect(__any(cand && bh > 0x7f800001u), 0)) bh = PivotScore(v[jj]) + 1u;
            bh = cand ? bh : 0u;
            const unsigned top = WaveMaxU32(bh);
            unsigned long long tie = __ballot(bh == top);
            if (__builtin_expect(__popcll(tie) != 1, 0))  // uniform
            {
                const unsigned low = WaveMaxU32(bh == top ? ~static_cast<unsigned>(pos) : 0u);
                tie = __ballot(bh == top && ~static_cast<unsigned>(pos) == low);
            }
            const int wl = __builtin_ctzll(tie);
            const int pp = __builtin_amdgcn_readlane(pos, wl);
            const bool isP = lane == wl;
            pos = isP ? k : (pos == k ? pp : pos);
            float2 u[8];
#pragma unroll
            for (int c = 0; c < 8; ++c) u[c] = make_float2(ReadLane(v[c].x, wl), ReadLane(v[c].y, wl));
            const bool z = u[jj].x == 0.0f && u[jj].y == 0.0f;  // uniform
            if (z && zeroCol == 0) zeroCol = k + 1;
            const double2 r = Recip64(z ? make_float2(1.0f, 0.0f) : u[jj]);
            const float2 q = Mul64(v[jj], r);
            const float2 l = isP || z ? make_float2(0.0f, 0.0f) : q;
            lm[jj] = l;
#pragma unroll
            for (int c = 0; c < 8; ++c)
                if (c != jj) v[c] = SubMul(v[c], l, u[c]);
            if (!z)
            {
                v[jj] = isP ? make_float2(1.0f, 0.0f) : make_float2(-l.x, -l.y);
                if (isP) sigma = r;
            }
        }
        // The pivot rows' other columns and their multipliers, by step.
        {
            const int rel = pos - steps;
            int slot0 = static_cast<unsigned>(rel) < 8u && pos < n ? rel : -1;
            if (slot0 >= 0)
#pragma unroll
                for (int c = 0; c < 8; c += 2)
                    *reinterpret_cast<float4*>(&s_l[slot0][c]) = make_float4(lm[c].x, lm[c].y, lm[c + 1].x, lm[c + 1].y);
            int slot1 = slot0;
            SwapHalves(slot0, slot1);
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                const int slot = t == 0 ? slot0 : slot1;
                if (slot >= 0)
                {
                    const int at = 4 * (lane >> 5);
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                    {
                        *reinterpret_cast<float4*>(&s_ur[slot][at + 8 * k]) =
                            make_float4(curR[t][4 * k], curR[t][4 * k + 1], curR[t][4 * k + 2], curR[t][4 * k + 3]);
                        *reinterpret_cast<float4*>(&s_ui[slot][at + 8 * k]) =
                            make_float4(curI[t][4 * k], curI[t][4 * k + 1], curI[t][4 * k + 2], curI[t][4 * k + 3]);
                        *reinterpret_cast<float4*>(&s_ur[slot][at + 32 + 8 * k]) =
                            make_float4(nxtR[t][4 * k], nxtR[t][4 * k + 1], nxtR[t][4 * k + 2], nxtR[t][4 * k + 3]);
                        *reinterpret_cast<float4*>(&s_ui[slot][at + 32 + 8 * k]) =
                            make_float4(nxtI[t][4 * k], nxtI[t][4 * k + 1], nxtI[t][4 * k + 2], nxtI[t][4 * k + 3]);
                    }
                }
            }
        }
        __syncthreads();
        // Lane: ring column lane. The block itself, and the steps that a last block lacks, take no
        // part.
        const int live = min(8, n - steps);
        float ur[8], ui[8];
#pragma unroll
        for (int s = 0; s < 8; ++s)
        {
            ur[s] = ui[s] = 0.0f;
            if (s < live)  // uniform
            {
                ur[s] = lane < 8 ? 0.0f : s_ur[s][lane];
                ui[s] = lane < 8 ? 0.0f : s_ui[s][lane];
#pragma unroll
                for (int e = 0; e < s; ++e)
                {
                    const float2 x = SubMul(make_float2(ur[s], ui[s]), s_l[s][e], make_float2(ur[e], ui[e]));
                    ur[s] = x.x;
                    ui[s] = x.y;
                }
            }
        }
        float br[2][4], bi[2][4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
        {
            SwapHalves(ur[2 * s], ur[2 * s + 1]);
            SwapHalves(ui[2 * s], ui[2 * s + 1]);
            br[0][s] = -lm[2 * s].x;
            br[1][s] = -lm[2 * s + 1].x;
            SwapHalves(br[0][s], br[1][s]);
            bi[0][s] = -lm[2 * s].y;
            bi[1][s] = -lm[2 * s + 1].y;
            SwapHalves(bi[0][s], bi[1][s]);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                curR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s], br[t][s], curR[t], 0, 0, 0);
                curI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ui[2 * s], br[t][s], curI[t], 0, 0, 0);
                nxtR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s + 1], br[t][s], nxtR[t], 0, 0, 0);
                nxtI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ui[2 * s + 1], br[t][s], nxtI[t], 0, 0, 0);
                curR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(-ui[2 * s], bi[t][s], curR[t], 0, 0, 0);
                curI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s], bi[t][s], curI[t], 0, 0, 0);
                nxtR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(-ui[2 * s + 1], bi[t][s], nxtR[t], 0, 0, 0);
                nxtI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s + 1], bi[t][s], nxtI[t], 0, 0, 0);
            }
        // The ring turns; the block goes to its end.
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            SwapHalves(v[r].x, v[4 + r].x);
            SwapHalves(v[r].y, v[4 + r].y);
        }
#pragma unroll
        for (int t = 0; t < 2; ++t)
        {
#pragma unroll
            for (int e = 0; e < 16; ++e)
            {
                curR[t][e] = e < 12 ? curR[t][(e + 4) & 15] : nxtR[t][e - 12];
                curI[t][e] = e < 12 ? curI[t][(e + 4) & 15] : nxtI[t][e - 12];
            }
#pragma unroll
            for (int e = 0; e < 16; ++e)
            {
                nxtR[t][e] = e < 12 ? nxtR[t][(e + 4) & 15] : v[4 * t + (e & 3)].x;
                nxtI[t][e] = e < 12 ? nxtI[t][(e + 4) & 15] : v[4 * t + (e & 3)].y;
            }
        }
        __syncthreads();  // the pivot rows in LDS are free again
    }
    if (valid) s_inv[pos] = lane;
    __syncthreads();
    // Ring column c holds matrix column (c + steps) mod 64; step j's column belongs to row s_inv[j].
    auto put = [&](int c, float2 x)
    {
        const int j = (c + steps) & 63;
        if (j < n && valid) C[static_cast<int64_t>(s_inv[j]) * ldc + pos] = Mul64(x, sigma);
    };
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int h = 0; h < 2; ++h)
            {
                const f32x16* const re = h == 0 ? curR : nxtR;
                const f32x16* const im = h == 0 ? curI : nxtI;
                float2 lo = make_float2(re[0][4 * k + r], im[0][4 * k + r]);
                float2 hi = make_float2(re[1][4 * k + r], im[1][4 * k + r]);
                SwapHalves(lo.x, hi.x);
                SwapHalves(lo.y, hi.y);
                put(32 * h + 8 * k + r, lo);
                put(32 * h + 8 * k + 4 + r, hi);
            }
    if (lane == 0) info[mat] = zeroCol;
}
}  // namespace

hipError_t CMatinvRows64(int n, const float2* const* Aarr, const float2* Abase, int lda, int64_t strideA,
                         float2* const* Carr, float2* Cbase, int ldc, int64_t strideC, int* info, int batch,
                         hipStream_t stream)
{
    if (n < 1 || n > 64) return hipErrorInvalidValue;
    hipLaunchKernelGGL(cmatinv_rows_kernel, dim3(batch), dim3(64), 0, stream, n, Aarr, Abase, static_cast<int64_t>(lda),
                       strideA, Carr, Cbase, static_cast<int64_t>(ldc), strideC, info);
    return hipGetLastError();
}
}  // namespace ops
