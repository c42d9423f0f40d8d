// Uneven batched LU solve (getrf + getrs per matrix), orders 65..256: leaf.hip's blocked columns
// over whole small matrices. Semantics of the pivots as in vbatched.hip.
//
// A workgroup of 2, 3 or 4 waves per matrix, one row per lane throughout (implicit pivoting: the
// position each row occupies is tracked). The augmented matrix [A | B] passes in panels of 64
// columns held in MFMA accumulator layout. A panel first receives the finished blocks of eight
// columns one after the other (multipliers from memory, this lane's own; the pivot rows' entries
// through LDS; one rank-8 update on the matrix cores each), then goes through its own blocks as a
// leaf does. The right-hand sides are the last columns, so the elimination substitutes them
// forward. Finished columns go to memory by original row; a pass at the end moves every row to
// its final position, and a wave per right-hand side substitutes back.
//
// Bound by the chain of a column (search, one exchange between the waves, seven updates) at four
// waves a SIMD: 128 registers a lane, so that four matrices of order 256 (five of 192, eight of
// 128) share a compute unit, where the column-cyclic kernels of vbatched.hip hold one or two of
// those and spend a column's chain on each in turn. 20000 systems of orders 1..256: 8.2 ms
// before, 4.8 ms with these kernels (2.6 ms the 193..256, 1.4 the 129..192, 0.5 the 65..128).
#include "vbrows.h"

#include <climits>

#include "backsub.h"
#include "internal.h"
#include "lanes.h"
#include "wave.h"

namespace ops
{
namespace
{
typedef float f32x16 __attribute__((ext_vector_type(16)));
constexpr int kMaxRhs = 4;

__device__ inline unsigned CyclicMax4(unsigned v)
{
    auto mx = [](unsigned a, unsigned b) { return a > b ? a : b; };
    v = mx(v, DppU32<0xB1>(v));
    return mx(v, DppU32<0x4E>(v));
}

template <int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(4))) void vb_rows_kernel(
    const int* __restrict__ order, const int* __restrict__ nArr, const long long* __restrict__ pivOff, int nrhs,
    float* const* __restrict__ Aarr, float* const* __restrict__ Barr, int* __restrict__ ipiv, int* __restrict__ info)
{
    constexpr int W = 64, US = W + 28;
    __shared__ uint2 s_key[2][4];
    __shared__ __align__(16) float s_val[2][4 * 8];
    __shared__ __align__(16) float s_u[2][8][US];
    __shared__ __align__(16) float s_l[2][8][8];
    __shared__ float s_y[kMaxRhs][64 * NW];
    __shared__ int s_pos[64 * NW];
    __shared__ unsigned s_zero[32];  // per block: its columns without a pivot

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int mi = order[blockIdx.x];
    const int n = nArr[mi];
    float* const A = Aarr[mi];
    float* const B = Barr[mi];
    int* const piv = ipiv + pivOff[mi];
    const int nt = n + nrhs;
    const int lr = wid * 64 + lane;
    const bool valid = lr < n;
    const int row = valid ? lr : 0;
    if (tid < 8) s_key[tid >> 2][tid & 3] = make_uint2(0u, 0u);  // of waves that are not there
    __syncthreads();
    int pos = valid ? lr : -1;
    int zeroCol = 0, buf = 0;
    f32x16 cur[2], nxt[2];

    for (int p0 = 0; p0 < nt; p0 += W)
    {
        const int wact = min(W, nt - p0);
        {
            float x[W];
#pragma unroll
            for (int c = 0; c < W; ++c)
            {
                const int j = min(p0 + c, nt - 1);  // columns beyond the last repeat it
                x[c] = (j < n ? A + j * n : B + (j - n) * n)[row];
            }
#pragma unroll
            for (int k = 0; k < 8; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    float lo = valid ? x[8 * k + r] : 0.0f, hi = valid ? x[8 * k + 4 + r] : 0.0f;
                    SwapHalves(lo, hi);
                    (k < 4 ? cur : nxt)[0][4 * (k % 4) + r] = lo;
                    (k < 4 ? cur : nxt)[1][4 * (k % 4) + r] = hi;
                }
        }
        // The block's pivot rows (columns of cur from `live` on, and of nxt) and multipliers to LDS,
        // its U by substitution, one panel column per lane, and the rank-8 update.
        auto publish = [&](int rel, const float (&lm)[8], int live, bool right)
        {
            int slot0 = static_cast<unsigned>(rel) < 8u ? rel : -1;
            if (slot0 >= 0)
            {
                float4* const d4 = reinterpret_cast<float4*>(&s_l[buf][slot0][0]);
                d4[0] = make_float4(lm[0], lm[1], lm[2], lm[3]);
                d4[1] = make_float4(lm[4], lm[5], lm[6], lm[7]);
            }
            int slot1 = slot0;
            SwapHalves(slot0, slot1);
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                const int slot = t == 0 ? slot0 : slot1;
                if (slot >= 0)
                {
                    float* const at = &s_u[buf][slot][4 * (lane >> 5)];
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        if (k < 3 || live == 0)
                            *reinterpret_cast<float4*>(at + live + 8 * k) =
                                make_float4(cur[t][4 * k], cur[t][4 * k + 1], cur[t][4 * k + 2], cur[t][4 * k + 3]);
                    if (right)  // uniform
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            *reinterpret_cast<float4*>(at + 32 + 8 * k) =
                                make_float4(nxt[t][4 * k], nxt[t][4 * k + 1], nxt[t][4 * k + 2], nxt[t][4 * k + 3]);
                }
            }
        };
        // cnt: columns of the block that had a pivot row (a last block may lack some).
        auto update = [&](const float (&lm)[8], int live, int cnt, bool left, bool right)
        {
            float u[8];
            const int col = (lane < 32 ? live : 32) + (lane & 31);
#pragma unroll
            for (int s = 0; s < 8; ++s) u[s] = s < cnt ? s_u[buf][s][col] : 0.0f;
#pragma unroll
            for (int i = 1; i < 8; ++i)
                if (i < cnt)  // uniform
#pragma unroll
                    for (int s = 0; s < i; ++s) u[i] = fmaf(-s_l[buf][i][s], u[s], u[i]);
            float bop[2][4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
            {
                SwapHalves(u[2 * s], u[2 * s + 1]);
                bop[0][s] = -lm[2 * s];
                bop[1][s] = -lm[2 * s + 1];
                SwapHalves(bop[0][s], bop[1][s]);
            }
            if (left)  // uniform
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        cur[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(u[2 * s], bop[t][s], cur[t], 0, 0, 0);
            if (right)  // uniform
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        nxt[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(u[2 * s + 1], bop[t][s], nxt[t], 0, 0, 0);
            buf ^= 1;
        };

        // The finished blocks. A row's multipliers are entries that this lane stored itself.
        const int done = min(p0, n);
        float ahead[8];
        auto fetch = [&](int b0)
        {
#pragma unroll
            for (int c = 0; c < 8; ++c) ahead[c] = A[min(b0 + c, n - 1) * n + row];
        };
        if (done > 0) fetch(0);
        for (int b0 = 0; b0 < done; b0 += 8)
        {
            const unsigned noPivot = s_zero[b0 >> 3];
            float lm[8];
#pragma unroll
            for (int c = 0; c < 8; ++c)
                lm[c] = pos > b0 + c && b0 + c < n && !((noPivot >> c) & 1u) ? ahead[c] : 0.0f;
            if (b0 + 8 < done) fetch(b0 + 8);
            publish(pos - b0, lm, 0, wact > 32);
            __syncthreads();
            update(lm, 0, min(8, n - b0), true, wact > 32);
        }

        // The panel's own blocks.
        for (int q = 0; 8 * q < wact; ++q)
        {
            const int b0 = p0 + 8 * q;
            float v[8], lm[8];
            unsigned noPivot = 0u;
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                v[r] = cur[0][r];
                v[4 + r] = cur[1][r];
                SwapHalves(v[r], v[4 + r]);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 12; ++e) cur[t][e] = cur[t][e + 4];
#pragma unroll
            for (int jj = 0; jj < 8; ++jj)
            {
                lm[jj] = 0.0f;
                const int j = b0 + jj;
                if (j >= n) continue;  // uniform: a right-hand side
                const int par = jj & 1;
                // Magnitude class and position of the lane's candidate, as in leaf.hip.
                const unsigned ab = __float_as_uint(v[jj]) & 0x7fffffffu;
                const unsigned mag = ab <= 0x7f800000u ? ab + 0x80000001u : (pos == j ? 0xffffffffu : 0x80000000u);
                const unsigned bh = pos >= j ? mag : 0u;
                float br = 1.0f / v[jj];
                unsigned top = WaveMaxU32(bh);
                unsigned long long tie = __ballot(bh == top);
                asm volatile("" : "+v"(br));  // beside the search, where its latency is hidden
                if (__builtin_expect(__popcll(tie) != 1, 0))  // uniform
                {
                    const unsigned low = WaveMaxU32(bh == top ? ~static_cast<unsigned>(pos) : 0u);
                    tie = __ballot(bh == top && ~static_cast<unsigned>(pos) == low);
                }
                int wl = __builtin_ctzll(tie);
                if (lane == wl)
                {
                    s_key[par][wid] = make_uint2(top, (static_cast<unsigned>(pos) & 0x7fffffffu) |
                                                          (__float_as_uint(v[jj]) & 0x80000000u));
                    s_val[par][wid * 8] = br;
#pragma unroll
                    for (int c = jj + 1; c < 8; ++c) s_val[par][wid * 8 + c] = v[c];
                }
                __syncthreads();
                const uint2 k = s_key[par][lane & 3];
                const float x0 = s_val[par][lane & 31];
                const unsigned t = CyclicMax4(k.x);
                top = __builtin_amdgcn_readfirstlane(t);
                unsigned hit = static_cast<unsigned>(__ballot(k.x == top)) & 15u;
                if (__builtin_expect(__popc(hit) != 1, 0))  // uniform
                {
                    const unsigned low = CyclicMax4(k.x == top ? 0x7fffffffu - (k.y & 0x7fffffffu) : 0u);
                    hit = static_cast<unsigned>(__ballot(k.x == top && 0x7fffffffu - (k.y & 0x7fffffffu) == low)) & 15u;
                }
                wl = __builtin_ctz(hit | 0x80000000u) & 3;
                const unsigned ky = __builtin_amdgcn_readlane(k.y, wl);
                const int bpos = static_cast<int>(ky & 0x7fffffffu);
                const float rec = ReadLane(x0, wl * 8);
                float u[8];
#pragma unroll
                for (int c = jj + 1; c < 8; ++c) u[c] = ReadLane(x0, wl * 8 + c);
                const unsigned dmag = (top & 0x7fffffffu) - 1u;  // |d| (a NaN class gives a NaN)
                pos = pos == bpos ? j : (pos == j ? bpos : pos);
                if (tid == 0) piv[j] = bpos + 1;
                const bool zero = dmag == 0u;  // uniform
                if (zero && zeroCol == 0) zeroCol = j + 1;
                noPivot |= zero ? 1u << jj : 0u;
                float qv = v[jj] * rec;
                if (__builtin_expect(dmag - 0x00800000u > 0x7f000000u, 0))  // uniform: subnormal, zero or NaN
                    qv = v[jj] / __uint_as_float(dmag | (ky & 0x80000000u));
                const bool below = pos > (zero ? INT_MAX : j);
                const float l = below ? qv : 0.0f;
                lm[jj] = l;
                v[jj] = below ? qv : v[jj];
#pragma unroll
                for (int c = jj + 1; c < 8; ++c) v[c] = fmaf(-l, u[c], v[c]);
            }
#pragma unroll
            for (int c = 0; c < 8; ++c)
            {
                const int j = b0 + c;
                if (j < n)  // uniform
                {
                    if (valid) A[j * n + lr] = v[c];
                }
                else if (j < nt && valid)
                    s_y[j - n][pos] = v[c];
            }
            if (tid == 0) s_zero[(b0 >> 3) & 31] = noPivot;
            const int live = 8 * (q + 1);
            if (live >= wact) break;  // uniform
            publish(pos - b0, lm, live, q < 4);
            __syncthreads();
            update(lm, live, min(8, n - b0), (q & 3) != 3, q < 4);
            if ((q & 3) == 3)  // uniform
            {
                cur[0] = nxt[0];
                cur[1] = nxt[1];
            }
        }
        __syncthreads();  // s_zero
    }

    if (valid) s_pos[lr] = pos;
    if (tid == 0) info[mi] = zeroCol;
    __syncthreads();
    // Columns from original to final row order, one wave a column.
    int to[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) to[i] = lane + 64 * i < n ? s_pos[lane + 64 * i] : -1;
    for (int j = wid; j < n; j += NW)
    {
        float* const col = A + j * n;
        float v[NW];
#pragma unroll
        for (int i = 0; i < NW; ++i) v[i] = to[i] >= 0 ? col[lane + 64 * i] : 0.0f;
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): every lane's loads are done
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
#pragma unroll
        for (int i = 0; i < NW; ++i)
            if (to[i] >= 0) col[to[i]] = v[i];
    }
    __syncthreads();
    constexpr int Q = (kMaxRhs + NW - 1) / NW;
    const int c0 = wid * Q;
    if (c0 >= nrhs) return;
    float y[Q][NW];
#pragma unroll
    for (int c = 0; c < Q; ++c)
#pragma unroll
        for (int i = 0; i < NW; ++i)
            y[c][i] = c0 + c < nrhs && lane + 64 * i < n ? s_y[c0 + c][lane + 64 * i] : 0.0f;
    BackSubSeg<NW - 1, NW, Q>(A, n, lane, y);
#pragma unroll
    for (int c = 0; c < Q; ++c)
#pragma unroll
        for (int i = 0; i < NW; ++i)
            if (c0 + c < nrhs && lane + 64 * i < n) B[(c0 + c) * n + lane + 64 * i] = y[c][i];
}
}  // namespace

hipError_t VbRowsLaunch(int waves, int count, const int* order, const int* nArr, const long long* pivOff, int nrhs,
                        float* const* A, float* const* B, int* ipiv, int* info, hipStream_t stream)
{
    if (count <= 0) return hipSuccess;
    if (nrhs < 0 || nrhs > kMaxRhs) return hipErrorInvalidValue;
    if (waves == 2)
        hipLaunchKernelGGL(vb_rows_kernel<2>, dim3(count), dim3(128), 0, stream, order, nArr, pivOff, nrhs, A, B, ipiv,
                           info);
    else if (waves == 3)
        hipLaunchKernelGGL(vb_rows_kernel<3>, dim3(count), dim3(192), 0, stream, order, nArr, pivOff, nrhs, A, B, ipiv,
                           info);
    else if (waves == 4)
        hipLaunchKernelGGL(vb_rows_kernel<4>, dim3(count), dim3(256), 0, stream, order, nArr, pivOff, nrhs, A, B, ipiv,
                           info);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}
}  // namespace ops
