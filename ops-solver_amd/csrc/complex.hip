// Complex64 LU family on gfx950: cgetrf, device cgetrs (trans N/T/C), batched direct
// inverse (cmatinv) and batched inverse from factors (cgetri_batched).
//
// Reference semantics (src/cgetrf/cgetrf_kernel.cpp:376-411, ComplexSolverGetrf):
//   * pivot = row with the largest L1 score |re|+|im| under the unsigned key of
//     src/utils/complex_solver_kernel.hpp:47-63 (NaN inactive, both zeros equal, an
//     overflow-safe half sum), lowest row on ties;
//   * multipliers are accurate quotients (the reference's Divide is specified to 4 ulp,
//     test/complex_solver/complex_solver_test.cpp:520-556): here a * (1/d) evaluated in
//     FP64 and rounded once;
//   * rank-1 updates use the fused order of SubMul (complex_solver_kernel.hpp:65-68);
//   * the trailing update is built from real MFMA products, C -= A B as
//     Re += Ar Br + (-Ai) Bi, Im += Ar Bi + Ai Br (the 4-product form of
//     src/utils/complex_solver_cube.cpp:206-214), FP32 v_mfma_f32_32x32x2_f32, FP32 accumulation.
// The blocked structure mirrors the real path: register-resident leaves with position
// tracking, in-panel interchange + TRSM + update, then outer interchanges, U12 solve and
// the MFMA trailing update.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>

#include "cleaf.h"
#include "complex_math.h"
#include "ctrs.h"
#include "internal.h"

namespace ops
{
namespace
{
typedef float f32x16 __attribute__((ext_vector_type(16)));

__global__ void cclear_slots_kernel(unsigned long long* slots, int words, int* err)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < words) slots[i] = 0ull;
    if (i == 0) *err = 0;
}

// The list of rows moved by a panel; empty after a wait that ran out (getrf.hip).
__global__ __launch_bounds__(1024) void ccompact_moves_kernel(int m, int j0, const int* __restrict__ rowsrc,
                                                              const int* __restrict__ err, int* __restrict__ moved)
{
    __shared__ int s_count;
    if (threadIdx.x == 0) s_count = 0;
    __syncthreads();
    const int hi = *err == 0 ? m : j0;
    for (int r = j0 + threadIdx.x; r < hi; r += blockDim.x)
    {
        const int s = rowsrc[r];
        if (s != r)
        {
            const int slot = atomicAdd(&s_count, 1);
            moved[1 + 2 * slot] = r;
            moved[2 + 2 * slot] = s;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) moved[0] = s_count;
}

constexpr int CNB = 512;  // complex outer block

// Applies a panel's moved-row list to the columns [lo1, hi1) and [lo2, hi2): one wave64 per
// column gathers every source row, then scatters.
__global__ __launch_bounds__(256) void couter_swap_kernel(float2* __restrict__ A, int lda, int lo1, int hi1, int lo2,
                                                          int hi2, const int* __restrict__ moved)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int idx = blockIdx.x * 4 + wave;
    const int n1 = hi1 - lo1;
    if (idx >= n1 + (hi2 - lo2)) return;
    const int c = idx < n1 ? lo1 + idx : lo2 + (idx - n1);
    float2* col = A + static_cast<size_t>(c) * lda;
    const int cnt = moved[0];
    constexpr int MAXQ = (2 * CNB + 63) / 64;
    float2 v[MAXQ];
    int d[MAXQ];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q)
    {
        const int e = lane + 64 * q;
        d[q] = -1;
        if (e < cnt)
        {
            d[q] = moved[1 + 2 * e];
            v[q] = col[moved[2 + 2 * e]];
        }
    }
#pragma unroll
    for (int q = 0; q < MAXQ; ++q)
        if (d[q] >= 0) col[d[q]] = v[q];
}

// C (MxN) -= op(A) (MxK) * B (KxN), complex64, four real FP32 MFMA products per block; op(A):
// transA 0 = A, 1 = A^T, 2 = A^H. Tiles of 64 Q x 64 Q per workgroup of 4 Q waves, 32 Q x 32 per
// wave, k chunks of 16 staged through LDS (parts apart) with the next chunk prefetched into
// registers; formed as C^T, so that an accumulator register holds 32 consecutive rows of C. Bound
// by the matrix cores and, beside a panel, by what the panel takes: 78 to 82 TF at 7680 x 7168 x 512
// (64 x 64 tiles without prefetch before: 67).
template <int TRANSA, int Q>
__global__ __launch_bounds__(256 * Q) __attribute__((amdgpu_waves_per_eu(4))) void cgemm_sub_kernel(
    int M, int N, int K, const float2* __restrict__ A, int64_t lda, const float2* __restrict__ B, int64_t ldb,
    float2* __restrict__ C, int64_t ldc, int tilesM, int tilesN)
{
    constexpr int KC = 16, TS = 64 * Q, E = 4;
    __shared__ float Ar[2][KC][TS + 4], Ai[2][KC][TS + 4], Br[2][KC][TS + 4], Bi[2][KC][TS + 4];
    int id = blockIdx.x;
    const int total = tilesM * tilesN;
    // Workgroups go round the XCDs: each XCD gets a run of tiles, so that neighbours share L2.
    if (total >= 64) id = id < (total & ~7) ? (id & 7) * (total >> 3) + (id >> 3) : id;
    const int row0 = id % tilesM * TS, col0 = id / tilesM * TS;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = (wave & 1) * 32 * Q + (lane & 31), wn = (wave >> 1) * 32 + (lane & 31), lk = lane >> 5;
    f32x16 accR[Q], accI[Q];
#pragma unroll
    for (int i = 0; i < Q; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) accR[i][v] = accI[i][v] = 0.0f;
    // Rows and columns beyond the edge repeat the last one: their products are not stored. Sixteen
    // lanes read the 128 bytes of a chunk of one column of B (of one row of op(A) when
    // transposed), so that a line is fetched by one load, not by eight.
    const int ar = TRANSA ? tid >> 4 : tid % TS, ak = TRANSA ? tid & 15 : tid / TS * E;
    const int bj = tid >> 4, bk = tid & 15;
    const float2* const Arow = A + static_cast<int64_t>(min(row0 + ar, M - 1)) * (TRANSA ? lda : 1);
    const float2* const Bcol = B + static_cast<int64_t>(min(col0 + bj, N - 1)) * ldb;
    float2 ra[E], rb[E];
    auto gload = [&](int k0)
    {
        const int kb = k0 + bk;
        const float2* pa = Arow + (TRANSA ? min(kb, K - 1) : 0);
        const float2* pb = Bcol + min(kb, K - 1);
#pragma unroll
        for (int q = 0; q < E; ++q)
        {
            const int ka = TRANSA ? kb : k0 + ak + q;
            ra[q] = TRANSA ? *pa : pa[static_cast<int64_t>(min(ka, K - 1)) * lda];
            rb[q] = *pb;
            if (ka >= K) ra[q] = make_float2(0.0f, 0.0f);
            if (kb >= K) rb[q] = make_float2(0.0f, 0.0f);
            if (TRANSA) pa += row0 + ar + 16 * Q * (q + 1) < M ? 16 * Q * lda : 0;
            pb += col0 + bj + 16 * Q * (q + 1) < N ? 16 * Q * ldb : 0;
        }
    };
    auto lstore = [&](int buf)
    {
#pragma unroll
        for (int q = 0; q < E; ++q)
        {
            const int k = TRANSA ? ak : ak + q, r = TRANSA ? ar + 16 * Q * q : ar;
            Ar[buf][k][r] = ra[q].x;
            Ai[buf][k][r] = TRANSA == 2 ? -ra[q].y : ra[q].y;
            Br[buf][bk][bj + 16 * Q * q] = rb[q].x;
            Bi[buf][bk][bj + 16 * Q * q] = rb[q].y;
        }
    };
    const int chunks = (K + KC - 1) / KC;
    gload(0);
    lstore(0);
    __syncthreads();
    for (int c = 0; c < chunks; ++c)
    {
        const int buf = c & 1;
        if (c + 1 < chunks) gload((c + 1) * KC);
#pragma unroll
        for (int kk = 0; kk < KC; kk += 2)
        {
            const float yr = Br[buf][kk + lk][wn], yi = Bi[buf][kk + lk][wn];
            float xr[Q], xi[Q];
#pragma unroll
            for (int i = 0; i < Q; ++i)
            {
                xr[i] = Ar[buf][kk + lk][wm + 32 * i];
                xi[i] = Ai[buf][kk + lk][wm + 32 * i];
            }
#pragma unroll
            for (int i = 0; i < Q; ++i)
            {
                accR[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(yr, xr[i], accR[i], 0, 0, 0);
                accI[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(yi, xr[i], accI[i], 0, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < Q; ++i)
            {
                accR[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(-yi, xi[i], accR[i], 0, 0, 0);
                accI[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(yr, xi[i], accI[i], 0, 0, 0);
            }
        }
        if (c + 1 < chunks) lstore(buf ^ 1);
        __syncthreads();
    }
    // Loads before stores, eight at a time (a load under its own condition waits by itself).
#pragma unroll
    for (int bi = 0; bi < Q; ++bi)
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            const int i = row0 + wm + 32 * bi, j0 = col0 + (wave >> 1) * 32 + 4 * lk + 16 * h;
            float2 x[8];
#pragma unroll
            for (int v = 0; v < 8; ++v)
                x[v] = C[static_cast<int64_t>(min(j0 + (v & 3) + 8 * (v >> 2), N - 1)) * ldc + min(i, M - 1)];
#pragma unroll
            for (int v = 0; v < 8; ++v)
            {
                const int j = j0 + (v & 3) + 8 * (v >> 2);
                if (i < M && j < N)
                    C[j * ldc + i] = make_float2(x[v].x - accR[bi][8 * h + v], x[v].y - accI[bi][8 * h + v]);
            }
        }
}

template <int CTRL>
__device__ inline float2 QuadBroadcast2(float2 v)
{
    return make_float2(__int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v.x), CTRL, 0xF, 0xF, false)),
                       __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v.y), CTRL, 0xF, 0xF, false)));
}

// B <- op(T)^{-1} B on one diagonal block of kb <= 64 rows, complex; op: 0 = T, 1 = T^T,
// 2 = T^H. Four lanes (a quad) share one column of B, lane q holding rows 16q .. 16q+15 in
// registers; the unknown of step s is broadcast in the quad with DPP, so a lane's serial
// chain is 16 updates per step. op(T) and the FP64 reciprocals of its diagonal sit in LDS.
// Per element: the same SubMul step per term, in pivot order, and the same FP64-reciprocal
// scaling per pivot as the unblocked complex solve; rows outside the triangle are kept by
// a select.
template <bool FWD, bool UNIT, int TRANS>
__global__ __launch_bounds__(256) void ctrsm_diag64_kernel(int kb, int N, const float2* __restrict__ T, int ldt,
                                                           float2* __restrict__ B, int ldb)
{
    __shared__ float2 Ts[64][64];  // Ts[s][i] = op(T)(i, s)
    __shared__ double2 Dinv[64];
    auto opT = [&](int i, int s2)
    { return Conj(TRANS ? T[static_cast<size_t>(i) * ldt + s2] : T[static_cast<size_t>(s2) * ldt + i], TRANS == 2); };
    for (int e = threadIdx.x; e < 64 * 64; e += 256)
    {
        const int s2 = e >> 6, i = e & 63;
        Ts[s2][i] = (i < kb && s2 < kb) ? opT(i, s2) : make_float2(0.0f, 0.0f);
    }
    if (!UNIT)
        for (int t = threadIdx.x; t < kb; t += 256) Dinv[t] = Recip64(opT(t, t));
    __syncthreads();
    const int col = blockIdx.x * 64 + (threadIdx.x >> 2), q = threadIdx.x & 3;
    const bool live = col < N;
    float2* b = B + static_cast<size_t>(live ? col : 0) * ldb;
    float2 x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) x[t] = (live && 16 * q + t < kb) ? b[16 * q + t] : make_float2(0.0f, 0.0f);
#pragma unroll
    for (int u = 0; u < 64; ++u)
    {
        const int s2 = FWD ? u : 63 - u;
        if (s2 >= kb) continue;  // uniform
        const int o = s2 >> 4, so = s2 & 15;
        float2 xs;
        if (o == 0)
            xs = QuadBroadcast2<0x00>(x[so]);
        else if (o == 1)
            xs = QuadBroadcast2<0x55>(x[so]);
        else if (o == 2)
            xs = QuadBroadcast2<0xAA>(x[so]);
        else
            xs = QuadBroadcast2<0xFF>(x[so]);
        if (!UNIT) xs = Mul64(xs, Dinv[s2]);
        if (q == o) x[so] = xs;
#pragma unroll
        for (int t = 0; t < 16; ++t)
        {
            const int row = 16 * q + t;
            const bool upd = FWD ? row > s2 : row < s2;
            const float2 nx = SubMul(x[t], Ts[s2][row], xs);
            x[t] = upd ? nx : x[t];
        }
    }
#pragma unroll
    for (int t = 0; t < 16; ++t)
        if (live && 16 * q + t < kb) b[16 * q + t] = x[t];
}

template <int Q>
hipError_t LaunchCGemm(int M, int N, int K, const float2* A, int lda, int transA, const float2* B, int ldb, float2* C,
                       int ldc, hipStream_t stream)
{
    const int tilesM = (M + 64 * Q - 1) / (64 * Q), tilesN = (N + 64 * Q - 1) / (64 * Q);
    const dim3 grid(tilesM * tilesN);
    // LDS for one workgroup of the large tiles per compute unit: with its 128 registers a lane on
    // eight waves the other half of the registers stays free for the panel beside it, whose leaves
    // otherwise wait for a tile to end (n = 8192: 37.9 ms with two workgroups of four waves, 37.2).
    const int pad = Q == 2 ? 16384 : 0;
#define CG_CASE(TR)                                                                                           \
    hipLaunchKernelGGL((cgemm_sub_kernel<TR, Q>), grid, dim3(256 * Q), pad, stream, M, N, K, A,               \
                       static_cast<int64_t>(lda), B, static_cast<int64_t>(ldb), C, static_cast<int64_t>(ldc), \
                       tilesM, tilesN)
    if (transA == 0)
        CG_CASE(0);
    else if (transA == 1)
        CG_CASE(1);
    else
        CG_CASE(2);
#undef CG_CASE
    return hipGetLastError();
}

hipError_t CGemmSub(int M, int N, int K, const float2* A, int lda, int transA, const float2* B, int ldb, float2* C,
                    int ldc, hipStream_t stream)
{
    if (M <= 0 || N <= 0 || K <= 0) return hipSuccess;
    const int64_t big = static_cast<int64_t>((M + 127) / 128) * ((N + 127) / 128);
    // At least a tile per compute unit (cgetrf n = 3000: lines at 64 / 256 / 1024 tiles 8.90 / 8.69 / 8.75
    // ms, n = 4500 15.04 / 14.81 / 14.96).
    if (big >= 256) return LaunchCGemm<2>(M, N, K, A, lda, transA, B, ldb, C, ldc, stream);
    return LaunchCGemm<1>(M, N, K, A, lda, transA, B, ldb, C, ldc, stream);
}

template <bool FWD, bool UNIT, int TRANS>
hipError_t LaunchCTrsmDiag(int kb, int N, const float2* T, int ldt, float2* B, int ldb, hipStream_t stream)
{
    hipLaunchKernelGGL((ctrsm_diag64_kernel<FWD, UNIT, TRANS>), dim3((N + 63) / 64), dim3(256), 0, stream, kb, N, T,
                       ldt, B, ldb);
    return hipGetLastError();
}

hipError_t CTrsmDiag(int kb, int N, const float2* T, int ldt, bool fwd, bool unit, int trans, float2* B, int ldb,
                     hipStream_t stream)
{
#define CD_CASE(F, U, TR) \
    if (fwd == F && unit == U && trans == TR) return LaunchCTrsmDiag<F, U, TR>(kb, N, T, ldt, B, ldb, stream)
    CD_CASE(true, true, 0);
    CD_CASE(true, false, 0);
    CD_CASE(false, true, 0);
    CD_CASE(false, false, 0);
    CD_CASE(true, true, 1);
    CD_CASE(true, false, 1);
    CD_CASE(false, true, 1);
    CD_CASE(false, false, 1);
    CD_CASE(true, true, 2);
    CD_CASE(true, false, 2);
    CD_CASE(false, true, 2);
    CD_CASE(false, false, 2);
#undef CD_CASE
    return hipErrorInvalidValue;
}

// B <- op(T)^{-1} B, complex, any K: 64-row diagonal solves interleaved with complex GEMM
// updates of the rows still to be solved.
hipError_t CTrsmBlock(int K, int N, const float2* T, int ldt, bool lower, bool unit, int trans, float2* B, int ldb,
                      hipStream_t stream)
{
    if (K <= 0 || N <= 0) return hipSuccess;
    const bool fwd = lower != (trans != 0);
    const int nblk = (K + 63) / 64;
    for (int q = 0; q < nblk; ++q)
    {
        const int bi = fwd ? q : nblk - 1 - q;
        const int k0 = bi * 64, kb = std::min(64, K - k0), k1 = k0 + kb;
        hipError_t e = CTrsmDiag(kb, N, T + static_cast<size_t>(k0) * ldt + k0, ldt, fwd, unit, trans, B + k0, ldb,
                                 stream);
        if (e != hipSuccess) return e;
        if (fwd && k1 < K)
        {
            const float2* Ablk = trans ? T + static_cast<size_t>(k1) * ldt + k0 : T + static_cast<size_t>(k0) * ldt + k1;
            e = CGemmSub(K - k1, N, kb, Ablk, ldt, trans, B + k0, ldb, B + k1, ldb, stream);
        }
        else if (!fwd && k0 > 0)
        {
            const float2* Ablk = trans ? T + k0 : T + static_cast<size_t>(k0) * ldt;
            e = CGemmSub(k0, N, kb, Ablk, ldt, trans, B + k0, ldb, B, ldb, stream);
        }
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

// Workspace: ints [0, m) row sources, two moved-row lists of 4 CNB + 8 (panel k uses list
// k % 2, so the look-ahead panel can build its list while the previous one is still being
// applied), the leaf's moved rows; then, 8-byte aligned, the exchange words of the
// multi-workgroup leaves, the rows a leaf's update takes, two panels' solve forms (unitlower.h) and
// the timeout flag.
constexpr int kCMovedInts = 4 * CNB + 8;
inline int CPanelBlocks(int m) { return (std::min(m, CNB) + 63) / 64; }
struct CWork
{
    int* rowsrc;
    int* moved[2];
    int* moves;
    unsigned long long* slots;
    float2* panelRows;
    float* forms[2];
    int* err;
};
inline size_t CWorkInts(int m) { return static_cast<size_t>(m) + 2 * kCMovedInts + 4 * kCLeafWidth + 2; }
inline size_t CWorkWords(int m)  // 8-byte words behind the ints
{
    const size_t blocks = static_cast<size_t>(CPanelBlocks(m));
    return kCLeafSlotWords + blocks * 64 * 64 + 2 * blocks * (kCFormBlock / 2) + 1;
}
CWork CLayout(void* base, int m)
{
    const size_t blocks = static_cast<size_t>(CPanelBlocks(m));
    CWork w;
    uintptr_t q = (reinterpret_cast<uintptr_t>(base) + 7) & ~static_cast<uintptr_t>(7);
    w.slots = reinterpret_cast<unsigned long long*>(q);
    w.panelRows = reinterpret_cast<float2*>(w.slots + kCLeafSlotWords);
    w.forms[0] = reinterpret_cast<float*>(w.panelRows + blocks * 64 * 64);
    w.forms[1] = w.forms[0] + blocks * kCFormBlock;
    w.err = reinterpret_cast<int*>(w.forms[1] + blocks * kCFormBlock);
    w.moves = w.err + 2;
    w.moved[0] = w.moves + 4 * kCLeafWidth;
    w.moved[1] = w.moved[0] + kCMovedInts;
    w.rowsrc = w.moved[1] + kCMovedInts;
    return w;
}

#define CRET(e)                          \
    do                                   \
    {                                    \
        hipError_t _e = (e);             \
        if (_e != hipSuccess) return _e; \
    } while (0)

}  // namespace

size_t ComplexGetrfWorkspaceBytes(int m, int n)
{
    (void)n;
    m = std::max(m, 1);
    return CWorkInts(m) * sizeof(int) + CWorkWords(m) * 8 + 16;
}

hipError_t ComplexGetrf(int m, int n, float2* a, int lda, int* ipiv, int* info, void* work, hipStream_t stream,
                        const LookAhead* la)
{
    if (m > kCLeafMaxRows) return hipErrorInvalidValue;
    CWork w = CLayout(work, m);
    FillInfo(info, 1, 0, stream);
    const bool multi = m > kCLeafSingleRows;
    {
        const int words = multi ? kCLeafSlotWords : 0;
        hipLaunchKernelGGL(cclear_slots_kernel, dim3(std::max(1, (words + 255) / 256)), dim3(256), 0, stream, w.slots,
                           words, w.err);
    }
    const int kmax = std::min(m, n);
    if (kmax == 0) return hipGetLastError();
    const int pivoting = ipiv != nullptr;
    const int npanel = (kmax + CNB - 1) / CNB;

    // Look-ahead, as in the real factorization: the caller's stream s0 carries the critical
    // path (the next block column's update and its panel), the side stream s1 the rest of
    // each trailing update.
    const bool two = la != nullptr && la->side != nullptr && npanel > 1;
    hipStream_t s0 = stream, s1 = two ? la->side : stream;
    if (two)
    {
        CRET(hipEventRecord(la->fork, stream));
        CRET(hipStreamWaitEvent(s1, la->fork, 0));
    }

    // Panel k: per 64 columns one leaf, one launch that applies its interchanges to the whole
    // panel and prepares its diagonal block, one that updates the panel columns to its right;
    // then the list of the panel's interchanges.
    auto panel = [&](int k) -> hipError_t
    {
        const int j0 = k * CNB, panelEnd = std::min(j0 + CNB, kmax);
        for (int c0 = j0; c0 < panelEnd; c0 += kCLeafWidth)
        {
            CLeafArgs l;
            l.A = a;
            l.lda = lda;
            l.m = m;
            l.j0 = j0;
            l.c0 = c0;
            l.wact = std::min(kCLeafWidth, panelEnd - c0);
            l.panelEnd = panelEnd;
            l.pivoting = pivoting;
            l.newPanel = c0 == j0;
            l.ipiv = ipiv;
            l.info = info;
            l.rowsrc = w.rowsrc;
            l.moves = w.moves;
            l.slots = w.slots;
            // The key words carry 16 bits of a tag: at most 256 leaves of 64 tags and the first.
            l.tagBase = static_cast<unsigned>(c0 + kCLeafWidth);
            l.err = w.err;
            l.spinLimit = SpinLimit();
            float* const form = w.forms[k & 1] + static_cast<size_t>((c0 - j0) / 64) * kCFormBlock;
            CRET(CLeafColumns(l, LeafSpread(), s0));
            CRET(CLeafFinish(l, form, w.panelRows, s0));
            if (c0 + l.wact < panelEnd) CRET(CPanelUpdate(l, form, w.panelRows, s0));
        }
        if (pivoting && (k > 0 || panelEnd < n))
            hipLaunchKernelGGL(ccompact_moves_kernel, dim3(1), dim3(1024), 0, s0, m, j0, w.rowsrc, w.err,
                               w.moved[k & 1]);
        return hipGetLastError();
    };
    // Applies panel k to the columns [lo, hi) (interchanges, U12 solve, trailing product)
    // and, when leftSwaps, its interchanges to the columns left of the panel.
    auto update = [&](int k, int lo, int hi, bool leftSwaps, hipStream_t st) -> hipError_t
    {
        const int j0 = k * CNB, nb = std::min(CNB, kmax - j0), pe = j0 + nb;
        const int cols = hi - lo, left = leftSwaps ? j0 : 0;
        if (pivoting && cols + left > 0)
            hipLaunchKernelGGL(couter_swap_kernel, dim3((cols + left + 3) / 4), dim3(256), 0, st, a, lda, 0, left, lo,
                               hi, w.moved[k & 1]);
        CRET(hipGetLastError());
        if (cols <= 0) return hipSuccess;
        CRET(CTrsmLowerUnit(nb, cols, a + static_cast<size_t>(j0) * lda + j0, lda, w.forms[k & 1],
                            a + static_cast<size_t>(lo) * lda + j0, lda, st));
        if (m - pe <= 0) return hipSuccess;
        ProfileScope prof(ProfileKernel::ComplexGemm, 8.0 * (m - pe) * cols * nb, st);
        return CGemmSub(m - pe, cols, nb, a + static_cast<size_t>(j0) * lda + pe, lda, 0,
                        a + static_cast<size_t>(lo) * lda + j0, lda, a + static_cast<size_t>(lo) * lda + pe, lda, st);
    };

    CRET(panel(0));
    if (two) CRET(hipEventRecord(la->panel[0], s0));
    for (int k = 0; k < npanel; ++k)
    {
        const int pe = std::min(kmax, (k + 1) * CNB);
        const int nbNext = k + 1 < npanel ? std::min(CNB, kmax - pe) : 0;
        // Bulk of the trailing update (s1): everything right of the next block column, and
        // the interchanges of panel k left of it.
        if (two) CRET(hipStreamWaitEvent(s1, la->panel[k & 1], 0));
        CRET(update(k, pe + nbNext, n, true, s1));
        if (two) CRET(hipEventRecord(la->bulk[k & 1], s1));
        // Critical path (s0): the next block column, then its panel.
        if (nbNext > 0)
        {
            if (two && k > 0) CRET(hipStreamWaitEvent(s0, la->bulk[(k - 1) & 1], 0));
            CRET(update(k, pe, pe + nbNext, false, s0));
            CRET(panel(k + 1));
            if (two) CRET(hipEventRecord(la->panel[(k + 1) & 1], s0));
        }
    }
    if (two) CRET(hipStreamWaitEvent(s0, la->bulk[(npanel - 1) & 1], 0));
    if (multi) FoldWaitError(w.err, info, s0);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// cgetrs (Device, column-major), trans 0 / 1 / 2
// ---------------------------------------------------------------------------------------
namespace
{
template <bool GATHER>
__global__ void cpermute_kernel(int n, int nrhs, const int* __restrict__ perm, const float2* __restrict__ src, int lds,
                                float2* __restrict__ dst, int ldd)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int c = blockIdx.y;
    if (i >= n) return;
    const int p = perm ? perm[i] : i;
    if (GATHER)
        dst[static_cast<size_t>(c) * ldd + i] = src[static_cast<size_t>(c) * lds + p];
    else
        dst[static_cast<size_t>(c) * ldd + p] = src[static_cast<size_t>(c) * lds + i];
}
}  // namespace

namespace
{
// The chain up to 2048 right-hand sides; n = 8192: 1 rhs 10.5 and 2.1 ms (per-block launches, chain),
// 256 12.0 and 3.1, 2048 22.1 and 13.0 (transposed 20.9 and 19.1); n = 400, 2048 rhs: 539 and 191
// us. Beyond, its published words (16 bytes an element) and the re-reading of the factors per 16
// columns outweigh the launches.
bool UseChain(int nrhs) { return nrhs <= kCTrsMaxRhs; }
}  // namespace

size_t ComplexGetrsWorkspaceBytes(int n, int nrhs, bool chain)
{
    if (chain && UseChain(nrhs)) return CTrsWorkspaceBytes(n, nrhs);
    return static_cast<size_t>(n) * std::max(nrhs, 1) * sizeof(float2) + (static_cast<size_t>(n) + 64) * sizeof(int);
}

hipError_t ComplexGetrs(int trans, int n, int nrhs, const float2* lu, int lda, const int* ipiv, float2* b, int ldb,
                        void* work, hipStream_t stream, int* info, bool chain)
{
    if (n <= 0 || nrhs <= 0) return hipSuccess;
    if (n > 16384) return hipErrorInvalidValue;
    if (chain && UseChain(nrhs)) return CTrsSolve(trans, n, nrhs, lu, lda, ipiv, b, ldb, info, work, stream);
    float2* x = static_cast<float2*>(work);
    int* perm = reinterpret_cast<int*>(x + static_cast<size_t>(n) * nrhs);
    if (ipiv) CRET(IpivToPerm(n, ipiv, perm, stream, true));
    const int* p = ipiv ? perm : nullptr;
    const dim3 grid((n + 255) / 256, nrhs);
    const int NBS = 128;
    if (trans == 0)
    {
        hipLaunchKernelGGL(cpermute_kernel<true>, grid, dim3(256), 0, stream, n, nrhs, p, b, ldb, x, n);
        for (int k = 0; k < n; k += NBS)
        {
            const int kb = std::min(NBS, n - k);
            CRET(CTrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, true, true, 0, x + k, n, stream));
            if (n - k - kb > 0)
                CRET(CGemmSub(n - k - kb, nrhs, kb, lu + static_cast<size_t>(k) * lda + k + kb, lda, 0, x + k, n,
                              x + k + kb, n, stream));
        }
        for (int k = ((n - 1) / NBS) * NBS; k >= 0; k -= NBS)
        {
            const int kb = std::min(NBS, n - k);
            CRET(CTrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, false, false, 0, x + k, n, stream));
            if (k > 0)
                CRET(CGemmSub(k, nrhs, kb, lu + static_cast<size_t>(k) * lda, lda, 0, x + k, n, x, n, stream));
        }
        hipLaunchKernelGGL(cpermute_kernel<true>, grid, dim3(256), 0, stream, n, nrhs, nullptr, x, n, b, ldb);
    }
    else
    {
        hipLaunchKernelGGL(cpermute_kernel<true>, grid, dim3(256), 0, stream, n, nrhs, nullptr, b, ldb, x, n);
        for (int k = 0; k < n; k += NBS)  // op(U) w = b, op(U) lower
        {
            const int kb = std::min(NBS, n - k);
            CRET(CTrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, false, false, trans, x + k, n,
                            stream));
            if (n - k - kb > 0)
                CRET(CGemmSub(n - k - kb, nrhs, kb, lu + static_cast<size_t>(k + kb) * lda + k, lda, trans, x + k, n,
                              x + k + kb, n, stream));
        }
        for (int k = ((n - 1) / NBS) * NBS; k >= 0; k -= NBS)  // op(L) z = w, op(L) upper unit
        {
            const int kb = std::min(NBS, n - k);
            CRET(CTrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, true, true, trans, x + k, n,
                            stream));
            if (k > 0) CRET(CGemmSub(k, nrhs, kb, lu + k, lda, trans, x + k, n, x, n, stream));
        }
        hipLaunchKernelGGL(cpermute_kernel<false>, grid, dim3(256), 0, stream, n, nrhs, p, x, n, b, ldb);
    }
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------
// Batched complex inverses, n <= 64: one wave64 group of NL lanes per matrix, lane = row.
// ---------------------------------------------------------------------------------------
namespace
{
template <int NL>
__device__ inline void CGroupArgmax(uint32_t val, int key, uint32_t* bestVal, int* bestKey)
{
    uint32_t b = val;
#pragma unroll
    for (int off = NL / 2; off > 0; off >>= 1) b = max(b, static_cast<uint32_t>(__shfl_xor(b, off)));
    int k = (val == b) ? key : INT_MAX;
#pragma unroll
    for (int off = NL / 2; off > 0; off >>= 1) k = min(k, __shfl_xor(k, off));
    *bestVal = b;
    *bestKey = k;
}

// Gauss-Jordan with implicit pivoting (see batched.hip for the real derivation).
template <int NL>
__global__ __launch_bounds__(256) void cmatinv_gj_kernel(int n, const float2* const* __restrict__ Aarr,
                                                         const float2* __restrict__ Abase, int lda, int64_t strideA,
                                                         float2* const* __restrict__ Carr, float2* __restrict__ Cbase,
                                                         int ldc, int64_t strideC, int* __restrict__ info, int batch)
{
    constexpr int GROUPS = 256 / NL;
    __shared__ float2 s_row[GROUPS][NL];
    __shared__ int s_inv[GROUPS][NL];
    const int tid = threadIdx.x;
    const int g = tid / NL, lane = tid % NL;
    const int mat = blockIdx.x * GROUPS + g;
    const bool live = mat < batch;
    const float2* A = nullptr;
    float2* C = nullptr;
    if (live)
    {
        A = Aarr ? Aarr[mat] : Abase + static_cast<int64_t>(mat) * strideA;
        C = Carr ? Carr[mat] : Cbase + static_cast<int64_t>(mat) * strideC;
    }
    const bool rowLive = live && lane < n;
    float2 S[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j)
        S[j] = (rowLive && j < n) ? A[static_cast<int64_t>(j) * lda + lane] : make_float2(0.0f, 0.0f);
    double2 sigma = make_double2(1.0, 0.0);
    int pos = lane;
    bool used = false;
    int zero = 0;
    // Slot j of S holds column (j + steps done) % NL: each step pivots slot 0 and rotates the
    // slots down by one (the processed column moves to the last slot), so no slot is ever
    // addressed by a run-time index, also where the step loop is not unrolled.
#pragma unroll
    for (int k = 0; k < NL; ++k)
    {
        if (k < n)
        {
            const float2 sk = S[0];
            const uint32_t cand = (rowLive && !used) ? PivotScore(sk) : 0u;
            uint32_t best;
            int key;
            CGroupArgmax<NL>(rowLive && !used ? cand : 0u, (rowLive && !used) ? ((pos << 8) | lane) : INT_MAX,
                             &best, &key);
            const int p = key & 0xFF;
            const int ppos = key >> 8;
            const bool isP = lane == p;
            if (pos == k) pos = ppos;
            if (isP) pos = k;
            if (isP)
            {
#pragma unroll
                for (int j = 0; j < NL; ++j) s_row[g][j] = S[j];
            }
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            const float2 d = s_row[g][0];
            const bool z = d.x == 0.0f && d.y == 0.0f;
            if (z && zero == 0) zero = k + 1;
            const double2 r = Recip64(z ? make_float2(1.0f, 0.0f) : d);
            const float2 c = (isP || z) ? make_float2(0.0f, 0.0f) : Mul64(sk, r);
            const float2 last = z ? sk : (isP ? make_float2(1.0f, 0.0f) : make_float2(-c.x, -c.y));
#pragma unroll
            for (int j = 1; j < NL; ++j) S[j - 1] = SubMul(S[j], c, s_row[g][j]);
            S[NL - 1] = last;
            if (!z && isP) sigma = r;
            if (isP) used = true;
            __builtin_amdgcn_wave_barrier();
        }
    }
    if (rowLive) s_inv[g][pos] = lane;
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    if (rowLive)
    {
#pragma unroll
        for (int kk = 0; kk < NL; ++kk)
        {
            const int j = kk + n < NL ? kk + n : kk + n - NL;  // the column slot kk holds
            if (j < n) C[static_cast<int64_t>(s_inv[g][j]) * ldc + pos] = Mul64(S[kk], sigma);
        }
    }
    if (live && lane == 0) info[mat] = zero;
}

template <int NL>
__global__ __launch_bounds__(256) void cgetri_small_kernel(int n, const float2* const* __restrict__ Aarr, int lda,
                                                           const int* __restrict__ piv,
                                                           float2* const* __restrict__ Carr, int ldc,
                                                           int* __restrict__ info, int batch)
{
    constexpr int GROUPS = 256 / NL;
    __shared__ float2 s_row[GROUPS][NL];
    __shared__ int s_perm[GROUPS][NL];
    const int tid = threadIdx.x;
    const int g = tid / NL, lane = tid % NL;
    const int mat = blockIdx.x * GROUPS + g;
    const bool live = mat < batch;
    const bool rowLive = live && lane < n;
    const float2* A = live ? Aarr[mat] : nullptr;
    float2* C = live ? Carr[mat] : nullptr;
    // The factor entries of this lane's row are read from memory one column per step (the
    // next column is fetched a step ahead), so no register array is indexed by the step.
    auto factor = [&](int q) -> float2
    { return (rowLive && q >= 0 && q < n) ? A[static_cast<int64_t>(q) * lda + lane] : make_float2(0.0f, 0.0f); };
    if (live && lane == 0)
    {
        for (int i = 0; i < n; ++i) s_perm[g][i] = i;
        for (int k = 0; k < n; ++k)
        {
            int p = piv ? piv[static_cast<int64_t>(mat) * n + k] - 1 : k;
            p = p < k || p >= n ? k : p;
            const int t = s_perm[g][k];
            s_perm[g][k] = s_perm[g][p];
            s_perm[g][p] = t;
        }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    float2 X[NL];
    const int pr = rowLive ? s_perm[g][lane] : -1;
#pragma unroll
    for (int j = 0; j < NL; ++j) X[j] = make_float2(j == pr ? 1.0f : 0.0f, 0.0f);
    float2 fnext = factor(0);
#pragma unroll(NL <= 32 ? NL : 1)
    for (int q = 0; q < NL; ++q)
    {
        if (q < n)
        {
            const float2 fq = fnext;
            fnext = factor(q + 1);
            if (lane == q)
            {
#pragma unroll
                for (int j = 0; j < NL; ++j) s_row[g][j] = X[j];
            }
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (lane > q && rowLive)
            {
                const float2 l = fq;
#pragma unroll
                for (int j = 0; j < NL; ++j) X[j] = SubMul(X[j], l, s_row[g][j]);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    fnext = factor(n - 1);
#pragma unroll(NL <= 32 ? NL : 1)
    for (int q = NL - 1; q >= 0; --q)
    {
        if (q < n)
        {
            const float2 fq = fnext;
            fnext = factor(q - 1);
            if (lane == q)
            {
                const float2 d = fq;
                const bool z = d.x == 0.0f && d.y == 0.0f;
                const double2 r = Recip64(z ? make_float2(1.0f, 0.0f) : d);
#pragma unroll
                for (int j = 0; j < NL; ++j)
                {
                    if (!z) X[j] = Mul64(X[j], r);
                    s_row[g][j] = X[j];
                }
            }
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (lane < q && rowLive)
            {
                const float2 uq = fq;
#pragma unroll
                for (int j = 0; j < NL; ++j) X[j] = SubMul(X[j], uq, s_row[g][j]);
            }
            __builtin_amdgcn_wave_barrier();
        }
    }
    const float2 diag = factor(lane);
    const unsigned long long zmask = __ballot(rowLive && diag.x == 0.0f && diag.y == 0.0f);
    const int shift = (g * NL) % 64;
    const unsigned long long gmask = (NL >= 64) ? ~0ull : ((~0ull >> (64 - NL)) << shift);
    const unsigned long long mine = zmask & gmask;
    const int zero = mine ? (__ffsll(static_cast<long long>(mine)) - 1 - shift) + 1 : 0;
    if (rowLive)
    {
#pragma unroll
        for (int j = 0; j < NL; ++j)
            if (j < n) C[static_cast<int64_t>(j) * ldc + lane] = X[j];
    }
    if (live && lane == 0) info[mat] = zero;
}

template <int NL>
hipError_t LaunchCMatinv(int n, const float2* const* Aarr, const float2* Abase, int lda, int64_t strideA,
                         float2* const* Carr, float2* Cbase, int ldc, int64_t strideC, int* info, int batch,
                         hipStream_t stream)
{
    constexpr int GROUPS = 256 / NL;
    hipLaunchKernelGGL(cmatinv_gj_kernel<NL>, dim3((batch + GROUPS - 1) / GROUPS), dim3(256), 0, stream, n, Aarr,
                       Abase, lda, strideA, Carr, Cbase, ldc, strideC, info, batch);
    return hipGetLastError();
}

template <int NL>
hipError_t LaunchCGetri(int n, const float2* const* Aarr, int lda, const int* piv, float2* const* Carr, int ldc,
                        int* info, int batch, hipStream_t stream)
{
    constexpr int GROUPS = 256 / NL;
    hipLaunchKernelGGL(cgetri_small_kernel<NL>, dim3((batch + GROUPS - 1) / GROUPS), dim3(256), 0, stream, n, Aarr,
                       lda, piv, Carr, ldc, info, batch);
    return hipGetLastError();
}
}  // namespace

hipError_t CMatinvBatched(int n, const float2* const* Aarr, const float2* Abase, int lda, int64_t strideA,
                          float2* const* Carr, float2* Cbase, int ldc, int64_t strideC, int* info, int batch,
                          hipStream_t stream)
{
    if (batch <= 0) return hipSuccess;
    if (n <= 8) return LaunchCMatinv<8>(n, Aarr, Abase, lda, strideA, Carr, Cbase, ldc, strideC, info, batch, stream);
    if (n <= 16)
        return LaunchCMatinv<16>(n, Aarr, Abase, lda, strideA, Carr, Cbase, ldc, strideC, info, batch, stream);
    if (n <= 32)
        return LaunchCMatinv<32>(n, Aarr, Abase, lda, strideA, Carr, Cbase, ldc, strideC, info, batch, stream);
    if (n <= 64) return CMatinvRows64(n, Aarr, Abase, lda, strideA, Carr, Cbase, ldc, strideC, info, batch, stream);
    return hipErrorNotSupported;  // 64 < n: the caller takes the factor-and-solve route
}

hipError_t CGetriSmallBatched(int n, const float2* const* Aarr, int lda, const int* piv, float2* const* Carr, int ldc,
                              int* info, int batch, hipStream_t stream)
{
    if (batch <= 0) return hipSuccess;
    if (n <= 8) return LaunchCGetri<8>(n, Aarr, lda, piv, Carr, ldc, info, batch, stream);
    if (n <= 16) return LaunchCGetri<16>(n, Aarr, lda, piv, Carr, ldc, info, batch, stream);
    if (n <= 32) return LaunchCGetri<32>(n, Aarr, lda, piv, Carr, ldc, info, batch, stream);
    if (n <= 64) return LaunchCGetri<64>(n, Aarr, lda, piv, Carr, ldc, info, batch, stream);
    return hipErrorNotSupported;
}

}  // namespace ops
