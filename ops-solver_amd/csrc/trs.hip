// Device triangular solves from packed LU factors with any number of right-hand sides, gfx950.
// Reference: src/sgetrs/real_getrs_kernel.cpp (row permutation, unit-lower and upper solves).
//
// One launch per triangle. A workgroup owns 64 rows of up to 64 right-hand sides and walks the
// blocks it depends on in the order in which they are finished: it waits for X_k, subtracts
// T(i, k) X_k on the FP32 matrix cores (the next tile of T is loaded meanwhile), and at the end
// applies the FP64 inverse of its diagonal block on the FP64 matrix cores and publishes X_i as
// tagged 64-bit words (32-bit tag, value), so that a consumer needs neither a flag nor a fence.
// Tickets hand out the blocks in dependency order: the block with the lowest unfinished ticket
// never waits for a workgroup that has not started. With the inverse in FP64 the block solve
// rounds once; an FP32 inverse, applied once or with a step of refinement in FP32, erred more
// than the substitution it replaces (Gaussian systems of order 64 to 4096, against 64 bits). The
// solve's backward error is that of a substitution in FP32 as long as Growth64 stays far below
// 2^53 / 2^24; blocks above 2^20 (a zero or tiny pivot, multipliers of one sign) are substituted.
// Factors of Gaussian, uniform and graded matrices of orders up to 2500 have 2^12 at most.
//
// What bounds it: the chain, one device-wide trip, two products and a few barriers per 64
// rows. 64 rows: the longest block whose inverse four waves apply from registers.
#include "trs.h"

#include <algorithm>
#include <cfloat>
#include <climits>

#include "growth.h"
#include "internal.h"
#include "lanes.h"
#include "permute.h"
#include "trtri64.h"

namespace ops
{
namespace
{
constexpr int NBK = 64;

__device__ inline unsigned long long LoadWord(const unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct Trs
{
    int trans, n, nrhs, lda, ldb;
    const float* lu;
    const int* ipiv;
    float* B;
    int* info;
    unsigned long long* pub;  // X words: [block][strip][row][column], 64 rows, strips of 16 CG columns
    double* inv;              // inverses of the diagonal blocks of op(L), op(U): row-major 64 x 64
    int* bad;                 // per diagonal block: its inverse is too large to be used (2 nb ints)
    int* perm;
    unsigned* ticket;         // [2]
    unsigned spinLimit;
};

// Preparation, by workgroup: 2 nb diagonal blocks inverted, the permutation (256 positions
// each), the publication words cleared.
__global__ __launch_bounds__(256) void trs_prep_kernel(Trs p, int nb, int np, size_t words)
{
    extern __shared__ __align__(16) double s_mem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int b = blockIdx.x;
    if (b == 0 && tid == 0)
    {
        p.ticket[0] = p.ticket[1] = 0u;
        if (p.info != nullptr) *p.info = 0;
    }
    if (b < 2 * nb)
    {
        const bool upper = b >= nb;
        const int k0 = (upper ? b - nb : b) * NBK, kb = min(NBK, p.n - k0);
        double* const s_l = s_mem;
        double* const s_i = s_mem + 64 * kInvStride;
        double* const s_t = s_i + 64 * kInvStride;
        double* const s_g = s_t + 32 * kInvStride;
        const float* const T = p.lu + static_cast<size_t>(k0) * p.lda + k0;
        // Lower: the block; upper: its transpose. Rows beyond the block are the identity.
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            const int c = wave * 16 + k;
            float v = lane < kb && c < kb ? T[static_cast<size_t>(c) * p.lda + lane] : 0.0f;
            if (lane == c && (!upper || lane >= kb)) v = 1.0f;
            if (upper ? lane > c : lane < c) v = 0.0f;
            s_l[upper ? c * kInvStride + lane : lane * kInvStride + c] = v;
            s_i[lane * kInvStride + c] = 0.0;
        }
        __syncthreads();
        // s_l is op(T) or, if flip, its transpose. The rows' maxima, in halves, beside the first phase
        // of the inversion, which these two waves have no part in.
        const bool flip = upper != (p.trans != 0);
        const int step = flip ? kInvStride : 1, first = flip ? lane : lane * kInvStride;
        if (wave >= 2)
        {
            double d = 0.0;
#pragma unroll
            for (int j = 0; j < 32; ++j) d = fmax(d, fabs(s_l[first + (32 * (wave - 2) + j) * step]));
            s_g[64 * (wave - 2) + lane] = d;
        }
        if (upper)
            InvertLower64<false>(s_l, s_i, s_t, tid);
        else
            InvertLower64<true>(s_l, s_i, s_t, tid);
        // Row-major inverse of op(T): L^-1 and (U^T)^-1 as they are, the other two transposed.
        double* const out = p.inv + static_cast<size_t>(b) * 4096;
        const double d = fmax(s_g[lane], s_g[64 + lane]);
        bool fine = true, small = true;
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            const int r = wave * 16 + k;
            const double v = flip ? s_i[lane * kInvStride + r] : s_i[r * kInvStride + lane];
            fine = fine && fabs(v) <= FLT_MAX;
            small = small && fabs(v) * d <= kSmallInverse;
            out[r * 64 + lane] = v;
        }
        if (!__syncthreads_and(fine && small))
        {
            float e[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) e[k] = fabs(s_l[first + (16 * wave + k) * step]);
            RowMaxima(s_g)[lane] = d;
            __syncthreads();
            const double grow = Growth64(e, [&](int j) { return fabs(s_i[first + j * step]); }, s_g, tid);
            fine = __syncthreads_and(fine && grow <= kInverseGrowth64);
        }
        if (tid == 0) p.bad[b] = fine ? 0 : 1;
        return;
    }
    b -= 2 * nb;
    if (b < np)
    {
        int* const s_piv = reinterpret_cast<int*>(s_mem);
        const int i = b * 256 + tid;
        bool plain = true;
        for (int k = tid; k < p.n; k += 256)
        {
            int v = p.ipiv[k] - 1;
            if (v < 0 || v >= p.n) v = k;
            plain = plain && v >= k;
            s_piv[k] = v;
        }
        plain = __syncthreads_and(plain);
        const int x = TracePosition(s_piv, p.n, i, b * 256 + wave * 64, plain);
        if (i < p.n) p.perm[i] = x;
        return;
    }
    b -= np;
    const size_t step = static_cast<size_t>(gridDim.x - 2 * nb - np) * 256;
    for (size_t w = static_cast<size_t>(b) * 256 + tid; w < words; w += step) p.pub[w] = 0ull;
}

// SECOND: the second substitution of the solve (reads the first one's words, writes B).
// TRANS: op(T) = T^T. CG: 16-column groups per strip.
// Tile operand: lane (li, g) holds row 16 wave + li of the tile and its columns 16 q + 4 g + t,
// q, t = 0..3, so that the four columns of a lane are consecutive; the other operand is read
// from LDS in the same order.
template <bool TRANS, bool SECOND, int CG>
__global__ __launch_bounds__(256) void trs_chain_kernel(Trs p, int nb, int strips)
{
    constexpr bool UPPER = TRANS != SECOND;  // N: L then U; T: U^T then L^T
    constexpr bool BACK = SECOND;            // both second substitutions run upward
    constexpr int NS = 16 * CG, S = NS + 4;
    constexpr int PER = 64 * NS / 256;
    constexpr unsigned TAG = SECOND ? 2u : 1u;
    __shared__ __align__(16) float s_x[2][64 * S];
    __shared__ unsigned s_id;
    __shared__ int s_fail;  // a wait of this workgroup ran out
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, g = lane >> 4;
    if (tid == 0)
    {
        s_id = atomicAdd(p.ticket + (SECOND ? 1 : 0), 1u);
        s_fail = 0;
    }
    __syncthreads();
    const int id = static_cast<int>(s_id);
    const int step = id / strips, strip = id - step * strips;
    const int ib = BACK ? nb - 1 - step : step;
    const int r0 = ib * NBK, c0 = strip * NS;
    const int row = r0 + 16 * wave + li;
    const bool inRow = row < p.n;
    const bool vec = TRANS && p.lda % 4 == 0 && (reinterpret_cast<uintptr_t>(p.lu) & 15) == 0;

    auto loadTile = [&](int kb, float (&t)[16])
    {
        const int k0 = kb * NBK;
        if (TRANS)
        {
            const float* const col = p.lu + static_cast<size_t>(inRow ? row : 0) * p.lda + k0 + 4 * g;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (vec && k0 + NBK <= p.n)  // uniform
                {
                    const float4 v = inRow ? *reinterpret_cast<const float4*>(col + 16 * q) : make_float4(0, 0, 0, 0);
                    t[4 * q] = v.x;
                    t[4 * q + 1] = v.y;
                    t[4 * q + 2] = v.z;
                    t[4 * q + 3] = v.w;
                }
                else
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        t[4 * q + e] = inRow && k0 + 16 * q + 4 * g + e < p.n ? col[16 * q + e] : 0.0f;
        }
        else
        {
            const float* const col = p.lu + static_cast<size_t>(k0) * p.lda + row;
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                {
                    const int k = 16 * q + 4 * g + e;
                    t[4 * q + e] = inRow && k0 + k < p.n ? col[static_cast<size_t>(k) * p.lda] : 0.0f;
                }
        }
    };
    auto multiply = [&](const float* s, const float (&t)[16], f32x4 (&acc)[CG])
    {
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < CG; ++c)
                    acc[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[(16 * q + 4 * g + e) * S + 16 * c + li],
                                                                  t[4 * q + e], acc[c], 0, 0, 0);
    };

    // Right-hand side: lane (li, g) holds row li of its wave, columns 16 c + 4 g + r.
    f32x4 rhs[CG];
    {
        int from = row;
        if (!SECOND && !TRANS && p.ipiv != nullptr && inRow) from = p.perm[row];
        const unsigned long long* const mine =
            p.pub + (static_cast<size_t>(ib) * strips + strip) * (64 * NS) + (16 * wave + li) * NS;
#pragma unroll
        for (int c = 0; c < CG; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const int col = 16 * c + 4 * g + r;
                float v = 0.0f;
                if (SECOND)
                    v = __uint_as_float(static_cast<unsigned>(mine[col]));
                else if (inRow && c0 + col < p.nrhs)
                    v = p.B[static_cast<size_t>(c0 + col) * p.ldb + from];
                rhs[c][r] = v;
            }
    }
    float cur[16], nxt[16];
    double iv[16];
    if (step > 0) loadTile(BACK ? nb - 1 : 0, cur);
    {
        const double* const in = p.inv + static_cast<size_t>(UPPER ? nb + ib : ib) * 4096 + (16 * wave + li) * 64 + 4 * g;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) iv[4 * q + e] = in[16 * q + e];
    }
    const int bad = p.bad[UPPER ? nb + ib : ib];
    bool failed = false;  // uniform over the workgroup
    for (int s = 0; s < step; ++s)
    {
        const int kb = BACK ? nb - 1 - s : s;
        if (s + 1 < step) loadTile(BACK ? kb - 1 : kb + 1, nxt);
        const unsigned long long* const words = p.pub + (static_cast<size_t>(kb) * strips + strip) * (64 * NS);
        unsigned long long w[PER];
        bool ok = false;
        const unsigned lim = failed ? 0u : p.spinLimit;
        for (unsigned spins = 0; spins < lim && !ok; ++spins)
        {
            // One word per lane until it is there, then all.
            w[0] = LoadWord(words + tid);
            ok = __all(static_cast<unsigned>(w[0] >> 32) == TAG);
            if (ok)
            {
#pragma unroll
                for (int i = 1; i < PER; ++i) w[i] = LoadWord(words + tid + 256 * i);
                bool all = true;
#pragma unroll
                for (int i = 1; i < PER; ++i) all = all && static_cast<unsigned>(w[i] >> 32) == TAG;
                ok = __all(all);
            }
            if (!ok) __builtin_amdgcn_s_sleep(1);
        }
        float* const x = s_x[s & 1];
#pragma unroll
        for (int i = 0; i < PER; ++i)
        {
            const int at = tid + 256 * i;
            x[(at / NS) * S + at % NS] = __uint_as_float(static_cast<unsigned>(w[i]));
        }
        if (!ok && lane == 0) s_fail = 1;
        __syncthreads();
        failed = s_fail != 0;
        // Each block's product is summed from zero and subtracted once: one long sum over the
        // row would round more.
        f32x4 acc[CG];
#pragma unroll
        for (int c = 0; c < CG; ++c) acc[c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        multiply(x, cur, acc);
#pragma unroll
        for (int c = 0; c < CG; ++c) rhs[c] = rhs[c] - acc[c];
#pragma unroll
        for (int e = 0; e < 16; ++e) cur[e] = nxt[e];
    }
    __syncthreads();
    float* const s_r = s_x[0];
    float* const s_y = s_x[1];
    f32x4 x0[CG];
#pragma unroll
    for (int c = 0; c < CG; ++c)
        *reinterpret_cast<f32x4*>(s_r + (16 * wave + li) * S + 16 * c + 4 * g) = rhs[c];
    __syncthreads();
    if (__builtin_expect(bad == 0, 1))  // uniform
    {
        // The FP64 matrix cores return row 4 r + g in element r: fed with the columns in the order
        // 4 (i mod 4) + i / 4, lane (li, g) gets columns 4 g + r as everywhere else.
        f64x4 wide[CG];
#pragma unroll
        for (int c = 0; c < CG; ++c) wide[c] = f64x4{0.0, 0.0, 0.0, 0.0};
        const int sig = 4 * (li & 3) + (li >> 2);
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < CG; ++c)
                    wide[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        static_cast<double>(s_r[(16 * q + 4 * g + e) * S + 16 * c + sig]), iv[4 * q + e], wide[c], 0, 0,
                        0);
#pragma unroll
        for (int c = 0; c < CG; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) x0[c][r] = static_cast<float>(wide[c][r]);
    }
    else
    {
        // A zero pivot, or an inverse that is too large: plain substitution, as LAPACK's. Lane: row,
        // NS / 4 columns a wave.
        constexpr int PC = NS / 4;
        const int64_t ld = p.lda;
        const float* const T = p.lu + r0 * ld + r0;
        float v[PC];
#pragma unroll
        for (int c = 0; c < PC; ++c) v[c] = s_r[lane * S + PC * wave + c];
        // Eight columns' entries at a time (their loads in flight together); those beyond the order
        // change nothing.
        const int last = p.n - 1 - r0;
#pragma unroll 1
        for (int e0 = 0; e0 < 64; e0 += 8)
        {
            float t[8], d[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                const int k = BACK ? 63 - e0 - e : e0 + e;
                const bool rest = (BACK ? lane < k : lane > k) && max(lane, k) <= last;
                t[e] = rest ? T[TRANS ? lane * ld + k : k * ld + lane] : 0.0f;
                d[e] = T[min(k, last) * ld + min(k, last)];
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                const int k = BACK ? 63 - e0 - e : e0 + e;
                const bool rest = (BACK ? lane < k : lane > k) && max(lane, k) <= last;
#pragma unroll
                for (int c = 0; c < PC; ++c)
                {
                    float x = ReadLane(v[c], k);
                    if (UPPER) x = x / d[e];
                    v[c] = rest ? fmaf(-t[e], x, v[c]) : (lane == k ? x : v[c]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < PC; ++c) s_y[lane * S + PC * wave + c] = v[c];
        __syncthreads();
#pragma unroll
        for (int c = 0; c < CG; ++c) x0[c] = *reinterpret_cast<const f32x4*>(s_y + (16 * wave + li) * S + 16 * c + 4 * g);
    }
    if (failed)
    {
#pragma unroll
        for (int c = 0; c < CG; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) x0[c][r] = __builtin_nanf("");
        if (tid == 0 && p.info != nullptr) *p.info = kInfoWaitTimeout;
    }
    unsigned long long* const words =
        p.pub + (static_cast<size_t>(ib) * strips + strip) * (64 * NS) + (16 * wave + li) * NS;
    int to = row;
    if (SECOND && TRANS && p.ipiv != nullptr && inRow) to = p.perm[row];
#pragma unroll
    for (int c = 0; c < CG; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int col = 16 * c + 4 * g + r;
            __hip_atomic_store(words + col,
                               (static_cast<unsigned long long>(TAG) << 32) | __float_as_uint(inRow ? x0[c][r] : 0.0f),
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    if (SECOND)
#pragma unroll
        for (int c = 0; c < CG; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                const int col = 16 * c + 4 * g + r;
                if (inRow && c0 + col < p.nrhs) p.B[static_cast<size_t>(c0 + col) * p.ldb + to] = x0[c][r];
            }
}

// 16 columns per strip for up to 32 right-hand sides, else 64.
int GroupsPerStrip(int nrhs) { return nrhs <= 32 ? 1 : 4; }

template <bool TRANS, int CG>
void Chains(const Trs& p, int nb, int strips, hipStream_t stream)
{
    hipLaunchKernelGGL((trs_chain_kernel<TRANS, false, CG>), dim3(nb * strips), dim3(256), 0, stream, p, nb, strips);
    hipLaunchKernelGGL((trs_chain_kernel<TRANS, true, CG>), dim3(nb * strips), dim3(256), 0, stream, p, nb, strips);
}

size_t Up(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }
size_t PublicationWords(int n, int nrhs)
{
    const int ns = 16 * GroupsPerStrip(nrhs);
    return static_cast<size_t>((n + NBK - 1) / NBK) * NBK * ((nrhs + ns - 1) / ns * ns);
}
}  // namespace

size_t TrsWorkspaceBytes(int n, int nrhs)
{
    const size_t nb = (n + NBK - 1) / NBK;
    return Up(2 * nb * 4096 * sizeof(double)) + Up(2 * nb * sizeof(int)) + Up(n * sizeof(int)) + 256 +
           Up(PublicationWords(n, nrhs) * 8) + 256;
}

hipError_t TrsSolve(int trans, int n, int nrhs, const float* lu, int lda, const int* ipiv, float* B, int ldb, int* info,
                    void* work, hipStream_t stream)
{
    if (n <= 0 || nrhs <= 0) return hipSuccess;
    if (n > kEngineMaxOrder) return hipErrorInvalidValue;
    const int nb = (n + NBK - 1) / NBK, cg = GroupsPerStrip(nrhs), strips = (nrhs + 16 * cg - 1) / (16 * cg);
    char* q = reinterpret_cast<char*>(Up(reinterpret_cast<uintptr_t>(work)));
    auto take = [&](size_t bytes) {
        char* const at = q;
        q += Up(bytes);
        return at;
    };
    Trs p{};
    p.trans = trans;
    p.n = n;
    p.nrhs = nrhs;
    p.lda = lda;
    p.ldb = ldb;
    p.lu = lu;
    p.ipiv = ipiv;
    p.B = B;
    p.info = info;
    p.inv = reinterpret_cast<double*>(take(static_cast<size_t>(2 * nb) * 4096 * sizeof(double)));
    p.bad = reinterpret_cast<int*>(take(static_cast<size_t>(2 * nb) * sizeof(int)));
    p.perm = reinterpret_cast<int*>(take(static_cast<size_t>(n) * sizeof(int)));
    p.ticket = reinterpret_cast<unsigned*>(take(256));
    const size_t words = PublicationWords(n, nrhs);
    p.pub = reinterpret_cast<unsigned long long*>(take(words * sizeof(unsigned long long)));
    p.spinLimit = SpinLimit();
    const int np = ipiv != nullptr ? (n + 255) / 256 : 0;
    const int nz = static_cast<int>(std::min<size_t>((words + 1023) / 1024, 1024));
    const size_t ldsBytes = std::max<size_t>(((2 * 64 + 32) * kInvStride + kGrowthScratch) * sizeof(double), ipiv ? ((n + 3) & ~3) * sizeof(int) : 0);
    hipLaunchKernelGGL(trs_prep_kernel, dim3(2 * nb + np + nz), dim3(256), ldsBytes, stream, p, nb, np, words);
    if (trans == 0)
        cg == 1 ? Chains<false, 1>(p, nb, strips, stream) : Chains<false, 4>(p, nb, strips, stream);
    else
        cg == 1 ? Chains<true, 1>(p, nb, strips, stream) : Chains<true, 4>(p, nb, strips, stream);
    return hipGetLastError();
}
}  // namespace ops
