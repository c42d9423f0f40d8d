// Device complex triangular solves from packed LU factors, gfx950: trs.hip's chains on pairs of
// real tiles. Reference semantics: src/cgetrs (row permutation, unit-lower and upper solves,
// trans N / T / C).
//
// One launch per triangle, a workgroup per 64 rows and 16 right-hand sides; FP32 products with
// the solved blocks, FP64 inverses of the diagonal blocks (or substitution where growth.h says so), blocks handed out by ticket in dependency order, solved rows published as
// tagged words. Bound by the chain: one device-wide
// trip, two products and a few barriers per 64 rows, 8 us a block and triangle (n = 8192, one
// right-hand side: 2.1 ms; 10.5 ms as two launches per block).
#include "ctrs.h"

#include <algorithm>
#include <cfloat>
#include <climits>

#include "complex_math.h"
#include "growth.h"
#include "internal.h"
#include "lanes.h"
#include "permute.h"
#include "trtri64.h"

namespace ops
{
namespace
{
constexpr int NBK = 64, NS = 16, S = NS + 4;
constexpr int kZ = 64 * kInvStride;   // doubles between the real and imaginary parts of a block
constexpr int kWords = 2 * 64 * NS;   // words of a published block: real parts, then imaginary

__device__ inline unsigned long long LoadWord(const unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

struct CTrs
{
    int trans, n, nrhs, lda, ldb;
    const float2* lu;
    const int* ipiv;
    float2* B;
    int* info;
    unsigned long long* pub;  // [block][strip][part][row][column]
    double* inv;              // inverses of the diagonal blocks of op(L), op(U): row-major, parts 4096 apart
    int* bad;                 // per diagonal block: its inverse is too large to be used (2 nb ints)
    int* perm;
    unsigned* ticket;         // [2]
    unsigned spinLimit;
};

// D = sign A B, 16 x K x 16, complex FP64 in LDS.
template <int K>
__device__ inline void ZProduct16(const double* a, const double* b, double* d, double sign, int lane)
{
    f64x4 re = {0.0, 0.0, 0.0, 0.0}, im = re;
    const int i = lane & 15, k0 = lane >> 4;
#pragma unroll
    for (int k = 0; k < K; k += 4)
    {
        const double ar = a[i * kInvStride + k + k0], ai = a[kZ + i * kInvStride + k + k0];
        const double br = b[(k + k0) * kInvStride + i], bi = b[kZ + (k + k0) * kInvStride + i];
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, br, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(ar, bi, im, 0, 0, 0);
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(-ai, bi, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(ai, br, im, 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        d[(4 * r + k0) * kInvStride + i] = sign * re[r];
        d[kZ + (4 * r + k0) * kInvStride + i] = sign * im[r];
    }
}

// trtri64.h's InvertLower64 for a complex block in place (parts kZ apart, zeros above the
// diagonal on entry); the intermediate product lies in the upper right quarter.
template <bool UNIT>
__device__ inline void ZInvertLower64(double* s, int tid)
{
    const int lane = tid & 63, wave = tid >> 6;
    double* const t = s + 32;
    if (wave == 0)
    {
        const int b = lane & 48;
        double2 x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            double2 v = make_double2(i == (lane & 15) ? 1.0 : 0.0, 0.0);
            const double* const row = s + (b + i) * kInvStride + b;
#pragma unroll
            for (int k = 0; k < i; ++k)
            {
                v.x = fma(row[kZ + k], x[k].y, fma(-row[k], x[k].x, v.x));
                v.y = fma(-row[kZ + k], x[k].x, fma(-row[k], x[k].y, v.y));
            }
            if (!UNIT)
            {
                const double dr = row[i], di = row[kZ + i], den = 1.0 / (dr * dr + di * di);
                v = make_double2((v.x * dr + v.y * di) * den, (v.y * dr - v.x * di) * den);
            }
            x[i] = v;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i)
        {
            s[(b + i) * kInvStride + lane] = x[i].x;
            s[kZ + (b + i) * kInvStride + lane] = x[i].y;
        }
    }
    __syncthreads();
    if (wave < 2)
        ZProduct16<16>(s + (32 * wave + 16) * kInvStride + 32 * wave, s + 32 * wave * kInvStride + 32 * wave,
                       t + 16 * wave * kInvStride, 1.0, lane);
    __syncthreads();
    if (wave < 2)
        ZProduct16<16>(s + (32 * wave + 16) * kInvStride + 32 * wave + 16, t + 16 * wave * kInvStride,
                       s + (32 * wave + 16) * kInvStride + 32 * wave, -1.0, lane);
    __syncthreads();
    const int qr = 16 * (wave >> 1), qc = 16 * (wave & 1);
    ZProduct16<32>(s + (32 + qr) * kInvStride, s + qc, t + qr * kInvStride + qc, 1.0, lane);
    __syncthreads();
    ZProduct16<32>(s + (32 + qr) * kInvStride + 32, t + qc, s + (32 + qr) * kInvStride + qc, -1.0, lane);
    __syncthreads();
}

// Preparation, by workgroup: 2 nb diagonal blocks inverted, the permutation (256 positions
// each), the publication words cleared.
__global__ __launch_bounds__(256) void ctrs_prep_kernel(CTrs p, int nb, int np, size_t words)
{
    extern __shared__ __align__(16) double s_mem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int b = blockIdx.x;
    if (b == 0 && tid == 0) p.ticket[0] = p.ticket[1] = 0u;
    if (b < 2 * nb)
    {
        const bool upper = b >= nb;
        const int k0 = (upper ? b - nb : b) * NBK, kb = min(NBK, p.n - k0);
        const float2* const T = p.lu + static_cast<size_t>(k0) * p.lda + k0;
        double* const s_g = s_mem + 2 * kZ;
        // Lower: the block; upper: its transpose. Rows beyond the block are the identity.
        float part = 0.0f;
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            const int c = wave * 16 + k;
            float2 v = lane < kb && c < kb ? T[static_cast<size_t>(c) * p.lda + lane] : make_float2(0.0f, 0.0f);
            if (lane == c && (!upper || lane >= kb)) v = make_float2(1.0f, 0.0f);
            if (upper ? lane > c : lane < c) v = make_float2(0.0f, 0.0f);
            const int at = upper ? c * kInvStride + lane : lane * kInvStride + c;
            s_mem[at] = v.x;
            s_mem[kZ + at] = v.y;
            part = fmaxf(part, fabsf(v.x) + fabsf(v.y));
        }
        // The maxima (|re| + |im|) of op(T)'s rows: T's own from the registers, its columns from LDS
        // (before the inversion, which works in place).
        const bool flip = upper != (p.trans != 0);
        const int step = flip ? kInvStride : 1, first = flip ? lane : lane * kInvStride;
        if (p.trans != 0)  // uniform
        {
            __syncthreads();
            part = 0.0f;
#pragma unroll
            for (int k = 0; k < 16; ++k)
            {
                const int at = first + (16 * wave + k) * step;
                part = fmaxf(part, static_cast<float>(fabs(s_mem[at]) + fabs(s_mem[kZ + at])));
            }
        }
        s_g[tid] = part;
        __syncthreads();
        if (wave == 3)
            RowMaxima(s_g)[lane] = fmax(fmax(s_g[lane], s_g[64 + lane]), fmax(s_g[128 + lane], s_g[192 + lane]));
        if (upper)
            ZInvertLower64<false>(s_mem, tid);
        else
            ZInvertLower64<true>(s_mem, tid);
        // Row-major inverse of op(T): L^-1 and (U^T)^-1 as they are, the other two transposed.
        double* const out = p.inv + static_cast<size_t>(b) * 8192;
        const double d = RowMaxima(s_g)[lane];
        bool fine = true, small = true;
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            const int r = wave * 16 + k;
            const int at = flip ? lane * kInvStride + r : r * kInvStride + lane;
            const bool in = flip ? lane >= r : r >= lane;
            const double x = in ? s_mem[at] : 0.0, y = in ? s_mem[kZ + at] : 0.0;
            fine = fine && fabs(x) <= FLT_MAX && fabs(y) <= FLT_MAX;
            small = small && (fabs(x) + fabs(y)) * d <= kSmallInverse;
            out[r * 64 + lane] = x;
            out[4096 + r * 64 + lane] = p.trans == 2 ? -y : y;
        }
        if (!__syncthreads_and(fine && small))
        {
            float e[16];  // op(T) by rows, again from memory
#pragma unroll
            for (int k = 0; k < 16; ++k)
            {
                const int r = p.trans ? wave * 16 + k : lane, c = p.trans ? lane : wave * 16 + k;
                const bool in = r < kb && c < kb && (upper ? r <= c : r > c);
                const float2 v = in ? T[static_cast<size_t>(c) * p.lda + r] : make_float2(0.0f, 0.0f);
                e[k] = r == c && (!upper || r >= kb) ? 1.0f : fabsf(v.x) + fabsf(v.y);
            }
            auto size = [&](int j)
            {
                const int at = first + j * step;
                return (flip ? j >= lane : lane >= j) ? fabs(s_mem[at]) + fabs(s_mem[kZ + at]) : 0.0;
            };
            const double grow = Growth64(e, size, s_g, tid);
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
        for (int k = tid; k < p.n; k += 256)
        {
            const int v = p.ipiv[k] - 1;
            s_piv[k] = v < k || v >= p.n ? k : v;
        }
        __syncthreads();
        const int x = TracePosition(s_piv, p.n, i, b * 256 + wave * 64, true);
        if (i < p.n) p.perm[i] = x;
        return;
    }
    b -= np;
    const size_t step = static_cast<size_t>(gridDim.x - 2 * nb - np) * 256;
    for (size_t w = static_cast<size_t>(b) * 256 + tid; w < words; w += step) p.pub[w] = 0ull;
}

// As trs_chain_kernel with one column group; TRANS: the tiles are read transposed (and
// conjugated for trans 2).
template <bool TRANS, bool SECOND>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void ctrs_chain_kernel(CTrs p, int nb, int strips)
{
    constexpr bool UPPER = TRANS != SECOND;  // N: L then U; T, C: op(U) then op(L)
    constexpr bool BACK = SECOND;            // both second substitutions run upward
    constexpr int PER = kWords / 256;
    constexpr unsigned TAG = SECOND ? 2u : 1u;
    __shared__ __align__(16) float s_x[2][2 * 64 * S];  // real parts, imaginary parts
    __shared__ unsigned s_id;
    __shared__ int s_fail;  // a wait of this workgroup ran out
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
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
    const float conj = TRANS && p.trans == 2 ? -1.0f : 1.0f;

    // Rows beyond the order repeat the last one (they are not used).
    auto loadTile = [&](int kb, float2 (&t)[16])
    {
        const int k0 = kb * NBK + 4 * g, last = p.n - 1;
        const int64_t ld = p.lda;
        const float2* const at = p.lu + (TRANS ? min(row, last) * ld : static_cast<int64_t>(min(row, last)));
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const int k = min(k0 + 16 * q + e, last);
                t[4 * q + e] = at[TRANS ? static_cast<int64_t>(k) : k * ld];
            }
        if (kb * NBK + NBK > p.n)  // uniform: no product of a zero row with an infinity
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (k0 + 16 * q + e > last) t[4 * q + e] = make_float2(0.0f, 0.0f);
    };
    const size_t base = (static_cast<size_t>(ib) * strips + strip) * kWords;

    // Right-hand side: lane (li, g) holds row li of its wave, columns 4 g + r.
    f32x4 rr, ri;
    {
        int from = row;
        if (!SECOND && !TRANS && p.ipiv != nullptr && inRow) from = p.perm[row];
        const unsigned long long* const mine = p.pub + base + (16 * wave + li) * NS;
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int col = 4 * g + r;
            float2 v = make_float2(0.0f, 0.0f);
            if (SECOND)
                v = make_float2(__uint_as_float(static_cast<unsigned>(mine[col])),
                                __uint_as_float(static_cast<unsigned>(mine[64 * NS + col])));
            else if (inRow && c0 + col < p.nrhs)
                v = p.B[static_cast<size_t>(c0 + col) * p.ldb + from];
            rr[r] = v.x;
            ri[r] = v.y;
        }
    }
    float2 cur[16], nxt[16];
    if (step > 0) loadTile(BACK ? nb - 1 : 0, cur);
    const int bad = p.bad[UPPER ? nb + ib : ib];
    bool failed = false;  // uniform over the workgroup
    for (int s = 0; s < step; ++s)
    {
        const int kb = BACK ? nb - 1 - s : s;
        if (s + 1 < step) loadTile(BACK ? kb - 1 : kb + 1, nxt);
        const unsigned long long* const words = p.pub + (static_cast<size_t>(kb) * strips + strip) * kWords;
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
        f32x4 ar = {0.0f, 0.0f, 0.0f, 0.0f}, ai = ar;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const int at = (16 * q + 4 * g + e) * S + li;
                const float xr = x[at], xi = x[64 * S + at], ty = conj * cur[4 * q + e].y;
                ar = __builtin_amdgcn_mfma_f32_16x16x4f32(xr, cur[4 * q + e].x, ar, 0, 0, 0);
                ai = __builtin_amdgcn_mfma_f32_16x16x4f32(xi, cur[4 * q + e].x, ai, 0, 0, 0);
                ar = __builtin_amdgcn_mfma_f32_16x16x4f32(-xi, ty, ar, 0, 0, 0);
                ai = __builtin_amdgcn_mfma_f32_16x16x4f32(xr, ty, ai, 0, 0, 0);
            }
        rr = rr - ar;
        ri = ri - ai;
#pragma unroll
        for (int e = 0; e < 16; ++e) cur[e] = nxt[e];
    }
    __syncthreads();
    float* const s_r = s_x[0];
    float* const s_y = s_x[1];
    {
        const int at = (16 * wave + li) * S + 4 * g;
        *reinterpret_cast<f32x4*>(s_r + at) = inRow ? rr : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        *reinterpret_cast<f32x4*>(s_r + 64 * S + at) = inRow ? ri : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    // The inverse's rows: asked for here, under the barrier; kept from the start of the chain
    // they would cost 64 registers.
    const double* const in = p.inv + static_cast<size_t>(UPPER ? nb + ib : ib) * 8192 + (16 * wave + li) * 64 + 4 * g;
    f32x4 x0, y0;
    __syncthreads();
    if (__builtin_expect(bad == 0, 1))  // uniform
    {
        // The FP64 matrix cores return row 4 r + g in element r: fed with the columns in the order
        // 4 (i mod 4) + i / 4, lane (li, g) gets columns 4 g + r as everywhere else.
        f64x4 re = {0.0, 0.0, 0.0, 0.0}, im = re;
        const int sig = 4 * (li & 3) + (li >> 2);
#pragma unroll
        for (int q = 0; q < 4; ++q)
        {
            if (BACK ? q < wave : q > wave) continue;  // uniform: zeros of the triangle
#pragma unroll
            for (int e = 0; e < 4; ++e)
            {
                const double lr = in[16 * q + e], lx = in[4096 + 16 * q + e];
                const int at = (16 * q + 4 * g + e) * S + sig;
                const double br = s_r[at], bi = s_r[64 * S + at];
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(br, lr, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(bi, lr, im, 0, 0, 0);
                re = __builtin_amdgcn_mfma_f64_16x16x4f64(-bi, lx, re, 0, 0, 0);
                im = __builtin_amdgcn_mfma_f64_16x16x4f64(br, lx, im, 0, 0, 0);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            x0[r] = static_cast<float>(re[r]);
            y0[r] = static_cast<float>(im[r]);
        }
    }
    else
    {
        // A zero pivot, or an inverse that is too large: plain substitution, as LAPACK's. Lane: row,
        // four columns a wave.
        const int64_t ld = p.lda;
        const float2* const T = p.lu + r0 * ld + r0;
        float2 v[NS / 4];
#pragma unroll
        for (int c = 0; c < NS / 4; ++c)
        {
            const int at = lane * S + NS / 4 * wave + c;
            v[c] = make_float2(s_r[at], s_r[64 * S + at]);
        }
        // Eight columns' entries at a time, as in trs.hip.
        const int last = p.n - 1 - r0;
#pragma unroll 1
        for (int e0 = 0; e0 < 64; e0 += 8)
        {
            float2 t[8], d[8];
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                const int k = BACK ? 63 - e0 - e : e0 + e;
                const bool rest = (BACK ? lane < k : lane > k) && max(lane, k) <= last;
                t[e] = rest ? T[TRANS ? lane * ld + k : k * ld + lane] : make_float2(0.0f, 0.0f);
                d[e] = T[min(k, last) * ld + min(k, last)];
                t[e].y *= conj;
                d[e].y *= conj;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e)
            {
                const int k = BACK ? 63 - e0 - e : e0 + e;
                const bool rest = (BACK ? lane < k : lane > k) && max(lane, k) <= last;
                const double2 r = Recip64(d[e]);
#pragma unroll
                for (int c = 0; c < NS / 4; ++c)
                {
                    float2 x = make_float2(ReadLane(v[c].x, k), ReadLane(v[c].y, k));
                    if (UPPER) x = Mul64(x, r);
                    const float2 y = SubMul(v[c], t[e], x);
                    v[c] = rest ? y : (lane == k ? x : v[c]);
                }
            }
        }
#pragma unroll
        for (int c = 0; c < NS / 4; ++c)
        {
            const int at = lane * S + NS / 4 * wave + c;
            s_y[at] = v[c].x;
            s_y[64 * S + at] = v[c].y;
        }
        __syncthreads();
        x0 = *reinterpret_cast<const f32x4*>(s_y + (16 * wave + li) * S + 4 * g);
        y0 = *reinterpret_cast<const f32x4*>(s_y + 64 * S + (16 * wave + li) * S + 4 * g);
    }
    if (failed)
    {
#pragma unroll
        for (int r = 0; r < 4; ++r) x0[r] = y0[r] = __builtin_nanf("");
        if (tid == 0 && p.info != nullptr) *p.info = kInfoWaitTimeout;
    }
    unsigned long long* const words = p.pub + base + (16 * wave + li) * NS;
    int to = row;
    if (SECOND && TRANS && p.ipiv != nullptr && inRow) to = p.perm[row];
#pragma unroll
    for (int r = 0; r < 4; ++r)
    {
        const unsigned long long tag = static_cast<unsigned long long>(TAG) << 32;
        __hip_atomic_store(words + 4 * g + r, tag | __float_as_uint(inRow ? x0[r] : 0.0f), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(words + 64 * NS + 4 * g + r, tag | __float_as_uint(inRow ? y0[r] : 0.0f), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    }
    if (SECOND)
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const int col = 4 * g + r;
            if (inRow && c0 + col < p.nrhs)
                p.B[static_cast<size_t>(c0 + col) * p.ldb + to] = make_float2(x0[r], y0[r]);
        }
}

template <bool TRANS>
void CChains(const CTrs& p, int nb, int strips, hipStream_t stream)
{
    hipLaunchKernelGGL((ctrs_chain_kernel<TRANS, false>), dim3(nb * strips), dim3(256), 0, stream, p, nb, strips);
    hipLaunchKernelGGL((ctrs_chain_kernel<TRANS, true>), dim3(nb * strips), dim3(256), 0, stream, p, nb, strips);
}

size_t Up(size_t b) { return (b + 255) & ~static_cast<size_t>(255); }
size_t PublicationWords(int n, int nrhs)
{
    return static_cast<size_t>((n + NBK - 1) / NBK) * ((nrhs + NS - 1) / NS) * kWords;
}
}  // namespace

size_t CTrsWorkspaceBytes(int n, int nrhs)
{
    const size_t nb = (n + NBK - 1) / NBK;
    return Up(2 * nb * 8192 * sizeof(double)) + Up(2 * nb * sizeof(int)) + Up(n * sizeof(int)) + 256 +
           Up(PublicationWords(n, nrhs) * 8) + 256;
}

hipError_t CTrsSolve(int trans, int n, int nrhs, const float2* lu, int lda, const int* ipiv, float2* B, int ldb,
                     int* info, void* work, hipStream_t stream)
{
    if (n <= 0 || nrhs <= 0) return hipSuccess;
    if (n > 16384 || nrhs > kCTrsMaxRhs) return hipErrorInvalidValue;
    const int nb = (n + NBK - 1) / NBK, strips = (nrhs + NS - 1) / NS;
    char* q = reinterpret_cast<char*>(Up(reinterpret_cast<uintptr_t>(work)));
    auto take = [&](size_t bytes) {
        char* const at = q;
        q += Up(bytes);
        return at;
    };
    CTrs p{};
    p.trans = trans;
    p.n = n;
    p.nrhs = nrhs;
    p.lda = lda;
    p.ldb = ldb;
    p.lu = lu;
    p.ipiv = ipiv;
    p.B = B;
    p.info = info;
    p.inv = reinterpret_cast<double*>(take(static_cast<size_t>(2 * nb) * 8192 * sizeof(double)));
    p.bad = reinterpret_cast<int*>(take(static_cast<size_t>(2 * nb) * sizeof(int)));
    p.perm = reinterpret_cast<int*>(take(static_cast<size_t>(n) * sizeof(int)));
    p.ticket = reinterpret_cast<unsigned*>(take(256));
    const size_t words = PublicationWords(n, nrhs);
    p.pub = reinterpret_cast<unsigned long long*>(take(words * 8));
    p.spinLimit = SpinLimit();
    const int np = ipiv != nullptr ? (n + 255) / 256 : 0;
    const int nz = static_cast<int>(std::min<size_t>((words + 1023) / 1024, 1024));
    const size_t ldsBytes = std::max<size_t>((2 * kZ + kGrowthScratch) * sizeof(double), ipiv ? ((n + 3) & ~3) * sizeof(int) : 0);
    hipLaunchKernelGGL(ctrs_prep_kernel, dim3(2 * nb + np + nz), dim3(256), ldsBytes, stream, p, nb, np, words);
    if (trans == 0)
        CChains<false>(p, nb, strips, stream);
    else
        CChains<true>(p, nb, strips, stream);
    return hipGetLastError();
}
}  // namespace ops
