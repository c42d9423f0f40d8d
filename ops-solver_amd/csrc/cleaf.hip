// Panel leaves of the complex LU and the launches that follow them, gfx950: the design of
// leaf.hip on pairs of real tiles. Reference semantics: src/cgetrf/cgetrf_kernel.cpp:376-411
// (largest L1 pivot score, lowest row on ties; accurate quotients; fused updates).
//
// Rows live in MFMA accumulator layout, real and imaginary tiles apart; the eight-column block
// being factored is held one row per lane; the columns to its right receive its eight pivots as
// a rank-8 update of four real products. Bound by a serial chain per column (score, exchange, one
// FP64 reciprocal) of some 290 instructions a wave in one workgroup and twice that for the wave
// that exchanges with other workgroups. 64 columns, the unrolled leaves of 32 or 16 columns before
// and this one: 8192 rows 281 and 130 us, 2048 to 513 rows 237 and 115 us, 512 rows 82 us, 256
// rows 60 us, 64 rows 47 us.
#include "cleaf.h"

#include <algorithm>
#include <climits>

#include "complex_math.h"
#include "internal.h"
#include "lanes.h"
#include "unitlower.h"
#include "wave.h"

namespace ops
{
namespace
{
typedef float f32x16 __attribute__((ext_vector_type(16)));

__device__ inline unsigned long long LoadWord(const unsigned long long* p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// local (uniform): the readers share the writer's XCD; the word stays in that XCD's L2.
__device__ inline void StoreWord(unsigned long long* p, unsigned long long v, bool local)
{
    if (local)
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    else
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline void StoreTagged(unsigned long long* p, unsigned tag, float v, bool local)
{
    StoreWord(p, (static_cast<unsigned long long>(tag) << 32) | __float_as_uint(v), local);
}

template <int NW>
__device__ inline unsigned CyclicMaxU32(unsigned v)
{
    auto mx = [](unsigned a, unsigned b) { return a > b ? a : b; };
    if (NW >= 2) v = mx(v, DppU32<0xB1>(v));
    if (NW >= 4) v = mx(v, DppU32<0x4E>(v));
    if (NW >= 8) v = mx(v, DppU32<0x124>(v));
    return v;
}

// NW waves of 64 rows per workgroup, up to 64 columns. MULTI: the rows are spread over up to
// kCLeafMaxGroups workgroups. Per column each publishes a key (16-bit tag, 32-bit score class,
// 14-bit rank of the position) and its candidate's values of the block as tagged words; one wave
// per workgroup polls the keys and all values together and takes the winner's (one trip to L2:
// the values after the keys would be a second). After a block
// the owners publish its pivot rows. An arrival gate, bounded waits, NaN rows after a timeout
// and SPREAD (participants on one XCD) are as in leaf.hip.
template <int NW, bool MULTI, bool SPREAD>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(MULTI && !SPREAD && NW == 4 ? 1 : 2))) void cpanel_leaf_kernel(CLeafArgs p)
{
    __builtin_amdgcn_s_setprio(3);  // before the trailing product's waves on the same SIMD
    constexpr int T = 64 * NW, W = kCLeafWidth;
    constexpr int US = W + 28;
    __shared__ uint2 s_key[2][NW];
    __shared__ __align__(16) float2 s_val[2][NW * 8];
    __shared__ __align__(16) float s_ur[8][US], s_ui[8][US];
    __shared__ __align__(16) float2 s_l[8][8];
    __shared__ float s_win[2][32];
    __shared__ int s_gave;  // a wait of this workgroup ran out

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (SPREAD && (blockIdx.x & 7) != 0) return;  // not a participant
    const int P = MULTI ? static_cast<int>(SPREAD ? gridDim.x >> 3 : gridDim.x) : 1;
    const int g = MULTI ? static_cast<int>(SPREAD ? blockIdx.x >> 3 : blockIdx.x) : 0;
    const int c0 = p.c0, mp = p.m - c0, wact = p.wact;
    const int64_t lda = p.lda;
    float2* const Ap = p.A + static_cast<int64_t>(c0) * lda + c0;
    const int lr = g * T + wid * 64 + lane;
    const bool valid = lr < mp;
    bool aborted = false;  // uniform over the workgroup

    f32x16 curR[2], curI[2], nxtR[2], nxtI[2];
    int srcv = 0;
    {
        const float2* src = Ap + lr;
        // In two halves: the loads of 32 columns in flight are enough, and 64 would not leave the
        // registers for the accumulators.
#pragma unroll
        for (int h = 0; h < 2; ++h)
        {
            float2 x[32];
#pragma unroll
            for (int c = 0; c < 32; ++c) x[c] = make_float2(0.0f, 0.0f);
            if (valid)
#pragma unroll
                for (int c = 0; c < 32; ++c)
                {
                    x[c] = *src;
                    src += 32 * h + c + 1 < wact ? lda : 0;
                }
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    SwapHalves(x[8 * k + r].x, x[8 * k + 4 + r].x);
                    SwapHalves(x[8 * k + r].y, x[8 * k + 4 + r].y);
                    (h == 0 ? curR : nxtR)[0][4 * k + r] = x[8 * k + r].x;
                    (h == 0 ? curI : nxtI)[0][4 * k + r] = x[8 * k + r].y;
                    (h == 0 ? curR : nxtR)[1][4 * k + r] = x[8 * k + 4 + r].x;
                    (h == 0 ? curI : nxtI)[1][4 * k + r] = x[8 * k + 4 + r].y;
                }
        }
        if (valid) srcv = p.newPanel ? c0 + lr : p.rowsrc[c0 + lr];
    }
    int pos = valid ? lr : -1;
    if constexpr (MULTI)
    {
        // No column is exchanged before every workgroup is resident and has its rows (leaf.hip).
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        unsigned long long* const arrival = p.slots + kCLeafArrivalWord;
        if (tid == 0) StoreWord(arrival + g, p.tagBase, SPREAD);
        if (wid == 0)
        {
            // After a wait that ran out, here or in an earlier leaf: no more waits (leaf.hip).
            const bool late = __any(__hip_atomic_load(p.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0);
            bool all = false;
            for (unsigned spins = 0; spins < p.spinLimit && !late; ++spins)
            {
                all = __all(lane >= P || LoadWord(arrival + lane) == p.tagBase);
                if (all) break;
                __builtin_amdgcn_s_sleep(16);
            }
            if (lane == 0)
            {
                s_gave = all ? 0 : 1;
                if (!all) __hip_atomic_store(p.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        __syncthreads();
        aborted = s_gave != 0;
    }
    int zeroCol = 0;
    int pivots = 0;  // lane j: the pivot's position in column j
    const unsigned span = p.pivoting ? 0x3fffffffu : 0u;

    for (int q = 0; 8 * q < wact; ++q)
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
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 12; ++e)
            {
                curR[t][e] = curR[t][e + 4];
                curI[t][e] = curI[t][e + 4];
            }
#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
        {
            const int j = 8 * q + jj;
            if (j >= wact) break;  // uniform
            const int par = jj & 1;
            // Score class of the lane's row: 0 none, else PivotScore + 1 (NaN ranks lowest; the
            // score of a finite sum is its bits + 1).
            const bool cand = static_cast<unsigned>(pos - j) <= span;
            unsigned bh = __float_as_uint(fabsf(v[jj].x) + fabsf(v[jj].y)) + 2u;
            if (__builtin_expect(__any(cand && bh > 0x7f800001u), 0)) bh = PivotScore(v[jj]) + 1u;
            bh = cand ? bh : 0u;
            unsigned top = WaveMaxU32(bh);
            unsigned long long tie = __ballot(bh == top);
            if (__builtin_expect(__popcll(tie) != 1, 0))  // uniform
            {
                const unsigned low = WaveMaxU32(bh == top ? ~static_cast<unsigned>(pos) : 0u);
                tie = __ballot(bh == top && ~static_cast<unsigned>(pos) == low);
            }
            int wl = __builtin_ctzll(tie);
            int pp;
            float2 d, u[8];
            float2 x0 = make_float2(0.0f, 0.0f);
            if constexpr (NW == 1)
            {
                pp = __builtin_amdgcn_readlane(pos, wl);
                d = make_float2(ReadLane(v[jj].x, wl), ReadLane(v[jj].y, wl));
#pragma unroll
                for (int c = jj + 1; c < 8; ++c) u[c] = make_float2(ReadLane(v[c].x, wl), ReadLane(v[c].y, wl));
            }
            else
            {
                if (lane == wl)
                {
                    s_key[par][wid] = make_uint2(top, static_cast<unsigned>(pos));
                    s_val[par][wid * 8] = v[jj];
#pragma unroll
                    for (int c = jj + 1; c < 8; ++c) s_val[par][wid * 8 + c] = v[c];
                }
                __syncthreads();
                const uint2 k = s_key[par][lane & (NW - 1)];
                x0 = s_val[par][lane & (NW * 8 - 1)];
                const unsigned t = CyclicMaxU32<NW>(k.x);
                top = __builtin_amdgcn_readfirstlane(t);
                unsigned hit = static_cast<unsigned>(__ballot(k.x == top)) & ((1u << NW) - 1u);
                if (__builtin_expect(__popc(hit) != 1, 0))  // uniform
                {
                    const unsigned low = CyclicMaxU32<NW>(k.x == top ? ~k.y : 0u);
                    hit = static_cast<unsigned>(__ballot(k.x == top && ~k.y == low)) & ((1u << NW) - 1u);
                }
                wl = __builtin_ctz(hit | 0x80000000u) & (NW - 1);
                pp = static_cast<int>(__builtin_amdgcn_readlane(k.y, wl));
                if constexpr (!MULTI)
                {
                    d = make_float2(ReadLane(x0.x, wl * 8), ReadLane(x0.y, wl * 8));
#pragma unroll
                    for (int c = jj + 1; c < 8; ++c)
                        u[c] = make_float2(ReadLane(x0.x, wl * 8 + c), ReadLane(x0.y, wl * 8 + c));
                }
            }
            if constexpr (MULTI)
            {
                static_assert(!MULTI || NW > 1, "the winner's values sit in eight lanes");
                const unsigned tag = p.tagBase + static_cast<unsigned>(j);
                unsigned long long* const keys = p.slots + (j & 1) * kCLeafMaxGroups;
                unsigned long long* const vals = p.slots + kCLeafValueWord + (j & 1) * (16 * kCLeafMaxGroups);
                if (wid == 0)  // uniform
                {
                    const int c = lane & 7;
                    if ((lane >> 3) == wl && (c == 0 || c > jj))
                    {
                        StoreTagged(vals + g * 16 + 2 * c, tag, x0.x, SPREAD);
                        StoreTagged(vals + g * 16 + 2 * c + 1, tag, x0.y, SPREAD);
                    }
                    if (lane == 0)
                        StoreWord(keys + g,
                                  (static_cast<unsigned long long>(tag & 0xffffu) << 48) |
                                      (top == 0u ? 0ull
                                                 : (static_cast<unsigned long long>(top) << 16) |
                                                       static_cast<unsigned>(0x3fff - pp)),
                                  SPREAD);
                    unsigned hi = 0u, lo = 0u, x = 0u;
                    int gw = 0;
                    bool got = false;
                    const bool mine = lane < P;
                    const int c2 = lane & 15;
                    const bool need = c2 < 2 || c2 > 2 * jj + 1;
                    const unsigned lim = aborted ? 0u : p.spinLimit;
                    for (unsigned spins = 0; spins < lim; ++spins)
                    {
                        unsigned long long w0 = static_cast<unsigned long long>(tag & 0xffffu) << 48, w[8];
                        if (mine) w0 = LoadWord(keys + lane);
#pragma unroll
                        for (int r = 0; r < 8; ++r)
                        {
                            w[r] = 0ull;
                            if (4 * r < P) w[r] = LoadWord(vals + 64 * r + lane);  // uniform
                        }
                        hi = static_cast<unsigned>(w0 >> 16);
                        lo = static_cast<unsigned>(w0) & 0x3fffu;
                        if (__all(static_cast<unsigned>(w0 >> 48) == (tag & 0xffffu)))
                        {
                            top = WaveMaxU32(hi);
                            tie = __ballot(hi == top && mine);
                            if (__builtin_expect(__popcll(tie) != 1, 0))  // uniform
                            {
                                const unsigned low = WaveMaxU32(hi == top && mine ? lo : 0u);
                                tie = __ballot(hi == top && mine && lo == low);
                            }
                            gw = __builtin_ctzll(tie | (1ull << 63)) & (kCLeafMaxGroups - 1);
                            unsigned long long xw = w[0];
#pragma unroll
                            for (int r = 1; r < 8; ++r) xw = (gw >> 2) == r ? w[r] : xw;  // uniform
                            x = static_cast<unsigned>(xw);
                            got = __all((lane >> 4) != (gw & 3) || !need || static_cast<unsigned>(xw >> 32) == tag);
                            if (got) break;
                        }
                        __builtin_amdgcn_s_sleep(1);
                    }
                    const unsigned ls = __builtin_amdgcn_readlane(lo, gw);
                    if (!got)
                    {
                        top = 0u;
                        if (lane == 0)
                        {
                            s_gave = 1;
                            __hip_atomic_store(p.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
                    }
                    if ((lane >> 4) == (gw & 3)) s_win[par][c2] = __uint_as_float(x);
                    if (lane == 0)
                    {
                        s_win[par][16] = __uint_as_float(top);
                        s_win[par][17] = __uint_as_float(ls);
                    }
                }
                __syncthreads();
                const float x = s_win[par][lane & 31];
                aborted = s_gave != 0;
                top = __builtin_amdgcn_readlane(__float_as_uint(x), 16);
                pp = 0x3fff - static_cast<int>(__builtin_amdgcn_readlane(__float_as_uint(x), 17));
                d = make_float2(ReadLane(x, 0), ReadLane(x, 1));
#pragma unroll
                for (int c = jj + 1; c < 8; ++c) u[c] = make_float2(ReadLane(x, 2 * c), ReadLane(x, 2 * c + 1));
            }
            const bool none = top == 0u || (MULTI && aborted);  // uniform
            const int bpos = none ? j : pp;
            pos = pos == bpos ? j : (pos == j ? bpos : pos);
            pivots = lane == j ? bpos : pivots;
            const bool zero = none || (d.x == 0.0f && d.y == 0.0f);  // uniform
            if (zero && zeroCol == 0 && !(MULTI && aborted)) zeroCol = j + 1;
            const double2 rinv = Recip64(zero ? make_float2(1.0f, 0.0f) : d);
            const bool below = pos > (zero ? INT_MAX : j);
            const float2 qv = Mul64(v[jj], rinv);
            const float2 l = below ? qv : make_float2(0.0f, 0.0f);
            lm[jj] = l;
            v[jj] = below ? qv : v[jj];
#pragma unroll
            for (int c = jj + 1; c < 8; ++c) v[c] = SubMul(v[c], l, u[c]);
        }

        {
            float2* dst = Ap + static_cast<int64_t>(8 * q) * lda + lr;
            if (valid)
#pragma unroll
                for (int c = 0; c < 8; ++c)
                {
                    if (8 * q + c < wact) *dst = v[c];  // uniform
                    dst += lda;
                }
        }
        const int live = 8 * (q + 1);  // first column that still lacks this block
        if (live >= wact) break;       // uniform

        {
            const int rel = pos - 8 * q;
            int slot0 = static_cast<unsigned>(rel) < 8u ? rel : -1;
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
                    // Stale groups of cur go to columns that nxt's groups, stored after them, or
                    // nothing at all owns.
                    const int at = 4 * (lane >> 5);
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                    {
                        *reinterpret_cast<float4*>(&s_ur[slot][at + live + 8 * k]) =
                            make_float4(curR[t][4 * k], curR[t][4 * k + 1], curR[t][4 * k + 2], curR[t][4 * k + 3]);
                        *reinterpret_cast<float4*>(&s_ui[slot][at + live + 8 * k]) =
                            make_float4(curI[t][4 * k], curI[t][4 * k + 1], curI[t][4 * k + 2], curI[t][4 * k + 3]);
                    }
                    if (q < 4)  // uniform
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                        {
                            *reinterpret_cast<float4*>(&s_ur[slot][at + 32 + 8 * k]) =
                                make_float4(nxtR[t][4 * k], nxtR[t][4 * k + 1], nxtR[t][4 * k + 2], nxtR[t][4 * k + 3]);
                            *reinterpret_cast<float4*>(&s_ui[slot][at + 32 + 8 * k]) =
                                make_float4(nxtI[t][4 * k], nxtI[t][4 * k + 1], nxtI[t][4 * k + 2], nxtI[t][4 * k + 3]);
                        }
                }
            }
        }
        if constexpr (MULTI)
        {
            // Row words: 64 real parts, 64 imaginary parts, then the eight multipliers.
            constexpr int RW = kCLeafRowStride;
            auto at = [&](int slot, int cc) -> float*
            {
                return cc < W ? &s_ur[slot][cc]
                              : cc < 2 * W ? &s_ui[slot][cc - W] : reinterpret_cast<float*>(&s_l[slot][0]) + (cc - 2 * W);
            };
            unsigned long long* const rows = p.slots + kCLeafRowWord + (q & 1) * (8 * kCLeafRowStride);
            const unsigned tag = p.tagBase + static_cast<unsigned>(8 * q);
            // Opaque here: addresses hoisted out of the block loop would not fit the registers.
            int wl = lane, wt = tid;
            asm volatile("" : "+v"(wl), "+v"(wt));
            const int rel = pos - 8 * q;
            unsigned long long own = __ballot(static_cast<unsigned>(rel) < 8u);
            while (own != 0ull)  // uniform
            {
                const int from = __builtin_ctzll(own);
                own &= own - 1ull;
                const int slot = __builtin_amdgcn_readlane(rel, from);
#pragma unroll
                for (int i = 0; i < (RW + 63) / 64; ++i)
                {
                    const int cc = wl + 64 * i;
                    if (cc < RW) StoreTagged(rows + slot * RW + cc, tag, *at(slot, cc), SPREAD);
                }
            }
            constexpr int PER = (8 * RW + T - 1) / T;
            unsigned long long w[PER];
            bool ok = false;
            const unsigned lim = aborted ? 0u : p.spinLimit;
            for (unsigned spins = 0; spins < lim; ++spins)
            {
                bool good = true;
#pragma unroll
                for (int i = 0; i < PER; ++i)
                {
                    const int idx = wt + i * T;
                    w[i] = idx < 8 * RW ? LoadWord(rows + idx) : static_cast<unsigned long long>(tag) << 32;
                    good = good && static_cast<unsigned>(w[i] >> 32) == tag;
                }
                if (__all(good))
                {
                    ok = true;
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (!ok)
            {
                if (lane == 0)
                {
                    s_gave = 1;
                    __hip_atomic_store(p.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            else
#pragma unroll
                for (int i = 0; i < PER; ++i)
                {
                    const int idx = wt + i * T, slot = idx / RW, cc = idx - slot * RW;
                    if (idx < 8 * RW) *at(slot, cc) = __uint_as_float(static_cast<unsigned>(w[i]));
                }
        }
        __syncthreads();
        if (MULTI) aborted = s_gave != 0;
        // U of the trailing columns (cur's in the lower half of the wave, nxt's in the upper) and
        // the rank-8 update: Re += Ur (-Lr) + (-Ui) (-Li), Im += Ui (-Lr) + Ur (-Li).
        float ur[8], ui[8];
        {
            const int col = (lane < 32 ? live : 32) + (lane & 31);
#pragma unroll
            for (int s = 0; s < 8; ++s)
            {
                ur[s] = s_ur[s][col];
                ui[s] = s_ui[s][col];
            }
#pragma unroll
            for (int i = 1; i < 8; ++i)
#pragma unroll
                for (int s = 0; s < i; ++s)
                {
                    const float2 x = SubMul(make_float2(ur[i], ui[i]), s_l[i][s], make_float2(ur[s], ui[s]));
                    ur[i] = x.x;
                    ui[i] = x.y;
                }
#pragma unroll
            for (int s = 0; s < 4; ++s)
            {
                SwapHalves(ur[2 * s], ur[2 * s + 1]);
                SwapHalves(ui[2 * s], ui[2 * s + 1]);
            }
        }
        float br[2][4], bi[2][4];
#pragma unroll
        for (int s = 0; s < 4; ++s)
        {
            br[0][s] = -lm[2 * s].x;
            br[1][s] = -lm[2 * s + 1].x;
            SwapHalves(br[0][s], br[1][s]);
            bi[0][s] = -lm[2 * s].y;
            bi[1][s] = -lm[2 * s + 1].y;
            SwapHalves(bi[0][s], bi[1][s]);
        }
        if ((q & 3) != 3)  // uniform: cur still has columns
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                {
                    curR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s], br[t][s], curR[t], 0, 0, 0);
                    curI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ui[2 * s], br[t][s], curI[t], 0, 0, 0);
                    curR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(-ui[2 * s], bi[t][s], curR[t], 0, 0, 0);
                    curI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s], bi[t][s], curI[t], 0, 0, 0);
                }
        if (q < 4)  // uniform: nxt lies right of the block
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int t = 0; t < 2; ++t)
                {
                    nxtR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s + 1], br[t][s], nxtR[t], 0, 0, 0);
                    nxtI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ui[2 * s + 1], br[t][s], nxtI[t], 0, 0, 0);
                    nxtR[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(-ui[2 * s + 1], bi[t][s], nxtR[t], 0, 0, 0);
                    nxtI[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(ur[2 * s + 1], bi[t][s], nxtI[t], 0, 0, 0);
                }
        if ((q & 3) == 3)  // uniform
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                curR[t] = nxtR[t];
                curI[t] = nxtI[t];
            }
    }

    if (MULTI && !aborted)
        aborted = __hip_atomic_load(p.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    if (MULTI && aborted && valid)
        for (int c = 0; c < wact; ++c) Ap[c * lda + lr] = make_float2(__builtin_nanf(""), __builtin_nanf(""));
    if (g == 0 && wid == 0)
    {
        if (p.ipiv != nullptr && lane < wact) p.ipiv[c0 + lane] = c0 + pivots + 1;
        if (lane == 0 && zeroCol != 0 && *p.info == 0) *p.info = c0 + zeroCol;
    }
    if (!MULTI) __syncthreads();  // every source was read before any is written
    if (valid)
    {
        p.rowsrc[c0 + pos] = srcv;
        int2* const list = reinterpret_cast<int2*>(p.moves);
        const int2 move = make_int2(c0 + pos, c0 + lr);
        if (pos < wact) list[pos] = pos != lr ? move : make_int2(-1, -1);
        if (lr < wact) list[W + lr] = pos >= wact ? move : make_int2(-1, -1);
    }
}

// unitlower.h's solve form of a unit-lower block, real parts, then imaginary parts 4096 floats
// further; s: the block's strictly lower triangle row-major in LDS, imaginary parts kC further.
// Growth in the norm |re| + |im|; 256: 768 diagonal blocks each of complex Gaussian, uniform and
// small-integer matrices with partial pivoting have 113, 132 and 131 at most.
constexpr int kC = 64 * kInvStride;
constexpr float kCInverseGrowth = 256.0f;
__device__ inline void CSolveForm64(const float* s, float* __restrict__ form, int tid)
{
    const int lane = tid & 63, wave = tid >> 6;
    if ((lane >> 4) != wave)
#pragma unroll
        for (int k = 0; k < 16; ++k)
        {
            const int c = 16 * wave + k, at = lane * kInvStride + c;
            const bool low = (lane >> 4) > wave;
            if (c != 63 || lane != 0) form[c * 64 + lane] = low ? -s[at] : 0.0f;
            form[4096 + c * 64 + lane] = low ? -s[kC + at] : 0.0f;
        }
    if (wave != 0) return;
    const int b = lane & 48;
    float2 x[16];
    float grow[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < 16; ++i)
    {
        float2 v = make_float2(i == (lane & 15) ? 1.0f : 0.0f, 0.0f);
        const float* const row = s + (b + i) * kInvStride + b;
#pragma unroll
        for (int k = 0; k < i; ++k)
        {
            const float2 l = make_float2(row[k], row[kC + k]);
            v = SubMul(v, l, x[k]);
            grow[k & 3] = fmaf(fabsf(l.x) + fabsf(l.y), fabsf(x[k].x) + fabsf(x[k].y), grow[k & 3]);
        }
        x[i] = v;
        grow[3] += fabsf(v.x) + fabsf(v.y);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i)
    {
        const bool low = i > (lane & 15);
        form[lane * 64 + b + i] = low ? x[i].x : 0.0f;
        form[4096 + lane * 64 + b + i] = low ? x[i].y : 0.0f;
    }
    const bool fine = (grow[0] + grow[1]) + (grow[2] + grow[3]) <= kCInverseGrowth;
    const bool all = __all(fine);
    if (lane == 0) form[kSubstituteFlag] = all ? 0.0f : 1.0f;
}

struct CSolveOperands
{
    float re[40], im[40];
    float substitute;
};
__device__ inline void LoadOperands(const float* __restrict__ form, int ui, int uk, CSolveOperands& o)
{
#pragma unroll
    for (int t = 0, x = 0; t < 4; ++t)
#pragma unroll
        for (int d = t; d < 4; ++d)
#pragma unroll
            for (int s = 0; s < 4; ++s, ++x)
            {
                const int at = (16 * t + 4 * uk + s) * 64 + 16 * d + ui;
                o.re[x] = form[at];
                o.im[x] = form[4096 + at];
            }
    o.substitute = form[kSubstituteFlag];
}

// unitlower.h's SolveColumns on pairs of real products.
__device__ inline bool CSolveColumns(const CSolveOperands& o, f32x4 (&re)[4], f32x4 (&im)[4])
{
    bool fine = o.substitute == 0.0f;
    auto add = [&](int x, float br, float bi, f32x4& r, f32x4& i)
    {
        r = __builtin_amdgcn_mfma_f32_16x16x4f32(o.re[x], br, r, 0, 0, 0);
        i = __builtin_amdgcn_mfma_f32_16x16x4f32(o.re[x], bi, i, 0, 0, 0);
        r = __builtin_amdgcn_mfma_f32_16x16x4f32(-o.im[x], bi, r, 0, 0, 0);
        i = __builtin_amdgcn_mfma_f32_16x16x4f32(o.im[x], br, i, 0, 0, 0);
    };
    f32x4 sr[4], si[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) sr[t] = si[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int t = 0, x = 0; t < 4; ++t)
    {
        if (t > 0)
        {
            re[t] = re[t] + sr[t];
            im[t] = im[t] + si[t];
        }
        f32x4 ur = {0.0f, 0.0f, 0.0f, 0.0f}, ux = ur;
#pragma unroll
        for (int s = 0; s < 4; ++s, ++x) add(x, re[t][s], im[t][s], ur, ux);
        re[t] = re[t] + ur;
        im[t] = im[t] + ux;
#pragma unroll
        for (int d = t + 1; d < 4; ++d)
#pragma unroll
            for (int s = 0; s < 4; ++s, ++x) add(x, re[t][s], im[t][s], sr[d], si[d]);
#pragma unroll
        for (int r = 0; r < 4; ++r) fine = fine && fabsf(re[t][r]) <= FLT_MAX && fabsf(im[t][r]) <= FLT_MAX;
    }
    return __all(fine);
}

__device__ inline void SubstituteColumns(const float2* __restrict__ T, int64_t ldt, int size, int lane, float2 (&v)[16])
{
#pragma unroll 1
    for (int k0 = 0; k0 < size; k0 += 8)
    {
        float2 l[8];
#pragma unroll
        for (int e = 0; e < 8; ++e)
            l[e] = lane > k0 + e && lane < size ? T[(k0 + e) * ldt + lane] : make_float2(0.0f, 0.0f);
#pragma unroll
        for (int e = 0; e < 8; ++e)
#pragma unroll
            for (int c = 0; c < 16; ++c)
            {
                const float2 y = SubMul(v[c], l[e], make_float2(ReadLane(v[c].x, k0 + e), ReadLane(v[c].y, k0 + e)));
                if (lane > k0 + e && lane < size) v[c] = y;
            }
    }
}

// leaf.hip's leaf_finish_kernel for complex columns.
__global__ __launch_bounds__(256) void cleaf_finish_kernel(float2* __restrict__ A, int64_t lda, int j0, int c0, int wact,
                                                           int hi, const int2* __restrict__ moves,
                                                           const int* __restrict__ err, float* __restrict__ form,
                                                           float2* __restrict__ ub)
{
    __builtin_amdgcn_s_setprio(3);  // before the trailing product's waves on the same SIMD
    constexpr int W = kCLeafWidth;
    __shared__ __align__(16) float s_l[2 * kC];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (*err != 0) return;  // after a timeout the list is not complete
    const int2 none = make_int2(-1, -1);
    const int2 m0 = lane < wact ? moves[lane] : none, m1 = lane < wact ? moves[W + lane] : none;
    const int from = m0.x >= 0 ? m0.y : c0 + lane;  // the row that ends at position lane
    const float2 zero2 = make_float2(0.0f, 0.0f);
    if (blockIdx.x > 0)
    {
        const int left = c0 - j0, q = static_cast<int>(blockIdx.x - 1) * 4 + wave;
        const int c = q < left ? j0 + q : c0 + wact + (q - left);
        if (c >= hi) return;
        float2* const col = A + c * lda;
        float2 x0 = zero2, x1 = zero2;
        if (lane < wact) x0 = col[from];
        if (m1.x >= 0) x1 = col[m1.y];
        if (q >= left)
            ub[static_cast<size_t>(q - left) * W + lane] = x0;
        else if (m0.x >= 0)
            col[m0.x] = x0;
        if (m1.x >= 0) col[m1.x] = x1;
        return;
    }
    float2 x0[16], x1[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
    {
        const int c = wave * 16 + k;
        x0[k] = x1[k] = zero2;
        if (c < wact && lane < wact)
        {
            const float2* const col = A + (c0 + c) * lda;
            x0[k] = col[from];
            if (m1.x >= 0) x1[k] = col[m1.y];
        }
    }
#pragma unroll
    for (int k = 0; k < 16; ++k)
    {
        const int c = wave * 16 + k;
        if (c < wact)
        {
            float2* const col = A + (c0 + c) * lda;
            if (m0.x >= 0) col[m0.x] = x0[k];
            if (m1.x >= 0) col[m1.x] = x1[k];
        }
        const bool in = lane > c && lane < wact;
        s_l[lane * kInvStride + c] = in ? x0[k].x : 0.0f;
        s_l[kC + lane * kInvStride + c] = in ? x0[k].y : 0.0f;
    }
    __syncthreads();
    CSolveForm64(s_l, form, tid);
}

// leaf.hip's panel_update_kernel for complex columns: 64 x 64 tiles of C, one 32 x 32 tile a wave
// (order 512, on average 15 us; 23 us with the product read back from LDS and operands in the loop).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void cpanel_update_kernel(
    float2* __restrict__ A, int64_t lda, int m, int c0, int hi, const float* __restrict__ form,
    const float2* __restrict__ ub)
{
    __builtin_amdgcn_s_setprio(3);  // before the trailing product's waves on the same SIMD
    constexpr int W = kCLeafWidth;
    constexpr int BS = W + 4;
    __shared__ __align__(16) float s_r[W * BS], s_i[W * BS];  // [column][row] of U
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 31, lk = lane >> 5, ui = lane & 15, uk = lane >> 4;
    const int col0 = static_cast<int>(blockIdx.y) * W, cols = min(W, hi - (c0 + W) - col0);
    const int row0 = c0 + W + static_cast<int>(blockIdx.x) * 64;
    float2* const Ct = A + (c0 + W + col0) * lda;
    const int row = row0 + (wave & 1) * 32 + li, strip = (wave >> 1) * 32;
    const bool inRow = row < m;
    const float2* const ubc = ub + static_cast<size_t>(col0 + 16 * wave) * W;
    CSolveOperands op;
    LoadOperands(form, ui, uk, op);
    f32x4 re[4], im[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
        {
            const float2 v = 16 * wave + ui < cols ? ubc[ui * W + 16 * t + 4 * uk + r] : make_float2(0.0f, 0.0f);
            re[t][r] = v.x;
            im[t][r] = v.y;
        }
    float2 l21[32];
    const float2* lp = A + c0 * lda + row + lk * lda;
#pragma unroll
    for (int t = 0; t < 32; ++t)
    {
        l21[t] = inRow ? *lp : make_float2(0.0f, 0.0f);
        lp += 2 * lda;
    }
    if (__builtin_expect(CSolveColumns(op, re, im), 1))  // uniform over the wave
    {
#pragma unroll
        for (int t = 0; t < 4; ++t)
        {
            *reinterpret_cast<f32x4*>(s_r + (16 * wave + ui) * BS + 16 * t + 4 * uk) = re[t];
            *reinterpret_cast<f32x4*>(s_i + (16 * wave + ui) * BS + 16 * t + 4 * uk) = im[t];
        }
    }
    else
    {
        float2 v[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = 16 * wave + c < cols ? ubc[c * W + lane] : make_float2(0.0f, 0.0f);
        SubstituteColumns(A + c0 * lda + c0, lda, W, lane, v);
#pragma unroll
        for (int c = 0; c < 16; ++c)
        {
            s_r[(16 * wave + c) * BS + lane] = v[c].x;
            s_i[(16 * wave + c) * BS + lane] = v[c].y;
        }
    }
    __syncthreads();
    if (blockIdx.x == 0)
#pragma unroll
        for (int k = 0; k < 16; ++k)
            if (16 * wave + k < cols)
                Ct[(16 * wave + k) * lda + c0 + lane] =
                    make_float2(s_r[(16 * wave + k) * BS + lane], s_i[(16 * wave + k) * BS + lane]);
    f32x16 ar, ai;
#pragma unroll
    for (int v = 0; v < 16; ++v) ar[v] = ai[v] = 0.0f;
#pragma unroll
    for (int t = 0; t < 32; ++t)
    {
        const float ur = s_r[(strip + li) * BS + 2 * t + lk], ux = s_i[(strip + li) * BS + 2 * t + lk];
        ar = __builtin_amdgcn_mfma_f32_32x32x2f32(ur, l21[t].x, ar, 0, 0, 0);
        ai = __builtin_amdgcn_mfma_f32_32x32x2f32(ux, l21[t].x, ai, 0, 0, 0);
        ar = __builtin_amdgcn_mfma_f32_32x32x2f32(-ux, l21[t].y, ar, 0, 0, 0);
        ai = __builtin_amdgcn_mfma_f32_32x32x2f32(ur, l21[t].y, ai, 0, 0, 0);
    }
    // All loads before the first store (a load under its own condition waits by itself).
    const float2* const Cr = Ct + min(row, m - 1);
    float2 x[16];
#pragma unroll
    for (int v = 0; v < 16; ++v) x[v] = Cr[min(strip + (v & 3) + 8 * (v >> 2) + 4 * lk, cols - 1) * lda];
#pragma unroll
    for (int v = 0; v < 16; ++v)
    {
        const int c = strip + (v & 3) + 8 * (v >> 2) + 4 * lk;
        if (inRow && c < cols) Ct[c * lda + row] = make_float2(x[v].x - ar[v], x[v].y - ai[v]);
    }
}

// B <- L^{-1} B, one workgroup of eight waves per 16 columns held in LDS (up to 512 rows, parts
// apart), as gemm.hip's trsm_lu_kernel: one wave solves the 64-row blocks from their solve forms,
// seven subtract L X_b from the rows below in tiles of 16. The critical path calls it with 512
// columns, so width is what spreads it: 512 x 512 takes 32 workgroups and 75 us alone (32
// columns and four waves 160 us), 122 us on average beside the product of order 8192.
constexpr int kCXStride = 17;
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void ctrsm_lu_kernel(
    int K, int N, const float2* __restrict__ T, int64_t ldt, const float* __restrict__ forms, float2* __restrict__ B,
    int64_t ldb)
{
    extern __shared__ __align__(16) float s_mem[];  // Kp rows of stride 17, real, then imaginary
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ui = lane & 15, uk = lane >> 4;
    const int nblk = (K + 63) / 64, Kp = nblk * 64;
    float* const xr = s_mem;
    float* const xi = s_mem + Kp * kCXStride;
    const int c0 = static_cast<int>(blockIdx.x) * 16, nc = min(16, N - c0);
    for (int c = wave; c < 16; c += 8)
        for (int r = lane; r < Kp; r += 64)
        {
            const float2 v = c < nc && r < K ? B[(c0 + c) * ldb + r] : make_float2(0.0f, 0.0f);
            xr[r * kCXStride + c] = v.x;
            xi[r * kCXStride + c] = v.y;
        }
    __syncthreads();
    // They meet twice a block.
    constexpr int UPD = 7;
    if (wave == UPD)
    {
        CSolveOperands op;
        LoadOperands(forms, ui, uk, op);
        for (int b = 0; b < nblk; ++b)
        {
            const int k0 = b * 64;
            f32x4 re[4], im[4];
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                {
                    const int at = (k0 + 16 * t + 4 * uk + r) * kCXStride + ui;
                    re[t][r] = xr[at];
                    im[t][r] = xi[at];
                }
            if (__builtin_expect(CSolveColumns(op, re, im), 1))  // uniform
            {
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                    {
                        const int at = (k0 + 16 * t + 4 * uk + r) * kCXStride + ui;
                        xr[at] = re[t][r];
                        xi[at] = im[t][r];
                    }
            }
            else
            {
                float2 v[16];
#pragma unroll
                for (int c = 0; c < 16; ++c)
                    v[c] = make_float2(xr[(k0 + lane) * kCXStride + c], xi[(k0 + lane) * kCXStride + c]);
                SubstituteColumns(T + k0 * ldt + k0, ldt, min(64, K - k0), lane, v);
#pragma unroll
                for (int c = 0; c < 16; ++c)
                {
                    xr[(k0 + lane) * kCXStride + c] = v[c].x;
                    xi[(k0 + lane) * kCXStride + c] = v[c].y;
                }
            }
            if (b + 1 < nblk) LoadOperands(forms + static_cast<size_t>(b + 1) * kCFormBlock, ui, uk, op);
            __syncthreads();
            __syncthreads();
        }
    }
    else
        for (int b = 0; b < nblk; ++b)
        {
            const int k0 = b * 64;
            int r0 = k0 + 64 + wave * 16;
            // Blocks with rows below them are full; rows beyond K repeat the last one.
            float2 lf[16];
            auto loadTile = [&]()
            {
                const float2* const Lc = T + k0 * ldt + min(r0 + ui, K - 1);
#pragma unroll
                for (int t = 0; t < 16; ++t) lf[t] = Lc[(4 * t + uk) * ldt];
            };
            if (r0 < K) loadTile();
            __syncthreads();
            while (r0 < K)
            {
                f32x4 ar = {0.0f, 0.0f, 0.0f, 0.0f}, ai = ar;
#pragma unroll
                for (int t = 0; t < 16; ++t)
                {
                    const int at = (k0 + 4 * t + uk) * kCXStride + ui;
                    const float ur = xr[at], ux = xi[at];
                    ar = __builtin_amdgcn_mfma_f32_16x16x4f32(ur, lf[t].x, ar, 0, 0, 0);
                    ai = __builtin_amdgcn_mfma_f32_16x16x4f32(ux, lf[t].x, ai, 0, 0, 0);
                    ar = __builtin_amdgcn_mfma_f32_16x16x4f32(-ux, lf[t].y, ar, 0, 0, 0);
                    ai = __builtin_amdgcn_mfma_f32_16x16x4f32(ur, lf[t].y, ai, 0, 0, 0);
                }
                const int row = r0 + ui;
                r0 += 16 * UPD;
                if (r0 < K) loadTile();
                if (row < K)
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                    {
                        const int at = row * kCXStride + 4 * uk + v;
                        xr[at] -= ar[v];
                        xi[at] -= ai[v];
                    }
            }
            __syncthreads();
        }
    for (int c = wave; c < nc; c += 8)
        for (int r = lane; r < K; r += 64)
            B[(c0 + c) * ldb + r] = make_float2(xr[r * kCXStride + c], xi[r * kCXStride + c]);
}

template <int NW>
hipError_t CMulti(CLeafArgs a, bool spread, hipStream_t stream)
{
    const int groups = (a.m - a.c0 + 64 * NW - 1) / (64 * NW);
    if (groups > kCLeafMaxGroups) return hipErrorInvalidValue;
    // Cooperative launch: the workgroups wait for each other every column, so the runtime must
    // make all of them resident at once (it refuses a grid that cannot be).
    void* kargs[] = {&a};
    const void* fn = spread ? reinterpret_cast<const void*>(&cpanel_leaf_kernel<NW, true, true>)
                            : reinterpret_cast<const void*>(&cpanel_leaf_kernel<NW, true, false>);
    return hipLaunchCooperativeKernel(fn, dim3((spread ? 8 : 1) * groups), dim3(64 * NW), kargs, 0, stream);
}
}  // namespace

hipError_t CLeafColumns(const CLeafArgs& a, bool spread, hipStream_t stream)
{
    const int mp = a.m - a.c0;
    if (mp <= 0 || mp > kCLeafMaxRows || a.wact <= 0 || a.wact > kCLeafWidth) return hipErrorInvalidValue;
    if (mp > 8192) return CMulti<8>(a, spread, stream);
    if (mp > kCLeafSingleRows) return CMulti<4>(a, spread, stream);
    if (mp <= 64)
        hipLaunchKernelGGL((cpanel_leaf_kernel<1, false, false>), dim3(1), dim3(64), 0, stream, a);
    else if (mp <= 128)
        hipLaunchKernelGGL((cpanel_leaf_kernel<2, false, false>), dim3(1), dim3(128), 0, stream, a);
    else if (mp <= 256)
        hipLaunchKernelGGL((cpanel_leaf_kernel<4, false, false>), dim3(1), dim3(256), 0, stream, a);
    else
        hipLaunchKernelGGL((cpanel_leaf_kernel<8, false, false>), dim3(1), dim3(512), 0, stream, a);
    return hipGetLastError();
}

hipError_t CLeafFinish(const CLeafArgs& a, float* form, float2* ub, hipStream_t stream)
{
    const int others = (a.c0 - a.j0) + (a.panelEnd - a.c0 - a.wact);
    hipLaunchKernelGGL(cleaf_finish_kernel, dim3(1 + (others + 3) / 4), dim3(256), 0, stream, a.A,
                       static_cast<int64_t>(a.lda), a.j0, a.c0, a.wact, a.panelEnd,
                       reinterpret_cast<const int2*>(a.moves), a.err, form, ub);
    return hipGetLastError();
}

hipError_t CPanelUpdate(const CLeafArgs& a, const float* form, const float2* ub, hipStream_t stream)
{
    const int cols = a.panelEnd - a.c0 - kCLeafWidth, rows = a.m - a.c0 - kCLeafWidth;
    if (a.wact != kCLeafWidth) return hipErrorInvalidValue;
    if (cols <= 0) return hipSuccess;
    hipLaunchKernelGGL(cpanel_update_kernel, dim3(std::max(1, (rows + 63) / 64), (cols + 63) / 64), dim3(256), 0, stream,
                       a.A, static_cast<int64_t>(a.lda), a.m, a.c0, a.panelEnd, form, ub);
    return hipGetLastError();
}

hipError_t CTrsmLowerUnit(int K, int N, const float2* T, int ldt, const float* forms, float2* B, int ldb,
                          hipStream_t stream)
{
    if (K <= 0 || N <= 0) return hipSuccess;
    if (K > 512) return hipErrorInvalidValue;
    const size_t lds = static_cast<size_t>((K + 63) / 64) * 64 * kCXStride * 2 * sizeof(float);
    hipLaunchKernelGGL(ctrsm_lu_kernel, dim3((N + 15) / 16), dim3(512), lds, stream, K, N, T, static_cast<int64_t>(ldt),
                       forms, B, static_cast<int64_t>(ldb));
    return hipGetLastError();
}
}  // namespace ops
