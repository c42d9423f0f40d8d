// Partial-pivoting panel leaves of the real LU, gfx950.
// Reference: src/sgetrf/real_lu_blocked_kernel.cpp:342-389, :467-482 (pivot choice, scaling,
// rank-1 update of the panel) and src/utils/kernel/real_lu.hpp:419-437.
//
// A leaf factors up to W columns of rows [c0, m). Per column its work is a serial chain
// (pivot search, exchange of the pivot row, update of the next column), so everything that
// is not needed for the next column is taken off that chain: columns are processed eight at
// a time, the eight-column block right-looking in registers with one matrix row per lane,
// and the columns right of the block receive its eight pivots afterwards as one rank-8
// update on the FP32 matrix cores. The rows of the leaf live in MFMA accumulator layout
// (v_mfma_f32_32x32x2_f32 with the matrix transposed: lane l and l + 32 of a 32-row tile
// hold the even and odd quads of columns of row l); v_permlane32_swap turns two tiles into
// the row-per-lane form of a block and back, and pairs of multiplier registers into the
// B operand, so no data passes through LDS for the change of layout.
//
// Pivoting is implicit: each row tracks the position it occupies under the LAPACK
// interchange sequence; the pivot of column j is the candidate (position >= j) with the
// largest |a| and, on ties, the lowest position. Finished columns are stored at once, every
// row where it started; leaf_swap_kernel then applies the leaf's interchanges to all panel
// columns with one wave per column (inside the leaf they would cost one workgroup a cache
// line per moved row and column: about 50 us for a 512-column panel).
//
// What bounds it: the latency of the chain, one column about 0.35 us on one workgroup (24 us
// of 64 columns) and 1.2 us over several (two trips through the XCD's L2 included), far from
// any rate of the chip. Eight columns per block: the block's own columns cost up to seven
// FMAs per row on the chain and the exchanged pivot row stays at eight words. A wave issues about
// one instruction in five clocks here, so their number is the time: about 190 a column, where
// the unrolled leaf this replaces had 265 and passed whole pivot rows through LDS. 64
// columns, alone on the GPU, before and after: 64 rows 56 -> 26 us, 512 rows 104 -> 48 us,
// 1024 rows 104 -> 66 us, 2048 rows 158 -> 89 us, 8192 rows 125 -> 92 us.
#include "leaf.h"

#include <algorithm>
#include <cfloat>
#include <climits>

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

// Maximum over the NW values that the lanes hold cyclically (lane l: value l % NW).
template <int NW>
__device__ inline unsigned CyclicMaxU32(unsigned v)
{
    auto mx = [](unsigned a, unsigned b) { return a > b ? a : b; };
    if (NW >= 2) v = mx(v, DppU32<0xB1>(v));
    if (NW >= 4) v = mx(v, DppU32<0x4E>(v));
    if (NW >= 8) v = mx(v, DppU32<0x124>(v));
    if (NW >= 16) v = mx(v, DppU32<0x128>(v));
    return v;
}

// NW waves per workgroup, RP groups of 64 rows per wave. MULTI: the rows are spread over
// gridDim.x workgroups (<= kLeafMaxGroups) that exchange one candidate each per column through
// tagged 64-bit words: word 0 the key (16-bit tag, 32-bit magnitude class, 14-bit rank of the
// position, sign), words 1..7 the candidate's values in the block's columns, word 8 the pivot's
// reciprocal; a workgroup polls all words of a column in one round trip. Words alternate with
// the column parity: a workgroup writes column j + 2 only after all have written j + 1, i.e.
// after all have read j. After a block the owners of its pivot rows publish those rows for the
// rank-8 update the same way. Spins are bounded: on a timeout the workgroup raises *err, runs
// on without waiting and stores NaN rows.
// SPREAD: the grid holds 8 workgroups per participant and only ids = 0 mod 8 take part.
// Workgroups go to the XCDs round-robin by id, so the participants share one XCD (checked
// per device by LeafSpreadProbe) and the words travel through its L2 only.
template <int NW, int RP, bool MULTI, bool SPREAD>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(NW > 8 ? 4 : 2)))
void panel_leaf_kernel(LeafArgs p)
{
    constexpr int T = 64 * NW, W = kLeafMaxWidth;
    static_assert(W == 64, "two 32-column chunks");
    constexpr int US = W + 28;  // pivot rows' stride: quads in different banks, room for stale columns
    __shared__ uint2 s_key[2][NW];
    __shared__ __align__(16) float s_val[2][NW * 8];
    __shared__ __align__(16) float s_u[8][US];
    __shared__ __align__(16) float s_l[8][8];
    __shared__ float s_win[2][16];
    __shared__ int s_gave;  // a wait of this workgroup ran out

    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (SPREAD && (blockIdx.x & 7) != 0) return;  // not a participant
    const int P = MULTI ? static_cast<int>(SPREAD ? gridDim.x >> 3 : gridDim.x) : 1;
    const int g = MULTI ? static_cast<int>(SPREAD ? blockIdx.x >> 3 : blockIdx.x) : 0;
    const int c0 = p.c0, mp = p.m - c0, wact = p.wact;
    const int64_t lda = p.lda;
    float* const Ap = p.A + static_cast<int64_t>(c0) * lda + c0;
    const int rbase = g * (T * RP) + wid * (64 * RP) + lane;
    bool aborted = false;  // uniform over the wave

    // cur: the 32-column chunk being factored, nxt the one right of it. Lane l of tile t holds
    // row l % 32 of the tile, columns 8 k + 4 (l / 32) + r in element 4 k + r. cur is rotated by
    // one block per step, so that the current block is always its group k = 0.
    f32x16 cur[RP][2], nxt[RP][2];
    int pos[RP], srcv[RP];
#pragma unroll
    for (int rp = 0; rp < RP; ++rp)
    {
        const int lr = rbase + rp * 64;
        const bool valid = lr < mp;
        float x[W];
#pragma unroll
        for (int c = 0; c < W; ++c) x[c] = 0.0f;
        srcv[rp] = 0;
        if (valid)
        {
            // One running address per lane; columns beyond wact repeat the last one (nothing
            // reads them).
            const float* src = Ap + lr;
#pragma unroll
            for (int c = 0; c < W; ++c)
            {
                x[c] = *src;
                src += c + 1 < wact ? lda : 0;
            }
            // Read before any workgroup can store (stores follow the last column's exchange).
            srcv[rp] = p.newPanel ? c0 + lr : p.rowsrc[c0 + lr];
        }
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                SwapHalves(x[8 * k + r], x[8 * k + 4 + r]);
                (k < 4 ? cur : nxt)[rp][0][4 * (k % 4) + r] = x[8 * k + r];
                (k < 4 ? cur : nxt)[rp][1][4 * (k % 4) + r] = x[8 * k + 4 + r];
            }
        pos[rp] = valid ? lr : -1;  // padding rows: never a candidate, never below a pivot
    }
    if constexpr (MULTI)
    {
        // No column is exchanged before every workgroup is resident and has its rows: full-rate
        // polling by the first ones holds up memory accesses on their XCD -- beside a kernel that
        // fills the chip (the trailing update of n >= 9000) so much that the loads of the last
        // workgroups, for which the first ones waited, did not return.
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        unsigned long long* const arrival = p.slots + kLeafArrivalWord;
        if (tid == 0) StoreWord(arrival + g, p.tagBase, SPREAD);
        if (wid == 0)
        {
            // A wait of this factorization has run out already, in an earlier leaf or in a workgroup
            // of this one that came before: no more waits, but NaN rows and a list of moves from
            // every workgroup all the same.
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
    // Candidates of column j: positions j .. j + span.
    const unsigned span = p.pivoting ? 0x3fffffffu : 0u;

    for (int q = 0; 8 * q < wact; ++q)
    {
        // The block in row-per-lane form: v[rp][c] is column 8 q + c.
        float v[RP][8], lm[RP][8];
#pragma unroll
        for (int rp = 0; rp < RP; ++rp)
        {
#pragma unroll
            for (int r = 0; r < 4; ++r)
            {
                v[rp][r] = cur[rp][0][r];
                v[rp][4 + r] = cur[rp][1][r];
                SwapHalves(v[rp][r], v[rp][4 + r]);
            }
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int e = 0; e < 12; ++e) cur[rp][t][e] = cur[rp][t][e + 4];
        }

#pragma unroll
        for (int jj = 0; jj < 8; ++jj)
        {
            const int j = 8 * q + jj;
            if (j >= wact) break;  // uniform
            const int par = jj & 1;
            // The lane's candidate: magnitude class (0: none; top bit and |a| bits + 1; a NaN is
            // the pivot on the diagonal position and ranks lowest elsewhere --
            // src/utils/kernel/real_lu.hpp:59-77, :100-109), position, value.
            unsigned bh = 0u;
            int bp = 0;
            float bv = 0.0f, sel[8];
#pragma unroll
            for (int rp = 0; rp < RP; ++rp)
            {
                const unsigned ab = __float_as_uint(v[rp][jj]) & 0x7fffffffu;
                const unsigned mag = ab <= 0x7f800000u ? ab + 0x80000001u : (pos[rp] == j ? 0xffffffffu : 0x80000000u);
                const unsigned h = static_cast<unsigned>(pos[rp] - j) <= span ? mag : 0u;
                const bool better = rp == 0 || h > bh || (h == bh && pos[rp] < bp);
                bh = better ? h : bh;
                bp = better ? pos[rp] : bp;
                bv = better ? v[rp][jj] : bv;
#pragma unroll
                for (int c = jj + 1; c < 8; ++c) sel[c] = better ? v[rp][c] : sel[c];
            }
            float br = 1.0f / bv;
            unsigned top = WaveMaxU32(bh);
            unsigned long long tie = __ballot(bh == top);
            asm volatile("" : "+v"(br));  // beside the search, where its latency is hidden
            if (__builtin_expect(__popcll(tie) != 1, 0))  // uniform
            {
                const unsigned low = WaveMaxU32(bh == top ? ~static_cast<unsigned>(bp) : 0u);
                tie = __ballot(bh == top && ~static_cast<unsigned>(bp) == low);
            }
            int wl = __builtin_ctzll(tie);
            int pp;           // position of the pivot
            unsigned dsign;   // its sign bit
            float rec, u[8];  // its reciprocal, its row in the block's columns beyond j
            float x0 = 0.0f, x1 = 0.0f;
            if constexpr (NW == 1)
            {
                pp = __builtin_amdgcn_readlane(bp, wl);
                dsign = __builtin_amdgcn_readlane(__float_as_uint(bv), wl) & 0x80000000u;
                rec = ReadLane(br, wl);
#pragma unroll
                for (int c = jj + 1; c < 8; ++c) u[c] = ReadLane(sel[c], wl);
            }
            else
            {
                if (lane == wl)
                {
                    s_key[par][wid] = make_uint2(top, (static_cast<unsigned>(bp) & 0x7fffffffu) |
                                                          (__float_as_uint(bv) & 0x80000000u));
                    s_val[par][wid * 8] = br;
#pragma unroll
                    for (int c = jj + 1; c < 8; ++c) s_val[par][wid * 8 + c] = sel[c];
                }
                __syncthreads();
                // Every wave reads all waves' candidates: lane l word l % 8 of wave l / 8.
                const uint2 k = s_key[par][lane & (NW - 1)];
                x0 = s_val[par][lane & (NW * 8 - 1)];
                if (NW > 8) x1 = s_val[par][64 + lane];
                const unsigned t = CyclicMaxU32<NW>(k.x);
                top = __builtin_amdgcn_readfirstlane(t);
                unsigned hit = static_cast<unsigned>(__ballot(k.x == top)) & ((1u << NW) - 1u);
                if (__builtin_expect(__popc(hit) != 1, 0))  // uniform
                {
                    const unsigned low = CyclicMaxU32<NW>(k.x == top ? 0x7fffffffu - (k.y & 0x7fffffffu) : 0u);
                    hit = static_cast<unsigned>(__ballot(k.x == top && 0x7fffffffu - (k.y & 0x7fffffffu) == low)) &
                          ((1u << NW) - 1u);
                }
                wl = __builtin_ctz(hit | 0x80000000u) & (NW - 1);
                const unsigned ky = __builtin_amdgcn_readlane(k.y, wl);
                pp = static_cast<int>(ky & 0x7fffffffu);
                dsign = ky & 0x80000000u;
                if constexpr (!MULTI)
                {
                    if (NW > 8) x0 = wl >= 8 ? x1 : x0;  // uniform
                    const int at = (wl & 7) * 8;
                    rec = ReadLane(x0, at);
#pragma unroll
                    for (int c = jj + 1; c < 8; ++c) u[c] = ReadLane(x0, at + c);
                }
            }
            if constexpr (MULTI)
            {
                static_assert(!MULTI || NW <= 8, "one value register per lane");
                const unsigned tag = p.tagBase + static_cast<unsigned>(j);
                unsigned long long* const words = p.slots + (j & 1) * (9 * kLeafMaxGroups);
                const unsigned long long key =
                    (static_cast<unsigned long long>(tag & 0xffffu) << 48) |
                    (top == 0u ? 0ull
                               : (static_cast<unsigned long long>(top) << 16) |
                                     static_cast<unsigned>(((0x3fff - pp) << 1) | (dsign != 0u ? 1 : 0)));
                if constexpr (NW == 1)
                {
                    if (lane == wl)
                    {
                        StoreWord(words + g, key, SPREAD);
                        StoreTagged(words + 8 * kLeafMaxGroups + g, tag, br, SPREAD);
#pragma unroll
                        for (int c = jj + 1; c < 8; ++c)
                            StoreTagged(words + c * kLeafMaxGroups + g, tag, sel[c], SPREAD);
                    }
                }
                else if (wid == 0)  // uniform
                {
                    // The winner's eight words sit in lanes 8 wl .. 8 wl + 7 of every wave.
                    const int c = lane & 7;
                    if ((lane >> 3) == wl && (c == 0 || c > jj))
                        StoreTagged(words + (c == 0 ? 8 : c) * kLeafMaxGroups + g, tag, x0, SPREAD);
                    if (lane == 0) StoreWord(words + g, key, SPREAD);
                }
                // One wave polls for its workgroup, at a bounded rate: polling from every wave at
                // full rate starves whatever else runs on the XCD of memory accesses, down to the
                // instruction fetches of workgroups that have not reached the column yet.
                if (NW == 1 || wid == 0)  // uniform
                {
                    unsigned hi = 0u, lo = 0u;
                    float wr = 0.0f, wv[8];
#pragma unroll
                    for (int c = 0; c < 8; ++c) wv[c] = 0.0f;
                    bool ok = false;
                    const bool mine = lane < P;
                    const unsigned lim = aborted ? 0u : p.spinLimit;
                    for (unsigned spins = 0; spins < lim; ++spins)
                    {
                        bool good = true;
                        if (mine)
                        {
                            const unsigned long long w0 = LoadWord(words + lane);
                            const unsigned long long w8 = LoadWord(words + 8 * kLeafMaxGroups + lane);
                            unsigned long long wc[8];
#pragma unroll
                            for (int c = jj + 1; c < 8; ++c) wc[c] = LoadWord(words + c * kLeafMaxGroups + lane);
                            unsigned diff = (static_cast<unsigned>(w0 >> 48) ^ (tag & 0xffffu)) |
                                            (static_cast<unsigned>(w8 >> 32) ^ tag);
                            wr = __uint_as_float(static_cast<unsigned>(w8));
#pragma unroll
                            for (int c = jj + 1; c < 8; ++c)
                            {
                                diff |= static_cast<unsigned>(wc[c] >> 32) ^ tag;
                                wv[c] = __uint_as_float(static_cast<unsigned>(wc[c]));
                            }
                            good = diff == 0u;
                            hi = static_cast<unsigned>(w0 >> 16);
                            lo = static_cast<unsigned>(w0) & 0x7fffu;
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
                        if (lane == 0) __hip_atomic_store(p.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        aborted = true;
                    }
                    top = WaveMaxU32(hi);
                    tie = __ballot(hi == top && mine);
                    if (__builtin_expect(__popcll(tie) != 1, 0))  // uniform
                    {
                        const unsigned low = WaveMaxU32(hi == top && mine ? lo : 0u);
                        tie = __ballot(hi == top && mine && lo == low);
                    }
                    wl = __builtin_ctzll(tie | (1ull << 63));
                    const unsigned ls = __builtin_amdgcn_readlane(lo, wl);
                    if constexpr (NW == 1)
                    {
                        pp = 0x3fff - static_cast<int>(ls >> 1);
                        dsign = (ls & 1u) << 31;
                        rec = ReadLane(wr, wl);
#pragma unroll
                        for (int c = jj + 1; c < 8; ++c) u[c] = ReadLane(wv[c], wl);
                    }
                    else
                    {
                        if (lane == wl)
                        {
                            s_win[par][0] = wr;
#pragma unroll
                            for (int c = jj + 1; c < 8; ++c) s_win[par][c] = wv[c];
                            s_win[par][8] = __uint_as_float(top);
                            s_win[par][9] = __uint_as_float(ls);
                        }
                        if (aborted && lane == 0) s_gave = 1;
                    }
                }
                if constexpr (NW > 1)
                {
                    __syncthreads();
                    const float x = s_win[par][lane & 15];
                    aborted = s_gave != 0;
                    top = __builtin_amdgcn_readlane(__float_as_uint(x), 8);
                    const unsigned ls = __builtin_amdgcn_readlane(__float_as_uint(x), 9);
                    pp = 0x3fff - static_cast<int>(ls >> 1);
                    dsign = (ls & 1u) << 31;
                    rec = ReadLane(x, 0);
#pragma unroll
                    for (int c = jj + 1; c < 8; ++c) u[c] = ReadLane(x, c);
                }
            }
            const bool none = top == 0u || (MULTI && aborted);  // uniform
            const int bpos = none ? j : pp;
            // |d| from the magnitude class (a NaN class gives a NaN).
            const unsigned dmag = none ? 0u : (top & 0x7fffffffu) - 1u;
            // Positions j and bpos are exchanged.
#pragma unroll
            for (int rp = 0; rp < RP; ++rp)
                pos[rp] = pos[rp] == bpos ? j : (pos[rp] == j ? bpos : pos[rp]);
            pivots = lane == j ? bpos : pivots;
            const bool zero = dmag == 0u;  // uniform
            if (zero && zeroCol == 0 && !(MULTI && aborted)) zeroCol = j + 1;
            // Multiplication by the reciprocal for a normal pivot, division otherwise; rows not
            // below the pivot (and every row under a zero pivot) take the multiplier 0.
            float qv[RP];
#pragma unroll
            for (int rp = 0; rp < RP; ++rp) qv[rp] = v[rp][jj] * rec;
            if (__builtin_expect(dmag - 0x00800000u > 0x7f000000u, 0))  // uniform: subnormal, zero or NaN
            {
                const float d = __uint_as_float(dmag | dsign);
#pragma unroll
                for (int rp = 0; rp < RP; ++rp) qv[rp] = v[rp][jj] / d;
            }
            const int floor = zero ? INT_MAX : j;
#pragma unroll
            for (int rp = 0; rp < RP; ++rp)
            {
                const bool below = pos[rp] > floor;
                const float l = below ? qv[rp] : 0.0f;
                lm[rp][jj] = l;
                v[rp][jj] = below ? qv[rp] : v[rp][jj];
#pragma unroll
                for (int c = jj + 1; c < 8; ++c) v[rp][c] = fmaf(-l, u[c], v[rp][c]);
            }
        }

        // The finished columns, rows where they started: the caller's launch moves them.
#pragma unroll
        for (int rp = 0; rp < RP; ++rp)
        {
            const int lr = rbase + rp * 64;
            float* dst = Ap + static_cast<int64_t>(8 * q) * lda + lr;
            if (lr < mp)
#pragma unroll
                for (int c = 0; c < 8; ++c)
                {
                    if (8 * q + c < wact) *dst = v[rp][c];  // uniform
                    dst += lda;
                }
        }
        const int live = 8 * (q + 1);  // first column that still lacks this block
        if (live >= wact) break;       // uniform

        // The block's pivot rows (their trailing columns as they were before the block) and
        // multipliers to LDS. Groups of cur beyond its last column are stale: they go to columns
        // that nxt's groups, stored after them, or nothing at all owns.
#pragma unroll
        for (int rp = 0; rp < RP; ++rp)
        {
            const int rel = pos[rp] - 8 * q;
            int slot0 = static_cast<unsigned>(rel) < 8u ? rel : -1;
            if (slot0 >= 0)
            {
                float4* const d4 = reinterpret_cast<float4*>(&s_l[slot0][0]);
                d4[0] = make_float4(lm[rp][0], lm[rp][1], lm[rp][2], lm[rp][3]);
                d4[1] = make_float4(lm[rp][4], lm[rp][5], lm[rp][6], lm[rp][7]);
            }
            int slot1 = slot0;
            SwapHalves(slot0, slot1);  // now per tile: both lanes of a row know its slot
#pragma unroll
            for (int t = 0; t < 2; ++t)
            {
                const int slot = t == 0 ? slot0 : slot1;
                if (slot >= 0)
                {
                    float* const row = &s_u[slot][4 * (lane >> 5)];
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        *reinterpret_cast<float4*>(row + live + 8 * k) =
                            make_float4(cur[rp][t][4 * k], cur[rp][t][4 * k + 1], cur[rp][t][4 * k + 2],
                                        cur[rp][t][4 * k + 3]);
                    if (q < 4)  // uniform
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            *reinterpret_cast<float4*>(row + 32 + 8 * k) =
                                make_float4(nxt[rp][t][4 * k], nxt[rp][t][4 * k + 1], nxt[rp][t][4 * k + 2],
                                            nxt[rp][t][4 * k + 3]);
                }
            }
        }
        if constexpr (MULTI)
        {
            // Owners publish their pivot rows, one coalesced store per 64 words; every workgroup
            // then collects all eight.
            constexpr int RW = W + 8;
            unsigned long long* const rows = p.slots + kLeafKeyWords + (q & 1) * (8 * kLeafRowStride);
            const unsigned tag = p.tagBase + static_cast<unsigned>(8 * q);
#pragma unroll
            for (int rp = 0; rp < RP; ++rp)
            {
                const int rel = pos[rp] - 8 * q;
                unsigned long long own = __ballot(static_cast<unsigned>(rel) < 8u);
                while (own != 0ull)  // uniform
                {
                    const int at = __builtin_ctzll(own);
                    own &= own - 1ull;
                    const int slot = __builtin_amdgcn_readlane(rel, at);
#pragma unroll
                    for (int cc = lane; cc < RW; cc += 64)
                        StoreTagged(rows + slot * kLeafRowStride + cc, tag,
                                    cc < W ? s_u[slot][cc] : s_l[slot][cc - W], SPREAD);
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
                    const int idx = tid + i * T, slot = idx / RW, cc = idx - slot * RW;
                    w[i] = idx < 8 * RW ? LoadWord(rows + slot * kLeafRowStride + cc)
                                        : static_cast<unsigned long long>(tag) << 32;
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
            {
#pragma unroll
                for (int i = 0; i < PER; ++i)
                {
                    const int idx = tid + i * T, slot = idx / RW, cc = idx - slot * RW;
                    if (idx < 8 * RW)
                    {
                        const float x = __uint_as_float(static_cast<unsigned>(w[i]));
                        if (cc < W)
                            s_u[slot][cc] = x;
                        else
                            s_l[slot][cc - W] = x;
                    }
                }
            }
        }
        __syncthreads();
        if (MULTI) aborted = s_gave != 0;
        // U of the trailing columns, one column per lane: cur's (from column live on) in the
        // lower half of the wave, nxt's in the upper half. A: U rows 2 s (lower half) and
        // 2 s + 1 of a chunk; B: -L likewise; both from one exchange of halves.
        float u[8];
        {
            const int col = (lane < 32 ? live : 32) + (lane & 31);
#pragma unroll
            for (int s = 0; s < 8; ++s) u[s] = s_u[s][col];
#pragma unroll
            for (int i = 1; i < 8; ++i)
#pragma unroll
                for (int s = 0; s < i; ++s) u[i] = fmaf(-s_l[i][s], u[s], u[i]);
#pragma unroll
            for (int s = 0; s < 4; ++s) SwapHalves(u[2 * s], u[2 * s + 1]);
        }
#pragma unroll
        for (int rp = 0; rp < RP; ++rp)
        {
            float bop[2][4];
#pragma unroll
            for (int s = 0; s < 4; ++s)
            {
                bop[0][s] = -lm[rp][2 * s];
                bop[1][s] = -lm[rp][2 * s + 1];
                SwapHalves(bop[0][s], bop[1][s]);
            }
            if ((q & 3) != 3)  // uniform: cur still has columns
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        cur[rp][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(u[2 * s], bop[t][s], cur[rp][t], 0, 0, 0);
            if (q < 4)  // uniform: nxt lies right of the block
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int t = 0; t < 2; ++t)
                        nxt[rp][t] = __builtin_amdgcn_mfma_f32_32x32x2f32(u[2 * s + 1], bop[t][s], nxt[rp][t], 0, 0, 0);
            if ((q & 3) == 3)  // uniform
#pragma unroll
                for (int t = 0; t < 2; ++t) cur[rp][t] = nxt[rp][t];
        }
    }

    // A wait of any workgroup that ran out spoils the whole leaf.
    if (MULTI && !aborted)
        aborted = __hip_atomic_load(p.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    if (MULTI && aborted)
    {
#pragma unroll
        for (int rp = 0; rp < RP; ++rp)
            if (rbase + rp * 64 < mp)
                for (int c = 0; c < wact; ++c) Ap[c * lda + rbase + rp * 64] = __builtin_nanf("");
    }
    if (g == 0 && wid == 0)
    {
        if (p.ipiv != nullptr && lane < wact) p.ipiv[c0 + lane] = c0 + pivots + 1;
        if (lane == 0 && zeroCol != 0 && *p.info == 0) *p.info = c0 + zeroCol;
    }
    if (!MULTI) __syncthreads();  // every source was read before any is written
    // Panel-level sources, and the leaf's moved rows: entry x < W is the row that ends at
    // position x, entry W + x the row that started there if it ends beyond the leaf's columns.
#pragma unroll
    for (int rp = 0; rp < RP; ++rp)
    {
        const int lr = rbase + rp * 64;
        if (lr < mp)
        {
            p.rowsrc[c0 + pos[rp]] = srcv[rp];
            int2* const list = reinterpret_cast<int2*>(p.moves);
            const int2 move = make_int2(c0 + pos[rp], c0 + lr);
            if (pos[rp] < wact) list[pos[rp]] = pos[rp] != lr ? move : make_int2(-1, -1);
            if (lr < wact) list[W + lr] = pos[rp] >= wact ? move : make_int2(-1, -1);
        }
    }
}

// The leaf's interchanges on the panel columns [lo, hi), its own among them: one wave per
// column gathers every moved row, then scatters.
__global__ __launch_bounds__(256) void leaf_swap_kernel(float* __restrict__ A, int lda, int lo, int hi, int wact,
                                                        const int2* __restrict__ moves, const int* __restrict__ err)
{
    const int c = lo + static_cast<int>(blockIdx.x * 4 + (threadIdx.x >> 6)), lane = threadIdx.x & 63;
    if (c >= hi || *err != 0) return;  // after a timeout the list is not complete
    float* const col = A + static_cast<size_t>(c) * lda;
    const int2 none = make_int2(-1, -1);
    const int2 m0 = lane < wact ? moves[lane] : none, m1 = lane < wact ? moves[kLeafMaxWidth + lane] : none;
    float x0 = 0.0f, x1 = 0.0f;
    if (m0.x >= 0) x0 = col[m0.y];
    if (m1.x >= 0) x1 = col[m1.y];
    if (m0.x >= 0) col[m0.x] = x0;
    if (m1.x >= 0) col[m1.x] = x1;
}

// What follows a leaf of 64 columns, in one launch: its interchanges on every panel column
// and the solve form of its unit-lower 64 x 64 diagonal block (unitlower.h). Workgroup 0 takes the
// leaf's own columns (it needs them in place for that), the others a wave per column left and
// right of it. The top 64 rows of the right columns go to ub (ld 64) instead of A: the launch
// that turns them into U writes A while its other workgroups still read them.
__global__ __launch_bounds__(256) void leaf_finish_kernel(float* __restrict__ A, int64_t lda, int j0, int c0, int wact,
                                                          int hi, const int2* __restrict__ moves,
                                                          const int* __restrict__ err, float* __restrict__ form,
                                                          float* __restrict__ ub)
{
    constexpr int W = kLeafMaxWidth;
    __shared__ __align__(16) float s_l[W * kInvStride];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    if (*err != 0) return;  // after a timeout the list is not complete
    const int2 none = make_int2(-1, -1);
    const int2 m0 = lane < wact ? moves[lane] : none, m1 = lane < wact ? moves[W + lane] : none;
    const int from = m0.x >= 0 ? m0.y : c0 + lane;  // the row that ends at position lane
    if (blockIdx.x > 0)
    {
        const int left = c0 - j0, q = static_cast<int>(blockIdx.x - 1) * 4 + wave;
        const int c = q < left ? j0 + q : c0 + wact + (q - left);
        if (c >= hi) return;
        float* const col = A + c * lda;
        float x0 = 0.0f, x1 = 0.0f;
        if (lane < wact) x0 = col[from];
        if (m1.x >= 0) x1 = col[m1.y];
        if (q >= left)
            ub[static_cast<size_t>(q - left) * W + lane] = x0;
        else if (m0.x >= 0)
            col[m0.x] = x0;
        if (m1.x >= 0) col[m1.x] = x1;
        return;
    }
    // The leaf's own columns, sixteen per wave, all loads in flight.
    float x0[16], x1[16];
#pragma unroll
    for (int k = 0; k < 16; ++k)
    {
        const int c = wave * 16 + k;
        x0[k] = x1[k] = 0.0f;
        if (c < wact && lane < wact)
        {
            const float* const col = A + (c0 + c) * lda;
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
            float* const col = A + (c0 + c) * lda;
            if (m0.x >= 0) col[m0.x] = x0[k];
            if (m1.x >= 0) col[m1.x] = x1[k];
        }
        // Rows and columns beyond the block are the identity.
        s_l[lane * kInvStride + c] = lane > c && lane < wact ? x0[k] : 0.0f;
    }
    __syncthreads();
    SolveForm64(s_l, form, tid);
}

// The panel columns right of a finished leaf: U = inv(L11) B (B: the 64 rows of ub) and
// C -= L21 U, one workgroup per 32 RT x 64 tile of C, four waves. Every workgroup forms the U
// of its 64 columns itself (40 products of 16 x 16 x 4 a wave, 0.5 us) rather than wait for a
// launch that does; those of the first tile row store it. Bound by latency for short panels
// and by the read and write of C for tall ones. The operands of the update are loaded before
// U is formed, so the launch waits for memory once; U's operands come in the layout of its products,
// so the waves meet once (order 512, on average 6.8 us; 11.4 us with three barriers).
template <int RT>
__global__ __launch_bounds__(256) void panel_update_kernel(float* __restrict__ A, int64_t lda, int m, int c0, int hi,
                                                           const float* __restrict__ form, const float* __restrict__ ub)
{
    constexpr int W = kLeafMaxWidth;
    constexpr int BS = W + 4;
    constexpr int NT = 2 * RT / 4;    // 32 x 32 tiles per wave: 1 (RT = 2) or 2 (RT = 4)
    static_assert(RT == 2 || RT == 4, "64 or 128 rows");
    __shared__ __align__(16) float s_b[W * BS];  // U, [column][row]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 31, lk = lane >> 5;
    const int col0 = static_cast<int>(blockIdx.y) * W, cols = min(W, hi - (c0 + W) - col0);
    const int row0 = c0 + W + static_cast<int>(blockIdx.x) * (32 * RT);
    float* const Ct = A + (c0 + W + col0) * lda;
    // Wave: rows wr .. wr + 31 of the tile, 32-column strips ws, ws + CT, ...
    const int row = row0 + (wave % RT) * 32 + li, ws = wave / RT;
    const bool inRow = row < m;
    // U, columns 16 wave .. 16 wave + 15.
    const int ui = lane & 15, uk = lane >> 4;
    const float* const ubc = ub + static_cast<size_t>(col0 + 16 * wave) * W;
    SolveOperands op;
    LoadOperands(form, ui, uk, op);
    f32x4 u[4];
#pragma unroll
    for (int t = 0; t < 4; ++t)
        u[t] = 16 * wave + ui < cols ? *reinterpret_cast<const f32x4*>(ubc + ui * W + 16 * t + 4 * uk)
                                     : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    float l21[32], cv[NT][16];
    const float* lp = A + c0 * lda + row + lk * lda;
#pragma unroll
    for (int t = 0; t < 32; ++t)
    {
        l21[t] = inRow ? *lp : 0.0f;
        lp += 2 * lda;
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int v = 0; v < 16; ++v)
        {
            const int c = (ws + n * (2 / NT)) * 32 + (v & 3) + 8 * (v >> 2) + 4 * lk;
            cv[n][v] = inRow && c < cols ? Ct[c * lda + row] : 0.0f;
        }
    if (__builtin_expect(SolveColumns(op, u), 1))  // uniform over the wave
    {
#pragma unroll
        for (int t = 0; t < 4; ++t) *reinterpret_cast<f32x4*>(s_b + (16 * wave + ui) * BS + 16 * t + 4 * uk) = u[t];
    }
    else
    {
        float v[16];
#pragma unroll
        for (int c = 0; c < 16; ++c) v[c] = 16 * wave + c < cols ? ubc[c * W + lane] : 0.0f;
        SubstituteColumns(A + c0 * lda + c0, lda, W, lane, v);
#pragma unroll
        for (int c = 0; c < 16; ++c) s_b[(16 * wave + c) * BS + lane] = v[c];
    }
    __syncthreads();
    if (blockIdx.x == 0)
#pragma unroll
        for (int k = 0; k < 16; ++k)
            if (16 * wave + k < cols) Ct[(16 * wave + k) * lda + c0 + lane] = s_b[(16 * wave + k) * BS + lane];
#pragma unroll
    for (int n = 0; n < NT; ++n)
    {
        const int strip = (ws + n * (2 / NT)) * 32;
        f32x16 acc;
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll
        for (int t = 0; t < 32; ++t)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(s_b[(strip + li) * BS + 2 * t + lk], l21[t], acc, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 16; ++v)
        {
            const int c = strip + (v & 3) + 8 * (v >> 2) + 4 * lk;
            if (inRow && c < cols) Ct[c * lda + row] = cv[n][v] - acc[v];
        }
    }
}

template <int NW, int RP>
hipError_t Single(const LeafArgs& a, hipStream_t stream)
{
    hipLaunchKernelGGL((panel_leaf_kernel<NW, RP, false, false>), dim3(1), dim3(64 * NW), 0, stream, a);
    return hipGetLastError();
}
}  // namespace

hipError_t LeafSingle(const LeafArgs& a, hipStream_t stream)
{
    const int mp = a.m - a.c0;
    if (mp <= 0 || mp > kLeafSingleRows || a.wact <= 0 || a.wact > kLeafMaxWidth) return hipErrorInvalidValue;
    // One row per lane and as many waves as that takes up to 512 rows (64 columns alone on the
    // GPU: 64 rows 27 us, 128 38, 256 43, 512 52; two rows per lane and half the waves 39, 51,
    // 56), two rows per lane above (1024 rows: 70 us, against 72 with 16 waves).
    if (mp <= 64) return Single<1, 1>(a, stream);
    if (mp <= 128) return Single<2, 1>(a, stream);
    if (mp <= 256) return Single<4, 1>(a, stream);
    if (mp <= 512) return Single<8, 1>(a, stream);
    return Single<8, 2>(a, stream);
}

namespace
{
// NW waves of RP x 64 rows per workgroup.
template <int NW, int RP>
hipError_t Multi(LeafArgs a, bool cooperative, bool spread, hipStream_t stream)
{
    constexpr int ROWS = 64 * NW * RP;
    const int groups = (a.m - a.c0 + ROWS - 1) / ROWS;
    if (groups > kLeafMaxGroups) return hipErrorInvalidValue;
    if (!cooperative)
    {
        hipLaunchKernelGGL((panel_leaf_kernel<NW, RP, true, false>), dim3(groups), dim3(64 * NW), 0, stream, a);
        return hipGetLastError();
    }
    // Cooperative launch: the workgroups wait for each other every column, so the runtime must
    // make all of them resident at once (it refuses a grid that cannot be).
    void* kargs[] = {&a};
    const void* fn = spread ? reinterpret_cast<const void*>(&panel_leaf_kernel<NW, RP, true, true>)
                            : reinterpret_cast<const void*>(&panel_leaf_kernel<NW, RP, true, false>);
    return hipLaunchCooperativeKernel(fn, dim3((spread ? 8 : 1) * groups), dim3(64 * NW), kargs, 0, stream);
}
}  // namespace

hipError_t LeafMulti(const LeafArgs& a, bool cooperative, bool spread, hipStream_t stream)
{
    const int mp = a.m - a.c0;
    if (mp <= 0 || mp > kLeafMultiRows || a.wact <= 0 || a.wact > kLeafMaxWidth) return hipErrorInvalidValue;
    // 256 rows per workgroup while that keeps the pollers at 32, 512 above (64 columns: 8192
    // rows 90 us against 108, 16384 rows 133 against 114). Four waves of two rows per lane take
    // 112 us there but spill: scratch must stay out of a kernel whose workgroups wait for each
    // other, since the waves with scratch that an engine keeps resident are limited.
    if (mp <= 8192) return Multi<4, 1>(a, cooperative, spread, stream);
    return Multi<8, 1>(a, cooperative, spread, stream);
}

hipError_t LeafSwap(const LeafArgs& a, hipStream_t stream)
{
    const int cols = a.panelEnd - a.j0;
    hipLaunchKernelGGL(leaf_swap_kernel, dim3((cols + 3) / 4), dim3(256), 0, stream, a.A, a.lda, a.j0, a.panelEnd, a.wact,
                       reinterpret_cast<const int2*>(a.moves), a.err);
    return hipGetLastError();
}

hipError_t LeafFinish(const LeafArgs& a, float* form, float* ub, hipStream_t stream)
{
    const int others = (a.c0 - a.j0) + (a.panelEnd - a.c0 - a.wact);
    hipLaunchKernelGGL(leaf_finish_kernel, dim3(1 + (others + 3) / 4), dim3(256), 0, stream, a.A,
                       static_cast<int64_t>(a.lda), a.j0, a.c0, a.wact, a.panelEnd,
                       reinterpret_cast<const int2*>(a.moves), a.err, form, ub);
    return hipGetLastError();
}

hipError_t PanelUpdate(const LeafArgs& a, const float* form, const float* ub, hipStream_t stream)
{
    const int cols = a.panelEnd - a.c0 - kLeafMaxWidth, rows = a.m - a.c0 - kLeafMaxWidth;
    if (a.wact != kLeafMaxWidth) return hipErrorInvalidValue;
    if (cols <= 0) return hipSuccess;
    const int nc = (cols + 63) / 64;
    // 64-row tiles while they leave the chip room (one wave then carries one 32 x 32 tile), 128
    // above, where the repeated formation of U would cost more.
    if ((rows + 63) / 64 * nc <= 512)
        hipLaunchKernelGGL(panel_update_kernel<2>, dim3(std::max(1, (rows + 63) / 64), nc), dim3(256), 0, stream, a.A,
                           static_cast<int64_t>(a.lda), a.m, a.c0, a.panelEnd, form, ub);
    else
        hipLaunchKernelGGL(panel_update_kernel<4>, dim3((rows + 127) / 128, nc), dim3(256), 0, stream, a.A,
                           static_cast<int64_t>(a.lda), a.m, a.c0, a.panelEnd, form, ub);
    return hipGetLastError();
}
}  // namespace ops
