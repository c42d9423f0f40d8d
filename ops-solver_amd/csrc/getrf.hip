// Real LU factorization (sgetrf) and the Device column-major solve, gfx950.
//
// Algorithm: right-looking blocked LU with partial pivoting, outer block width NB.
// Reference: src/sgetrf/real_lu_blocked_kernel.cpp:1469-1499 (BlockedFactorLaunch::Run:
// panel, swap+TRSM, trailing product per block). The MI355X design:
//   * panel: a sequence of register-resident leaf factorizations (leaf.hip) of up to 64
//     columns, one workgroup or, for tall panels, several.
//   * the panel is right-looking by 64 columns: after a leaf, one launch applies its interchanges
//     (a gather/scatter of the <= 128 moved rows) to all panel columns, and one solves for U
//     and updates the columns right of it. With tournament pivoting it is halved recursively.
//   * after the panel, the composed interchanges of all NB pivots are applied to every
//     column outside the panel (one coalesced gather/scatter per column), then the NB x NB
//     unit-lower TRSM on the U12 block and the MFMA trailing update A22 -= L21 * U12.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cfloat>
#include <climits>
#include <cstdlib>
#include <type_traits>

#include "leaf.h"
#include "lu_kernels.h"
#include "trs.h"
#include "trsv.h"
#include "tslu.h"
#include "wave.h"

namespace ops
{
namespace
{

constexpr int kMaxRows = kLeafMultiRows;  // largest m the register-resident leaves support

// Workspace layout (ints): [0, m) panel row sources; two moved-row lists of 4*NBMAX + 8
// (panel k uses list k % 2, so the look-ahead panel can build its list while the previous
// one is still being applied); then the global permutation (m ints).
constexpr int NBMAX = 512;
constexpr int kMovedInts = 4 * NBMAX + 8;
// After the ints (8-byte aligned): the exchange words of the multi-workgroup leaves, the
// moved-row list of the one-workgroup leaves, and the timeout flag.
constexpr size_t kSlotBytes = (256 + 2ull * 128 * 64) * sizeof(unsigned long long);
static_assert((kLeafSlotWords * 2 + kLeafMoveInts) * sizeof(int) <= kSlotBytes, "leaf words");
constexpr int kProbeGroups = 8 * 128;  // workgroups of the placement probe
constexpr size_t kFormPanelBytes = (NBMAX / 64) * 4096 * sizeof(float);  // solve forms of one panel's L11 (unitlower.h)
struct Work
{
    int* rowsrc;
    int* moved[2];
    int* movedAll;  // every panel's moved-row list (deferred interchanges), kMovedInts each
    int* composed;  // m ints: composed row map of the deferred interchanges
    int* perm;
    unsigned long long* slots;
    int* leafMoves;
    int* err;
    unsigned* epoch;       // host counter: tag base of the next multi-workgroup leaf
    float* formNode;       // tournament panels: solve forms for their internal solves
    float* panelRows;      // the same space: 64 rows of the panel columns right of a leaf (panel stream only)
    float* formPanel[2];   // solve forms of panel k's L11 in slot k % 2 (both streams read them)
    void* tslu;            // scratch of the tournament leaves
    bool tournament;       // tall leaves pivot by tournament (TsluLeaf)
};
// (sized for panels of 128 columns; they are NBMAX wide)
inline size_t MaxPanels(int m) { return static_cast<size_t>(m) / 128 + 2; }
inline size_t WorkInts(int m) { return static_cast<size_t>(m) * 3 + (2 + MaxPanels(m)) * kMovedInts; }
inline Work Layout(void* base, int m)
{
    int* p = static_cast<int*>(base);
    Work w;
    w.rowsrc = p;
    w.moved[0] = p + m;
    w.moved[1] = w.moved[0] + kMovedInts;
    w.perm = w.moved[1] + kMovedInts;
    w.composed = w.perm + m;
    w.movedAll = w.composed + m;
    uintptr_t q = reinterpret_cast<uintptr_t>(p + WorkInts(m));
    q = (q + 7) & ~static_cast<uintptr_t>(7);
    w.slots = reinterpret_cast<unsigned long long*>(q);
    w.leafMoves = reinterpret_cast<int*>(w.slots + kLeafSlotWords);
    w.err = reinterpret_cast<int*>(q + kSlotBytes);
    w.epoch = nullptr;
    q = (q + kSlotBytes + 16 + 255) & ~static_cast<uintptr_t>(255);
    w.formNode = w.panelRows = reinterpret_cast<float*>(q);
    static_assert(NBMAX * kLeafMaxWidth * sizeof(float) <= kFormPanelBytes, "panel rows");
    w.formPanel[0] = reinterpret_cast<float*>(q + kFormPanelBytes);
    w.formPanel[1] = reinterpret_cast<float*>(q + 2 * kFormPanelBytes);
    w.tslu = reinterpret_cast<void*>(q + 3 * kFormPanelBytes);
    w.tournament = false;
    return w;
}

__global__ void clear_slots_kernel(unsigned long long* slots, int words, int* err)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < words) slots[i] = 0ull;
    if (i == 0) *err = 0;
}

// Builds the list of rows moved by the whole panel (rowsrc[r] != r) and applies it to the
// global permutation. One workgroup. After a wait that ran out (*err) the workgroups of a leaf
// may disagree on the pivots, so that rowsrc need not be a permutation: the list is empty then.
__global__ __launch_bounds__(1024) void compact_moves_kernel(int m, int j0, const int* __restrict__ rowsrc,
                                                             const int* __restrict__ err, int* __restrict__ moved,
                                                             int* __restrict__ perm)
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
    const int cnt = s_count;
    if (threadIdx.x == 0) moved[0] = cnt;
    if (perm != nullptr)
    {
        int vals[2];
        int dsts[2];
#pragma unroll
        for (int q = 0; q < 2; ++q)
        {
            const int e = threadIdx.x + q * 1024;
            dsts[q] = -1;
            if (e < cnt)
            {
                dsts[q] = moved[1 + 2 * e];
                vals[q] = perm[moved[2 + 2 * e]];
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 2; ++q)
            if (dsts[q] >= 0) perm[dsts[q]] = vals[q];
    }
}

// Applies the panel's moved-row list to the columns [lo1, hi1) and [lo2, hi2): one wave64
// per column gathers every source row, then scatters.
__global__ __launch_bounds__(256) void outer_swap_kernel(float* __restrict__ A, int lda, int lo1, int hi1, int lo2,
                                                         int hi2, const int* __restrict__ moved)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int idx = blockIdx.x * 4 + wave;
    const int n1 = hi1 - lo1;
    if (idx >= n1 + (hi2 - lo2)) return;
    const int c = idx < n1 ? lo1 + idx : lo2 + (idx - n1);
    float* col = A + static_cast<size_t>(c) * lda;
    const int cnt = moved[0];
    constexpr int MAXQ = (2 * NBMAX + 63) / 64;
    float v[MAXQ];
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

// Deferred interchanges of the columns left of later panels. composed[r] <- mu(composed[r])
// for r in [lo, m), with mu the row map of one panel's moved-row list (dst -> src; every
// dst and src of that list is >= lo), built in LDS. One workgroup.
__global__ __launch_bounds__(1024) void compose_moves_kernel(int m, int lo, const int* __restrict__ moved,
                                                             int* __restrict__ composed)
{
    extern __shared__ int s_map[];  // m - lo entries
    const int len = m - lo;
    for (int r = threadIdx.x; r < len; r += blockDim.x) s_map[r] = lo + r;
    __syncthreads();
    const int cnt = moved[0];
    for (int e = threadIdx.x; e < cnt; e += blockDim.x) s_map[moved[1 + 2 * e] - lo] = moved[2 + 2 * e];
    __syncthreads();
    for (int r = threadIdx.x; r < len; r += blockDim.x) composed[lo + r] = s_map[composed[lo + r] - lo];
}

// Column c0 + blockIdx.x, rows [lo, m): row r takes the value of row composed[r], gathered
// through LDS (the whole column part first, then written back in order).
__global__ __launch_bounds__(256) void gather_rows_kernel(float* __restrict__ A, int lda, int c0, int lo, int m,
                                                          const int* __restrict__ composed)
{
    extern __shared__ float s_col[];  // m - lo values
    float* col = A + static_cast<size_t>(c0 + blockIdx.x) * lda;
    const int len = m - lo;
    for (int r = threadIdx.x; r < len; r += blockDim.x) s_col[r] = col[composed[lo + r]];
    __syncthreads();
    for (int r = threadIdx.x; r < len; r += blockDim.x) col[lo + r] = s_col[r];
}

__global__ void iota_kernel(int* p, int n)
{
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

// Panels with more active rows than this run their leaves over several workgroups;
// OPS_SOLVER_MULTI_LEAF_ROWS lowers it (a one-workgroup leaf takes at most kLeafSingleRows).
int MultiLeafRows()
{
    static const int rows = []
    {
        const char* e = std::getenv("OPS_SOLVER_MULTI_LEAF_ROWS");
        const int v = e != nullptr ? std::atoi(e) : 0;
        return v > 0 ? std::min(v, kLeafSingleRows) : kLeafSingleRows;
    }();
    return rows;
}
inline bool UseMultiLeaf(int mp) { return mp > MultiLeafRows(); }

// Multi-workgroup leaves by cooperative launch (OPS_SOLVER_LEAF_COOP, default 1).
bool LeafCooperative()
{
    static const bool on = []
    {
        const char* e = std::getenv("OPS_SOLVER_LEAF_COOP");
        return e == nullptr || std::atoi(e) != 0;
    }();
    return on;
}

// Per device: 1 when LeafSpreadProbe found the workgroups with ids = 0 mod 8 of a
// 1024-workgroup cooperative launch on one XCD, -1 when not, 0 before the probe.
constexpr int kMaxDevices = 64;
std::atomic<int> g_spreadOk[kMaxDevices];
__device__ int g_xccOfGroup[kProbeGroups];

__global__ void xcc_probe_kernel()
{
    if (threadIdx.x == 0) g_xccOfGroup[blockIdx.x] = static_cast<int>(__builtin_amdgcn_s_getreg((3 << 11) | 20) & 0xfu);
}

}  // namespace

// Full-width tall leaves run spread over 8x the grid and exchange through one XCD's L2 when
// the probe allowed it; OPS_SOLVER_LEAF_XCD=0 turns that off (read per launch).
bool LeafSpread()
{
    const char* e = std::getenv("OPS_SOLVER_LEAF_XCD");
    if (e != nullptr && std::atoi(e) == 0) return false;
    int device = 0;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices) return false;
    return g_spreadOk[device].load(std::memory_order_relaxed) == 1;
}

namespace
{

// Panels with more active rows than this take tournament leaves when the caller allows
// them; OPS_SOLVER_TSLU_ROWS overrides it.
int TsluRows()
{
    static const int rows = []
    {
        const char* e = std::getenv("OPS_SOLVER_TSLU_ROWS");
        return e != nullptr ? std::atoi(e) : 1024;
    }();
    return rows;
}
inline bool UseTslu(const Work& w, int mp) { return w.tournament && mp > TsluRows() && mp <= kTsluMaxRows; }

int LeafWidth(int mp, const Work& w) { return UseTslu(w, mp) ? kTsluWidth : kLeafMaxWidth; }

// The leaf itself; its interchanges (LeafSwap, LeafFinish) are the caller's.
hipError_t LeafColumns(LeafArgs& a, const Work& w, hipStream_t stream)
{
    const int mp = a.m - a.c0;
    // Algorithmic traffic of a leaf: its panel columns read and written once.
    ProfileScope prof(ProfileKernel::PanelLeaf, 8.0 * mp * a.wact, stream);
    if (UseMultiLeaf(mp))
    {
        // Key words carry 16-bit tags: within one factorization (slots cleared at its start)
        // the tags must not wrap. At most n / 64 <= 256 leaves (plus tournament epochs) use them.
        a.tagBase = (*w.epoch)++ * kLeafMaxWidth;
        if (a.tagBase + kLeafMaxWidth > 0xffffu) return hipErrorInvalidValue;
        return LeafMulti(a, LeafCooperative(), LeafSpread(), stream);
    }
    return LeafSingle(a, stream);
}

LeafArgs MakeLeaf(float* A, int lda, int m, int j0, int c0, int wact, int panelEnd, int pivoting, int* ipiv, int* info,
                  const Work& w)
{
    return LeafArgs{A,    lda,      m,           j0,      c0, wact,  panelEnd,   pivoting, c0 == j0, ipiv,
                    info, w.rowsrc, w.leafMoves, w.slots, 0u, w.err, SpinLimit()};
}

#define RET_IF(e)                          \
    do                                     \
    {                                      \
        hipError_t _e = (e);               \
        if (_e != hipSuccess) return _e;   \
    } while (0)

// The panel [j0, panelEnd) of rows [j0, m): per 64 columns one leaf, one launch that applies its
// interchanges to the whole panel and prepares its diagonal block, and one that updates all
// panel columns to its right. The solve forms (4096 floats per 64 columns) serve the
// U12 solves of the trailing columns afterwards.
// Right-looking by 64 columns rather than recursive: the same number of updates, each one
// launch instead of two to four, for somewhat more traffic on the panel.
hipError_t Panel(float* a, int lda, int m, int j0, int panelEnd, int pivoting, int* ipiv, int* info, const Work& wk,
                 float* forms, hipStream_t stream)
{
    for (int c0 = j0; c0 < panelEnd; c0 += kLeafMaxWidth)
    {
        const int wact = std::min(kLeafMaxWidth, panelEnd - c0);
        LeafArgs l = MakeLeaf(a, lda, m, j0, c0, wact, panelEnd, pivoting, ipiv, info, wk);
        float* const form = forms + static_cast<size_t>(c0 - j0) * kLeafMaxWidth;
        RET_IF(LeafColumns(l, wk, stream));
        RET_IF(LeafFinish(l, form, wk.panelRows, stream));
        if (c0 + wact < panelEnd) RET_IF(PanelUpdate(l, form, wk.panelRows, stream));
    }
    return hipSuccess;
}

// Tournament pivoting: factors columns [c0, c0 + w) of the outer panel [j0, panelEnd) over
// rows [c0, m); every panel column already holds the updates of the columns left of c0. The
// left half is factored first (recursively), its L11 solves the right half's top rows and an
// MFMA product updates the rest of the right half, then the right half is factored. The
// interchanges of each leaf are applied to all other panel columns.
hipError_t PanelRec(float* a, int lda, int m, int j0, int panelEnd, int c0, int w, int pivoting, int* ipiv, int* info,
                    const Work& wk, hipStream_t stream)
{
    const int W = LeafWidth(m - c0, wk);
    if (w <= W)
    {
        if (UseTslu(wk, m - c0))
        {
            ProfileScope prof(ProfileKernel::PanelLeaf, 8.0 * (m - c0) * w, stream);
            return TsluLeaf(a, lda, m, j0, c0, w, panelEnd, c0 == j0, ipiv, info, wk.rowsrc, wk.tslu, (*wk.epoch)++,
                            wk.err, stream);
        }
        LeafArgs l = MakeLeaf(a, lda, m, j0, c0, w, panelEnd, pivoting, ipiv, info, wk);
        RET_IF(LeafColumns(l, wk, stream));
        return LeafSwap(l, stream);
    }
    const int h = (w / 2 + W - 1) / W * W;  // whole leaves on the left
    RET_IF(PanelRec(a, lda, m, j0, panelEnd, c0, h, pivoting, ipiv, info, wk, stream));
    const int r = w - h;
    const float* L11 = a + static_cast<size_t>(c0) * lda + c0;
    float* B12 = a + static_cast<size_t>(c0 + h) * lda + c0;
    if (h <= 64)  // one diagonal block: a single substitution launch
        RET_IF(TrsmBlock(h, r, L11, lda, true, true, false, B12, lda, stream));
    else
    {
        RET_IF(TrsmLowerUnitForms(h, L11, lda, wk.formNode, stream));
        RET_IF(TrsmLowerUnitApply(h, r, L11, lda, wk.formNode, B12, lda, stream));
    }
    if (m - c0 - h > 0)
        RET_IF(GemmSub(m - c0 - h, r, h, a + static_cast<size_t>(c0) * lda + c0 + h, lda, 0,
                       a + static_cast<size_t>(c0 + h) * lda + c0, lda, a + static_cast<size_t>(c0 + h) * lda + c0 + h,
                       lda, Precision::FP32, stream));
    return PanelRec(a, lda, m, j0, panelEnd, c0 + h, r, pivoting, ipiv, info, wk, stream);
}

}  // namespace

size_t RealGetrfWorkspaceBytes(int m, int n)
{
    (void)n;
    // The tournament leaves' scratch only where one can run (a panel taller than TsluRows).
    return WorkInts(std::max(m, 1)) * sizeof(int) + 8 + kSlotBytes + 16 + 256 + 3 * kFormPanelBytes +
           (m > TsluRows() ? TsluScratchBytes(m) : 0);
}

int* RealGetrfErrorWord(void* work, int m) { return Layout(work, std::max(m, 1)).err; }

// ipiv == nullptr selects no pivoting. perm (optional, m ints) receives the row
// permutation P with (P A)[i] = A[perm[i]]. pack (optional, BF16 / BF16X3 trailing
// precisions): GemmPackedWorkspaceBytes(m, n, 512) bytes for the packed trailing update.
hipError_t RealGetrfPerm(int m, int n, float* a, int lda, int* ipiv, int* info, void* work, Precision trailing,
                         int* permOut, hipStream_t stream, void* pack, const LookAhead* la, bool tournament)
{
    if (m > kMaxRows) return hipErrorInvalidValue;
    Work w = Layout(work, m);
    if (permOut) w.perm = permOut;
    w.tournament = tournament && ipiv != nullptr && m > TsluRows();
    if (w.tournament) RET_IF(TsluClear(w.tslu, m, stream));
    unsigned epoch = 1;
    w.epoch = &epoch;
    FillInfo(info, 1, 0, stream);
    {
        // The multi-workgroup leaves' exchange slots (when they run) and the timeout flag
        // shared by every bounded wait of the factorization.
        const int words = UseMultiLeaf(m) ? kLeafSlotWords : 0;
        hipLaunchKernelGGL(clear_slots_kernel, dim3(std::max(1, (words + 255) / 256)), dim3(256), 0, stream, w.slots,
                           words, w.err);
    }
    const int kmax = std::min(m, n);
    if (kmax == 0) return hipGetLastError();
    const int pivoting = ipiv != nullptr;
    if (permOut) hipLaunchKernelGGL(iota_kernel, dim3((m + 255) / 256), dim3(256), 0, stream, permOut, m);
    // Panels of 512 columns at every order: a panel step is one leaf and two launches however
    // wide the panel, and each panel border costs a list of its interchanges, a swap, a solve and
    // a product more (n = 512: 759 / 698 / 575 us with 128 / 256 / 512 columns, n = 2100 4.48 /
    // 4.31 / 4.29 ms, n = 16384 FP32 101 / 87.9 / 83.6 ms, SB 93.2 / 73.7 / 67.3 ms).
    constexpr int NB = NBMAX;
    const int npanel = (kmax + NB - 1) / NB;
    // Deferred interchanges (default; OPS_SOLVER_DEFER_SWAPS=0 turns them off): the columns
    // left of a panel receive its interchanges not panel by panel but once at the end,
    // through the composition of all later panels' row maps (every panel keeps its moved-row
    // list for that): about n^2/2 gathers instead of ~2 n^2 scattered reads and writes,
    // which in column-major storage cost a cache line each and compete with the panel.
    const char* dz = std::getenv("OPS_SOLVER_DEFER_SWAPS");
    const bool defer = pivoting && npanel > 1 && (dz == nullptr || std::atoi(dz) != 0) &&
                       static_cast<size_t>(npanel) <= MaxPanels(m);
    auto moved = [&](int k) { return defer ? w.movedAll + static_cast<size_t>(k) * kMovedInts : w.moved[k & 1]; };

    // Look-ahead: the caller's stream s0 carries the critical path (the next block column's
    // update and its panel); the side stream s1 carries the rest of each trailing update.
    const bool two = la != nullptr && la->side != nullptr && npanel > 1;
    const bool split = two && la->panelStream != nullptr;  // panel path on its own CUs
    hipStream_t s0 = split ? la->panelStream : stream, s1 = two ? la->side : stream;
    if (two)
    {
        RET_IF(hipEventRecord(la->fork, stream));
        RET_IF(hipStreamWaitEvent(s1, la->fork, 0));
        if (split) RET_IF(hipStreamWaitEvent(s0, la->fork, 0));
    }

    // Panel k: factor, then list its interchanges and fold them into perm.
    auto panel = [&](int k) -> hipError_t
    {
        const int j0 = k * NB, nb = std::min(NB, kmax - j0);
        float* const forms = w.formPanel[k & 1];
        if (w.tournament)
            RET_IF(PanelRec(a, lda, m, j0, j0 + nb, j0, nb, pivoting, ipiv, info, w, s0));
        else
            RET_IF(Panel(a, lda, m, j0, j0 + nb, pivoting, ipiv, info, w, forms, s0));
        // The first panel's list serves the columns right of it and perm only.
        if (pivoting && (k > 0 || j0 + nb < n || permOut != nullptr))
            hipLaunchKernelGGL(compact_moves_kernel, dim3(1), dim3(1024), 0, s0, m, j0, w.rowsrc, w.err,
                               moved(k), permOut);
        RET_IF(hipGetLastError());
        // The U12 solves of both streams use the solve forms of this panel's L11.
        if (!w.tournament) return hipSuccess;
        return TrsmLowerUnitForms(nb, a + static_cast<size_t>(j0) * lda + j0, lda, forms, s0);
    };
    // Applies panel k to the columns [lo, hi) (interchanges, U12 solve, trailing product)
    // and, when leftSwaps, its interchanges to the columns left of the panel.
    auto update = [&](int k, int lo, int hi, bool leftSwaps, bool packed, hipStream_t st) -> hipError_t
    {
        const int j0 = k * NB, nb = std::min(NB, kmax - j0), pe = j0 + nb;
        const int cols = hi - lo, left = leftSwaps ? j0 : 0;
        if (pivoting && cols + left > 0)
            hipLaunchKernelGGL(outer_swap_kernel, dim3((cols + left + 3) / 4), dim3(256), 0, st, a, lda, 0, left, lo,
                               hi, moved(k));
        RET_IF(hipGetLastError());
        if (cols <= 0) return hipSuccess;
        RET_IF(TrsmLowerUnitApply(nb, cols, a + static_cast<size_t>(j0) * lda + j0, lda, w.formPanel[k & 1],
                                  a + static_cast<size_t>(lo) * lda + j0, lda, st));
        if (m - pe <= 0) return hipSuccess;
        const float* L21 = a + static_cast<size_t>(j0) * lda + pe;
        const float* U12 = a + static_cast<size_t>(lo) * lda + j0;
        float* A22 = a + static_cast<size_t>(lo) * lda + pe;
        if (packed && pack != nullptr)
            return GemmSubPacked(m - pe, cols, nb, L21, lda, U12, lda, A22, lda, trailing, pack, st);
        return GemmSub(m - pe, cols, nb, L21, lda, 0, U12, lda, A22, lda, trailing, st);
    };

    RET_IF(panel(0));
    if (two) RET_IF(hipEventRecord(la->panel[0], s0));
    for (int k = 0; k < npanel; ++k)
    {
        const int pe = std::min(kmax, (k + 1) * NB);
        const int nbNext = k + 1 < npanel ? std::min(NB, kmax - pe) : 0;
        // Bulk of the trailing update (s1): everything right of the next block column.
        if (two) RET_IF(hipStreamWaitEvent(s1, la->panel[k & 1], 0));
        RET_IF(update(k, pe + nbNext, n, !defer, true, s1));
        if (two) RET_IF(hipEventRecord(la->bulk[k & 1], s1));
        // Critical path (s0): the next block column, then its panel.
        if (nbNext > 0)
        {
            if (two && k > 0) RET_IF(hipStreamWaitEvent(s0, la->bulk[(k - 1) & 1], 0));
            RET_IF(update(k, pe, pe + nbNext, false, false, s0));
            RET_IF(panel(k + 1));
            if (two) RET_IF(hipEventRecord(la->panel[(k + 1) & 1], s0));
        }
    }
    if (two) RET_IF(hipStreamWaitEvent(s0, la->bulk[(npanel - 1) & 1], 0));
    if (defer)
    {
        // Backward over the panels: composed = mu_{p+1} o ... o mu_last, then panel p's
        // columns gather their rows [(p+1) NB, m) through it.
        hipLaunchKernelGGL(iota_kernel, dim3((m + 255) / 256), dim3(256), 0, s0, w.composed, m);
        for (int p = npanel - 2; p >= 0; --p)
        {
            const int lo = (p + 1) * NB, nb = std::min(NB, kmax - p * NB);
            if (lo >= m) continue;
            const size_t lds = static_cast<size_t>(m - lo) * sizeof(int);
            hipLaunchKernelGGL(compose_moves_kernel, dim3(1), dim3(1024), lds, s0, m, lo, moved(p + 1), w.composed);
            hipLaunchKernelGGL(gather_rows_kernel, dim3(nb), dim3(256), lds, s0, a, lda, p * NB, lo, m, w.composed);
        }
        RET_IF(hipGetLastError());
    }
    FoldWaitError(w.err, info, s0);
    if (split)
    {
        RET_IF(hipEventRecord(la->join, s0));
        RET_IF(hipStreamWaitEvent(stream, la->join, 0));
    }
    return hipGetLastError();
}

hipError_t RealGetrf(int m, int n, float* a, int lda, int* ipiv, int* info, void* work, Precision trailing,
                     hipStream_t stream)
{
    return RealGetrfPerm(m, n, a, lda, ipiv, info, work, trailing, nullptr, stream, nullptr, nullptr);
}

// ---------------------------------------------------------------------------------------
// getrs on Device column-major data.
// ---------------------------------------------------------------------------------------
namespace
{
// ipiv (LAPACK interchange sequence) -> permutation, perm[i] = source row of row i of P*B.
// With s_k the interchange of rows k and ipiv[k] - 1 (applied for k = 0, 1, ...), row i of
// P*B comes from row s_0(s_1(... s_{n-1}(i))): one lane per position traces it backward
// through the interchanges, ipiv staged in LDS (padded to a multiple of 4 with identities,
// read four at a time as broadcasts). An out-of-range entry (and, with CLAMP_BELOW, one
// pointing above its own row) is taken as no interchange.
template <bool CLAMP_BELOW>
__global__ __launch_bounds__(64) void ipiv_to_perm_kernel(int n, const int* __restrict__ ipiv, int* __restrict__ perm)
{
    extern __shared__ int s_piv[];
    const int n4 = (n + 3) & ~3;
#pragma unroll 16  // 16 loads per lane in flight
    for (int k = threadIdx.x; k < n4; k += 64)
    {
        int p = k < n ? ipiv[k] - 1 : k;
        if (p < 0 || p >= n || (CLAMP_BELOW && p < k)) p = k;
        s_piv[k] = p;
    }
    __syncthreads();
    const int i = blockIdx.x * 64 + static_cast<int>(threadIdx.x);
    int x = i;
    const int4* q = reinterpret_cast<const int4*>(s_piv);
#pragma unroll 4
    for (int k = n4 - 4; k >= 0; k -= 4)
    {
        const int4 p = q[k >> 2];
        x = x == k + 3 ? p.w : (x == p.w ? k + 3 : x);
        x = x == k + 2 ? p.z : (x == p.z ? k + 2 : x);
        x = x == k + 1 ? p.y : (x == p.y ? k + 1 : x);
        x = x == k ? p.x : (x == p.x ? k : x);
    }
    if (i < n) perm[i] = x;
}

// dst(:, c) = src(perm, c) (gather) or dst(perm, c) = src(:, c) (scatter).
template <bool GATHER>
__global__ void permute_rows_kernel(int n, int nrhs, const int* __restrict__ perm, const float* __restrict__ src,
                                    int lds, float* __restrict__ dst, int ldd)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int c = blockIdx.y;
    if (i >= n || c >= nrhs) return;
    const int p = perm ? perm[i] : i;
    if (GATHER)
        dst[static_cast<size_t>(c) * ldd + i] = src[static_cast<size_t>(c) * lds + p];
    else
        dst[static_cast<size_t>(c) * ldd + p] = src[static_cast<size_t>(c) * lds + i];
}

int SolveBlock(int n) { return n >= 4096 ? 256 : 128; }
}  // namespace

namespace
{
// Chained substitutions (trs.hip) or, for many right-hand sides of a large system, blocked ones.
// Microseconds, blocked and chained: n = 100, 1 rhs 72 and 24, 8192 rhs 101 and 55; n = 1000, 33 rhs 842
// and 251, 8192 1252 and 500; n = 4096, 33 rhs 3740 and 1039, 2048 4989 and 1615, 8192 8638 and 5103
// (transposed 10769 and 5374); n = 16384, 256 rhs 20061 and 5544. Up to 4096 the chain won at every
// number of right-hand sides, above it was measured to 256. Blocked also where the chain's
// padding to 64 rows would waste memory, and for the few problems that the no-allocation entry
// point takes and whose chain does not fit its array (it promises the results of the
// allocating one).
bool UseTrs(int n, int nrhs)
{
    if (n > 4096 && nrhs > 256) return false;
    if (n < 16 && nrhs > 1024) return false;
    return RealGetrsStagingBytes(n, nrhs) > ACLSOLVER_NOALLOC_SCRATCH_BYTES ||
           TrsWorkspaceBytes(n, nrhs) <= kNoAllocArrayBytes;
}
}  // namespace

// The term of the former chained solve of one right-hand side stays: the size is documented.
size_t RealGetrsStagingBytes(int n, int nrhs)
{
    const size_t vectors =
        ((static_cast<size_t>(n) * std::max(nrhs, 1) + static_cast<size_t>(n) + 64) * sizeof(float) + 255) / 256 * 256;
    return vectors + TrsvChainStateBytes(std::max(n, 1));
}

size_t RealGetrsWorkspaceBytes(int n, int nrhs)
{
    return UseTrs(n, nrhs) ? TrsWorkspaceBytes(n, nrhs) : RealGetrsStagingBytes(n, nrhs);
}

// Triangular solves on a column-major n x nrhs block X (ldx) with packed LU factors.
hipError_t RealLuSolveInPlace(int trans, int n, int nrhs, const float* lu, int lda, float* x, int ldx,
                              hipStream_t stream)
{
    const int NBS = SolveBlock(n);
    if (trans == 0)
    {
        for (int k = 0; k < n; k += NBS)  // L y = b (unit lower)
        {
            const int kb = std::min(NBS, n - k);
            RET_IF(TrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, true, true, false, x + k, ldx,
                             stream));
            if (n - k - kb > 0)
                RET_IF(GemmSub(n - k - kb, nrhs, kb, lu + static_cast<size_t>(k) * lda + k + kb, lda, 0, x + k, ldx,
                               x + k + kb, ldx, Precision::FP32, stream));
        }
        for (int k = ((n - 1) / NBS) * NBS; k >= 0; k -= NBS)  // U x = y
        {
            const int kb = std::min(NBS, n - k);
            RET_IF(TrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, false, false, false, x + k, ldx,
                             stream));
            if (k > 0)
                RET_IF(GemmSub(k, nrhs, kb, lu + static_cast<size_t>(k) * lda, lda, 0, x + k, ldx, x, ldx,
                               Precision::FP32, stream));
        }
    }
    else
    {
        for (int k = 0; k < n; k += NBS)  // U^T w = b (lower, non-unit)
        {
            const int kb = std::min(NBS, n - k);
            RET_IF(TrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, false, false, true, x + k, ldx,
                             stream));
            if (n - k - kb > 0)  // x[k+kb:] -= U[k:k+kb, k+kb:]^T w[k:k+kb]
                RET_IF(GemmSub(n - k - kb, nrhs, kb, lu + static_cast<size_t>(k + kb) * lda + k, lda, 1, x + k, ldx,
                               x + k + kb, ldx, Precision::FP32, stream));
        }
        for (int k = ((n - 1) / NBS) * NBS; k >= 0; k -= NBS)  // L^T z = w (upper, unit)
        {
            const int kb = std::min(NBS, n - k);
            RET_IF(TrsmBlock(kb, nrhs, lu + static_cast<size_t>(k) * lda + k, lda, true, true, true, x + k, ldx,
                             stream));
            if (k > 0)  // x[0:k] -= L[k:k+kb, 0:k]^T z[k:k+kb]
                RET_IF(GemmSub(k, nrhs, kb, lu + k, lda, 1, x + k, ldx, x, ldx, Precision::FP32, stream));
        }
    }
    return hipGetLastError();
}

hipError_t IpivToPerm(int n, const int* ipiv, int* perm, hipStream_t stream, bool clampBelow)
{
    if (n > kMaxRows) return hipErrorInvalidValue;
    if (n <= 0) return hipSuccess;
    const dim3 grid((n + 63) / 64);
    const size_t lds = static_cast<size_t>((n + 3) & ~3) * sizeof(int);
    if (clampBelow)
        hipLaunchKernelGGL(ipiv_to_perm_kernel<true>, grid, dim3(64), lds, stream, n, ipiv, perm);
    else
        hipLaunchKernelGGL(ipiv_to_perm_kernel<false>, grid, dim3(64), lds, stream, n, ipiv, perm);
    return hipGetLastError();
}

hipError_t PermuteRows(bool gather, int n, int nrhs, const int* perm, const float* src, int lds, float* dst, int ldd,
                       hipStream_t stream)
{
    dim3 grid((n + 255) / 256, nrhs);
    if (gather)
        hipLaunchKernelGGL(permute_rows_kernel<true>, grid, dim3(256), 0, stream, n, nrhs, perm, src, lds, dst, ldd);
    else
        hipLaunchKernelGGL(permute_rows_kernel<false>, grid, dim3(256), 0, stream, n, nrhs, perm, src, lds, dst, ldd);
    return hipGetLastError();
}

namespace
{
// dst (column-major, ldd) <- src (row-major rows x cols, lds); 32x32 tiles through LDS so
// both the read and the write are coalesced.
__global__ __launch_bounds__(256) void transpose_rm_kernel(int rows, int cols, const float* __restrict__ src,
                                                           int64_t lds, float* __restrict__ dst, int64_t ldd)
{
    __shared__ float tile[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int q = ty; q < 32; q += 8)
    {
        const int r = r0 + q, c = c0 + tx;
        if (r < rows && c < cols) tile[q][tx] = src[r * lds + c];
    }
    __syncthreads();
    for (int q = ty; q < 32; q += 8)
    {
        const int c = c0 + q, r = r0 + tx;
        if (r < rows && c < cols) dst[c * ldd + r] = tile[tx][q];
    }
}
}  // namespace

hipError_t TransposeRM(int rows, int cols, const float* src, int64_t lds, float* dst, int64_t ldd, hipStream_t stream)
{
    dim3 grid((cols + 31) / 32, (rows + 31) / 32);
    hipLaunchKernelGGL(transpose_rm_kernel, grid, dim3(256), 0, stream, rows, cols, src, lds, dst, ldd);
    return hipGetLastError();
}

hipError_t RealGetrs(int trans, int n, int nrhs, const float* lu, int lda, const int* ipiv, float* b, int ldb,
                     void* work, hipStream_t stream, int* info, bool chain)
{
    if (n <= 0 || nrhs <= 0) return hipSuccess;
    if (chain && UseTrs(n, nrhs)) return TrsSolve(trans, n, nrhs, lu, lda, ipiv, b, ldb, info, work, stream);
    if (info != nullptr) FillInfo(info, 1, 0, stream);
    float* x = static_cast<float*>(work);
    int* perm = reinterpret_cast<int*>(x + static_cast<size_t>(n) * nrhs);
    if (ipiv) RET_IF(IpivToPerm(n, ipiv, perm, stream));
    const int* p = ipiv ? perm : nullptr;
    if (trans == 0)
    {
        RET_IF(PermuteRows(true, n, nrhs, p, b, ldb, x, n, stream));
        RET_IF(RealLuSolveInPlace(0, n, nrhs, lu, lda, x, n, stream));
        // copy back
        RET_IF(PermuteRows(true, n, nrhs, nullptr, x, n, b, ldb, stream));
    }
    else
    {
        RET_IF(PermuteRows(true, n, nrhs, nullptr, b, ldb, x, n, stream));
        RET_IF(RealLuSolveInPlace(1, n, nrhs, lu, lda, x, n, stream));
        RET_IF(PermuteRows(false, n, nrhs, p, x, n, b, ldb, stream));
    }
    return hipGetLastError();
}

// Records the XCD of every workgroup of a 1024-workgroup cooperative launch and allows the
// spread tall leaves on this device when those with ids = 0 mod 8 share one XCD. Runs once
// per device (the device current), synchronously on the null stream; two threads probing
// one device at once both store the same result.
void LeafSpreadProbe(int device)
{
    if (device < 0 || device >= kMaxDevices || g_spreadOk[device].load() != 0) return;
    constexpr int G = kProbeGroups;
    int result = -1;
    if (hipLaunchCooperativeKernel(reinterpret_cast<const void*>(&xcc_probe_kernel), dim3(G), dim3(64), nullptr, 0,
                                   nullptr) == hipSuccess &&
        hipStreamSynchronize(nullptr) == hipSuccess)
    {
        int h[G];
        if (hipMemcpyFromSymbol(h, HIP_SYMBOL(g_xccOfGroup), sizeof(h)) == hipSuccess)
        {
            result = 1;
            for (int k = 1; k < G / 8; ++k)
                if (h[8 * k] != h[0]) result = -1;
        }
    }
    (void)hipGetLastError();
    g_spreadOk[device].store(result);
}

}  // namespace ops
