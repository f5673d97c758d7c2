/*
 * loop.hip -- the Newton-Raphson loop driven from the device.
 *
 * The host-driven loop (solver.hip) reads the active-leaf count, the list total and the
 * counters back after every pass and sizes each launch from them.  Here every kernel of a
 * pass takes its counts from a small control block in device memory (PassCtl), so a pass is
 * a fixed sequence of launches: K passes are captured once in a HIP graph and the graph is
 * replayed until the loop is over, one host synchronisation per replay.  The density kernel
 * runs as a persistent grid whose wavefronts pull work items from the pass's queue: the
 * costliest items first, cut into sub-items where one would end the pass alone, then the rest in
 * the leaves' Hilbert order, so neighbouring items share j-particles in L2.
 *
 * One pass (the pass of src/density_base.cu:782-887), 9 launches:
 *   lists       count walk (2), scan with the longest list and the capacity check, fill walk (2):
 *               the tight gather lists
 *   items       work items of sparse leaves; the heavy items to the queue's head
 *   density     both item forms as persistent grids; the one not selected exits at once
 *   compaction  the active leaves in place, hmax and hRem of the ones that stay, their item
 *               offsets; its last block writes the log record and sets up the next pass
 *               (halt: no active leaf, or the NR pass cap reached)
 * Most of a pass's launches last a few microseconds whatever they do: with a launch per step of
 * this list (22) the lists, items and compaction of a pass took 64 us on the 16-wide lattice (5,760
 * particles), now 51; 9.2 ms instead of 10.4 for the 21 passes of a 12-set ensemble.
 *
 * A pass whose lists would overflow the list buffer stops at the scan with nothing changed;
 * the host grows the buffer, captures again and replays.  The items of a pass, their lists
 * and every pair are those of the host-driven pass; only the order in which wavefronts take
 * items differs, and no item's result depends on it.  With no item cut (split_len = 0) h, rho and
 * d(rho)/d(h) are bit-identical to the host-driven loop's; the parts of a cut item add their FP64
 * sums in another order.
 */
#include "density.hpp"
#include "lookback.hpp"
#include "loop.hpp"
#include "tile.hpp"
#include "tree.hpp"

#include <algorithm>
#include <cstring>
#include <vector>

namespace csph
{

__device__ inline int iceilDev(int a, int b) { return (a + b - 1) / b; }

__device__ inline unsigned long long clockNow() { return (unsigned long long)wall_clock64(); }

constexpr int kItemThreads = 256;
constexpr int kHeavySpan   = 2;   // heavy: a list at least 1/4 as long as the longest (in buckets)
constexpr int kHeavyMean   = 8;   // ... and at least 8 times the mean list length of the pass
constexpr int kFewItems    = 4096;   // a pass of at most this many items leaves most of the chip idle
constexpr double   kHeadDiv = 8, kHeadMean = 2;   // heavy: a share's eighth, twice the mean cost (queueItem)
constexpr uint32_t kMinPart = 32;    // list entries of a sub-item, at least
constexpr uint32_t kTileParticles = 5;   // particles of a leaf to a sub-item that sweeps every n-th tile

struct ItemArgs
{
    PassCtl*        C;
    const int*      leaves;
    const uint32_t* layout;
    const uint8_t*  state;
    int             sparse;
    const uint32_t* itemOff;
    const uint32_t* leafRem;    // by position: the leaf's particles still to evaluate
    const uint32_t* jCount;
    int*            itemPos;
    int*            itemPart;
    int*            qOrder;   // nullptr: no heavy items
    uint8_t*        qFlag;
    uint32_t*       qSub;
    int             splitLen;   // list length beyond which heavy items are split, 0: none are; < 0: by the pass's load
    int             waves;      // of the density kernel's grid
    int             mixed;
    int             maxParts;   // slots of the sub-items' partials
};

// What makes an item of a pass heavy.
struct QueueRule
{
    int                cut;        // a list in this bucket or above ...
    unsigned long long heavyLen;   // ... with at least this many entries,
    uint32_t           cost;       // or a cost above this;
    uint32_t           part;       // the cost of a sub-item
    int                range;      // mixed whole leaves: list ranges for lists in this longBin or above
    uint32_t           rangeLen;   // list entries of a sub-item that is a range by length
};

// Work queue: the heavy items first (qOrder[0, qBucket[1]), in no particular order: started last
// they would be the pass's tail), then every item in its own order (the leaves' Hilbert order, which
// keeps the j-particles that neighbouring items share in L2), skipping the heavy ones (qFlag).
//
// An item that costs a good part of its wavefront's share of the pass, taken late, or more than the
// share, ends the pass alone: the first pass of a disc of 250k particles (14,000 items, 2.7 a wavefront)
// ran 2.1 ms with 0.9 ms of work a wavefront.  So an item goes to the head from an eighth of the share
// on, but not below twice the mean (the order of the rest is worth keeping: lists of neighbours are in
// L2), or half the share where that is less; and it is cut into sub-items of half a share, up to
// kMaxSub: list ranges of one particle's items and of FP64 whole leaves, every n-th tile of mixed whole
// leaves (each sub-item stages all of them, so n is bounded by the particles that the staging serves).
// Density kernels of a solve without and with it: that disc (mixed) 13.3 and 8.4 ms, 12 sets of
// 10k-53k particles 4.1 and 3.3 ms, a 2M-particle mixture 169 and 161 ms, a step of 1M 3.7 and 2.4 ms;
// items all alike (lattices) are not touched.
//
// Called by whole wavefronts (`is`: the lane has an item): one atomic per wavefront and counter.
// `batch`: one particle, or a leaf of at most 64 particles, rem of them still to evaluate.
__device__ inline void queueItem(const ItemArgs& A, const QueueRule& R, bool is, int k, uint32_t len, bool onePart,
                                 bool batch, uint32_t rem)
{
    PassCtl* const C = A.C;
    const bool longest = listBucket(len) >= R.cut && (unsigned long long)len >= R.heavyLen;
    const uint32_t cost = itemCost(len, onePart ? 1u : rem);
    uint32_t want = 0u;      // entries at the queue's head
    bool byTiles = false, range = false;
    if (is && (longest || cost > R.cost))
    {
        want = 1u;
        if (A.splitLen > 0)
        {
            if (batch && longest && len > R.rangeLen) want = (len + R.rangeLen - 1u) / R.rangeLen;
        }
        else if (A.splitLen < 0 && batch)
        {
            range = A.mixed && !onePart && longest && len > (uint32_t)kSplitLen && longBin(len) >= R.range;
            if (range) want = (len + (uint32_t)kSplitLen - 1u) / (uint32_t)kSplitLen;
            else       want = min((cost + R.part - 1u) / R.part, max(len / kMinPart, 1u));
            if (A.mixed && !onePart && !range)
            {
                byTiles = true;
                want = min(want, max(rem / kTileParticles, 1u));
            }
        }
        want = min(want, (uint32_t)kMaxSub);
    }
    if (!ballot64(want > 0u))
    {
        if (is) A.qFlag[k] = 0;
        return;
    }
    uint32_t part0 = 0u;
    if (ballot64(want > 1u))
    {
        const uint32_t parts = want > 1u ? want : 0u, incl = waveInclusiveScan(parts);
        uint32_t p = 0;
        if (laneId() == kWave - 1) p = atomicAdd(&C->nParts, incl);
        part0 = (uint32_t)__shfl((int)p, kWave - 1, kWave) + incl - parts;
        if (part0 + parts > (uint32_t)A.maxParts) want = min(want, 1u);   // (never: QueueRule)
        const uint64_t m = ballot64(want > 1u);
        if (laneId() == 0 && m) atomicAdd(&C->nSplit, (uint32_t)__popcll(m));
    }
    const uint32_t incl = waveInclusiveScan(want);
    uint32_t base = 0;
    if (laneId() == kWave - 1) base = atomicAdd(&C->qBucket[1], incl);
    base = (uint32_t)__shfl((int)base, kWave - 1, kWave) + incl - want;
    if (is) A.qFlag[k] = want > 0u ? 1 : 0;
    for (uint32_t s = 0; s < want; ++s)
    {
        A.qOrder[base + s] = k;
        if (A.qSub) A.qSub[base + s] = want > 1u ? packSub(s, want, byTiles, part0) : 0u;
    }
}

// Items of the pass: whole leaves are items already (item a = position a, a thread each to sort
// out the heavy ones); in a pass with per-particle items a wavefront per leaf writes the leaf's
// items at itemOff[a]: (a, -1) for a whole leaf, else (a, p) for every particle p in state != 0, in
// particle order (the count of itemsOf).
__global__ __launch_bounds__(kItemThreads) void itemsKernel(ItemArgs A)
{
    const PassCtl* C = A.C;
    if (C->skip) return;
    const int n = (int)C->nAL;
    const unsigned long long mean = n ? C->listNeed / (unsigned long long)n : 0ull;
    QueueRule R;
    R.cut = (int)C->qBucket[0] - kHeavySpan;
    // heavy: among the longest lists and, unless the pass has too few items to fill the chip,
    // well above the mean
    R.heavyLen = (int)C->nItems <= kFewItems ? 0ull : kHeavyMean * mean;
    R.cost = R.part = 0x7FFFFFFFu;
    R.range = kLongBins;
    R.rangeLen = (uint32_t)max(A.splitLen, 1);
    // An item cut into parts of cost p has fewer than 2 cost / p of them (one with a single part is not
    // cut): with p at least 2 / slots of the cost of all items, the slots are enough whatever the items are.
    // Which ones are cut then does not depend on the order in which wavefronts get here.
    const unsigned long long costs = C->itemCosts;
    if (A.splitLen > 0)
    {
        const unsigned long long entries = costs / (kStageCost + 1u);   // at least those of all items' lists
        R.rangeLen = (uint32_t)min(max((unsigned long long)R.rangeLen, 2ull * entries / (unsigned long long)A.maxParts + 1ull),
                                   0x7FFFFFFFull);
    }
    if (A.splitLen < 0)
    {
        // list ranges of the longest lists, by whole bins, up to kMaxSplit items: lane l counts the l-th bin
        // from the longest list's bucket down (kHeavySpan + 1 buckets: all that can be heavy)
        int slots = A.maxParts;
        if (A.mixed)
        {
            const uint32_t most = (uint32_t)min(kMaxSplit, A.maxParts / (2 * kMaxSub));
            const uint32_t least = (uint32_t)min(max(R.heavyLen, (unsigned long long)kSplitLen), 0xFFFFFFFFull);
            const int bin = ((int)C->qBucket[0] - 11) * 8 + 7 - laneId();
            const bool in = laneId() < (kHeavySpan + 1) * 8 && bin >= longBin(least);
            const uint32_t above = waveInclusiveScan(in ? C->nLong[bin] : 0u);
            const uint64_t fit = ballot64(in && above <= most);   // a run of lanes from 0 on
            if (fit) R.range = ((int)C->qBucket[0] - 11) * 8 + 8 - __popcll(fit);
            slots -= (int)most * kMaxSub;
        }
        const unsigned long long leastPart = 2ull * costs / (unsigned long long)slots + 1ull;
        // mean cost of the pass's items and the share of one of the grid's wavefronts
        const double mc = C->perParticle ? (double)itemCost((uint32_t)mean, 1u)
                                         : (double)mean * ((double)kStageCost + (double)C->nRem / (double)max(n, 1));
        const double share = mc * (double)C->nItems / (double)max(A.waves, 1);
        R.cost = (uint32_t)fmin(fmax(share / kHeadDiv, fmin(kHeadMean * mc, share / 2)), 2e9);
        R.part = (uint32_t)min(max((unsigned long long)fmin(fmax(share / 2, 8.0), 2e9), leastPart), 0x7FFFFFFFull);
    }
    if (!C->perParticle)
    {
        if (!A.qOrder) return;
        for (int a0 = blockIdx.x * kItemThreads; a0 < n; a0 += gridDim.x * kItemThreads)
        {
            const int a = a0 + threadIdx.x, l = a < n ? A.leaves[a] : 0;
            const bool batch = A.layout[l + 1] - A.layout[l] <= (uint32_t)kWave;
            queueItem(A, R, a < n, a, a < n ? A.jCount[a] : 0u, false, batch, a < n ? A.leafRem[a] : 0u);
        }
        return;
    }
    for (int a = blockIdx.x * (kItemThreads / kWave) + (threadIdx.x >> 6); a < n; a += gridDim.x * (kItemThreads / kWave))
    {
        const int l = A.leaves[a];
        const uint32_t p0 = A.layout[l], p1 = A.layout[l + 1], len = A.jCount[a], rem = A.leafRem[a];
        uint32_t o = A.itemOff[a];
        if (rem > (uint32_t)A.sparse)
        {
            const bool one = laneId() == 0;
            if (one)
            {
                A.itemPos[o] = a;
                A.itemPart[o] = -1;
            }
            if (A.qOrder) queueItem(A, R, one, (int)o, len, false, p1 - p0 <= (uint32_t)kWave, rem);
            continue;
        }
        for (uint32_t q0 = p0; q0 < p1; q0 += kWave)
        {
            const uint32_t p = q0 + laneId();
            const bool live = p < p1 && A.state[p] != 0;
            const uint64_t m = ballot64(live);
            const uint32_t k = o + (uint32_t)__popcll(m & lanemaskLt());
            if (live)
            {
                A.itemPos[k] = a;
                A.itemPart[k] = (int)p;
            }
            if (A.qOrder) queueItem(A, R, live, (int)k, len, true, true, rem);
            o += (uint32_t)__popcll(m);
        }
    }
}

struct CompactArgs
{
    PassCtl*        C;
    int*            leaves;
    uint32_t*       itemOff;
    uint32_t*       leafRem;
    const uint32_t* layout;
    const uint8_t*  state;
    const double*   h;
    double*         hmaxLeaf;
    double*         hRem;
    unsigned long long* counters;
    PassLogDev*     log;
    int*            heavyN;
    uint32_t*       qHead;
    ScanHead*       head;
    unsigned long long* words;      // look-back words: active leaves, then (wordCap on) work items
    int             wordCap;
    int             logCap, sparse, maxIter, tailLeaves, flat;
};

constexpr int kCompactThreads = 1024;
constexpr int kCompactTile    = 256;                           // leaves per block
constexpr int kCompactLanes   = 16;                            // lanes per leaf
constexpr int kCompactGroups  = kCompactThreads / kCompactLanes;

// The end of a pass and the start of the next: for every active leaf, whether it has a particle left
// in state != 0, its work items, and hmax / hRem (max finite h of all its particles, of those in
// state != 0: the h of the next pass's lists); the leaves that stay move to their new positions in
// place (a tile writes below its own start, where earlier tiles have read what they need before
// they published; its own leaves it has read itself).  INIT: leaf a is a, the loop's first pass.
// The last block to finish logs the pass and sets up the next one.
template<bool INIT>
__global__ __launch_bounds__(kCompactThreads) void compactKernel(CompactArgs A)
{
    __shared__ int      leafOf[kCompactTile];
    __shared__ uint32_t lo[kCompactTile], hi[kCompactTile], left[kCompactTile];
    __shared__ uint32_t tot[2][kCompactTile / kWave], before[2];
    __shared__ unsigned long long red[kNumCounters][4];
    __shared__ uint32_t shTile, shEpoch, shIter, shRem, shLast;
    PassCtl* const C = A.C;
    if (C->skip) return;
    const int n = (int)C->nAL;
    const int tiles = max(iceilDev(n, kCompactTile), 1);
    if ((int)blockIdx.x >= tiles) return;
    const int t = threadIdx.x;
    if (t == 0)
    {
        if (!INIT && blockIdx.x == 0) C->tEnd = clockNow();   // the density kernel has ended
        shTile = tiles > 1 ? atomicAdd(&A.head->ticket, 1u) : 0u;
        shEpoch = A.head->epoch;
        shIter = 0u;
        shRem = 0u;
    }
    __syncthreads();
    const int tile = (int)shTile, a0 = tile * kCompactTile, held = min(kCompactTile, n - a0);
    if (t < kCompactTile)
    {
        const int l = t < held ? (INIT ? a0 + t : A.leaves[a0 + t]) : -1;
        leafOf[t] = l;
        lo[t] = l >= 0 ? A.layout[l] : 0u;
        hi[t] = l >= 0 ? A.layout[l + 1] : 0u;
    }
    __syncthreads();
    {
        const int sub = t % kCompactLanes;
        uint32_t it = 0;   // particles in state 1 seen by this lane
#pragma unroll
        for (int r = 0; r < kCompactTile / kCompactGroups; ++r)
        {
            const int e = t / kCompactLanes + r * kCompactGroups;
            const uint32_t p0 = lo[e], p1 = hi[e];
            uint32_t rem = 0;
            double m = 0.0, mr = 0.0;
            for (uint32_t p = p0 + sub; p < p1; p += kCompactLanes)
            {
                const uint8_t s = A.state[p];
                const double v = A.h[p];
                it += s == 1 ? 1u : 0u;
                rem += s ? 1u : 0u;
                if (isfinite(v))
                {
                    m = fmax(m, v);
                    if (s != 0) mr = fmax(mr, v);
                }
            }
            for (int off = 1; off < kCompactLanes; off <<= 1)
            {
                rem += __shfl_xor(rem, off, kCompactLanes);
                m = fmax(m, __shfl_xor(m, off, kCompactLanes));
                mr = fmax(mr, __shfl_xor(mr, off, kCompactLanes));
            }
            if (sub == 0)
            {
                left[e] = rem;
                if (rem)
                {
                    atomicAdd(&shRem, rem);
                    A.hmaxLeaf[leafOf[e]] = m;
                    A.hRem[leafOf[e]] = mr;
                }
            }
        }
        it = waveReduceSum(it);
        if (laneId() == 0 && it) atomicAdd(&shIter, it);
    }
    __syncthreads();
    const int w = t >> 6;
    uint32_t keep = 0, items = 0, inclK = 0, inclI = 0;
    if (t < kCompactTile)
    {
        keep = left[t] ? 1u : 0u;
        items = itemsOf(left[t], A.sparse);
        inclK = waveInclusiveScan(keep);
        inclI = waveInclusiveScan(items);
        if (laneId() == kWave - 1)
        {
            tot[0][w] = inclK;
            tot[1][w] = inclI;
        }
    }
    __syncthreads();
    if (w < 2)
    {
        uint32_t own = 0;
        for (int k = 0; k < kCompactTile / kWave; ++k) own += tot[w][k];
        const uint32_t b = tiles > 1 ? tilePrefix(A.words + (size_t)w * A.wordCap, tile, shEpoch, own) : 0u;
        if (laneId() == 0) before[w] = b;
    }
    __syncthreads();
    if (t < kCompactTile && keep)
    {
        uint32_t k = before[0] + inclK - 1u, o = before[1] + inclI - items;
        for (int q = 0; q < w; ++q)
        {
            k += tot[0][q];
            o += tot[1][q];
        }
        A.leaves[k] = leafOf[t];
        A.itemOff[k] = o;
        A.leafRem[k] = left[t];
    }
    if (t == 0)
    {
        if (shIter) atomicAdd(&C->accIterating, (unsigned long long)shIter);
        if (shRem) atomicAdd(&C->accRem, (unsigned long long)shRem);
        __threadfence();
        shLast = (tiles == 1 || atomicAdd(&A.head->done, 1u) == (uint32_t)tiles - 1u) ? 1u : 0u;
    }
    __syncthreads();
    if (!shLast) return;

    // ---- the last block: sums of the pass's counters (a slot per thread), then the next pass ----
    if (t < kCounterSlots)
    {
        for (int c = 0; c < kNumCounters; ++c)
        {
            unsigned long long* ctr = A.counters + (size_t)t * kCounterStride + c;
            const unsigned long long v = waveReduceSum(*ctr);
            *ctr = 0ull;
            if (laneId() == 0) red[c][w] = v;
        }
    }
    if (t < 2) A.heavyN[t] = 0;
    if (t < (int)kQueueHeads) A.qHead[t * kQueueStride] = 0u;
    if (t < kLongBins) C->nLong[t] = 0u;
    __syncthreads();
    if (t != 0) return;
    __threadfence();
    uint32_t nNext, itemsNext;
    if (tiles > 1)
    {
        nNext = (uint32_t)published(A.words + tiles - 1);
        itemsNext = (uint32_t)published(A.words + (size_t)A.wordCap + tiles - 1);
        A.head->ticket = 0u;
        A.head->done = 0u;
        A.head->epoch = shEpoch + 1u;
    }
    else
    {
        nNext = itemsNext = 0u;
        for (int k = 0; k < kCompactTile / kWave; ++k)
        {
            nNext += tot[0][k];
            itemsNext += tot[1][k];
        }
    }
    if (!INIT)
    {
        unsigned long long sum[kNumCounters];
        for (int c = 0; c < kNumCounters; ++c) sum[c] = red[c][0] + red[c][1] + red[c][2] + red[c][3];
        if ((int)C->passes < A.logCap)
        {
            PassLogDev& r = A.log[C->passes];
            r.nAL = (unsigned long long)n;
            r.nItems = C->nItems;
            r.nIterating = C->nIterating;
            r.cand = sum[kCtrCand];
            r.pairs = sum[kCtrPairs];
            r.closCand = sum[kCtrClosCand];
            r.closPairs = sum[kCtrClosPairs];
            r.tBegin = C->tBegin;
            r.tKStart = C->tStart;
            r.tKEnd = C->tEnd;
            r.tEnd = clockNow();
            r.perParticle = C->perParticle;
            r.listTotal = C->listNeed;
            r.isNR = C->isNR;
            r.maxListLog2 = C->qBucket[0];
            r.heavyItems = C->qBucket[1];
            r.splitItems = C->nSplit;
        }
        C->passes += 1u;
        if (C->isNR) C->iters += 1u;
    }
    const unsigned long long iterating = __hip_atomic_load(&C->accIterating, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    C->nRem = __hip_atomic_load(&C->accRem, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    C->accIterating = 0ull;
    C->accRem = 0ull;
    C->nIterating = iterating;
    C->nAL = nNext;
    C->qBucket[0] = 0u;
    C->qBucket[1] = 0u;
    C->nSplit = 0u;
    C->nParts = 0u;
    C->itemCosts = 0ull;
    C->tStart = ~0ull;
    C->tEnd = 0ull;
    C->tBegin = clockNow();
    C->listNeed = 0ull;
    const bool nr = iterating > 0ull;
    C->isNR = nr ? 1u : 0u;
    C->perParticle = (A.sparse > 0 && (A.flat || (int)nNext <= A.tailLeaves)) ? 1u : 0u;
    C->nItems = C->perParticle ? itemsNext : nNext;
    if (nNext == 0u || (nr && (int)C->iters >= A.maxIter))
    {
        C->halt = 1u;
        C->skip = 1u;
    }
}

// ---------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------
namespace
{

struct Plan
{
    PassCtl*    ctl;
    ItemArgs    items;
    CompactArgs compact;
    char*       scan;
    uint32_t*   jc;
    uint32_t*   jo;
    int*        jList;
    unsigned long long listCap;
    unsigned long long* listCand;
    int         L;
    int         precision;
    bool        periodic;
    int         blocks;
    int         itemBlocks;
    DensArgs    da;
};

void enqueueCompact(State& s, const Plan& P, bool init)
{
    const int grid = std::max(iceil(P.L, kCompactTile), 1);
    if (init) compactKernel<true><<<grid, kCompactThreads, 0, s.stream>>>(P.compact);
    else      compactKernel<false><<<grid, kCompactThreads, 0, s.stream>>>(P.compact);
    LAUNCH_CHECK();
}

void enqueuePass(State& s, const Plan& P)
{
    hipStream_t st = s.stream;
    launchGatherListsDevice(s, P.items.leaves, P.L, P.jc, nullptr, nullptr, P.ctl);
    scanLists(P.jc, P.jo, P.L, P.scan, P.ctl, P.listCap, st, P.items.leafRem, P.items.sparse);
    launchGatherListsDevice(s, P.items.leaves, P.L, P.jc, P.jo, P.jList, P.ctl);
    if (P.listCand)
        launchListCand(P.ctl, P.L, P.items.leaves, P.jo, P.jc, P.jList, P.items.layout, P.items.state, P.listCand, st);
    itemsKernel<<<P.itemBlocks, kItemThreads, 0, st>>>(P.items);
    LAUNCH_CHECK();
    launchDensityPersistent(P.da, P.precision, P.periodic, P.blocks, st);
    enqueueCompact(s, P, false);
}

// Everything a captured launch depends on: a graph is replayed only while this is unchanged.
std::vector<unsigned long long> planKey(const State& s, const Plan& P, int K)
{
    std::vector<unsigned long long> k;
    auto add = [&](const void* p, size_t bytes) {
        const size_t n = (bytes + 7) / 8;
        const size_t at = k.size();
        k.resize(at + n, 0ull);
        std::memcpy(k.data() + at, p, bytes);
    };
    add(&P, sizeof(Plan));
    for (const DevBuf* b : {&s.layout, &s.leafNode, &s.leafSet, &s.intFirst, &s.nodeChild, &s.nodeCx, &s.nodeCy,
                            &s.nodeCz, &s.nodeSx, &s.nodeSy, &s.nodeSz, &s.hmaxLeaf, &s.hRemLeaf, &s.box, &s.h,
                            &s.ovf, &s.scanTmp, &s.nodeLeaves, &s.heavyN, &s.heavyList, &s.heavyFlag, &s.tokPool,
                            &s.tokAt, &s.slotTok, &s.slotN, &s.fullStart, &s.fullOrder})
        k.push_back((unsigned long long)(uintptr_t)b->p);
    k.push_back((unsigned long long)s.nSets);
    k.push_back((unsigned long long)s.nodeCap);
    k.push_back((unsigned long long)s.leafCap);
    for (int v : {s.slotCap, s.listSlot, s.listHeavySteps, s.listHeavyFactor, s.listExpandLeaves, s.countList ? 1 : 0})   // of the list walks
        k.push_back((unsigned long long)(long long)v);
    k.push_back((unsigned long long)K);
    return k;
}

} // namespace

struct LoopGraph
{
    hipGraph_t     graph = nullptr;
    hipGraphExec_t exec = nullptr;
    std::vector<unsigned long long> key;
    unsigned long long lastUse = 0;

    void drop()
    {
        if (exec) HIP_CHECK(hipGraphExecDestroy(exec));
        if (graph) HIP_CHECK(hipGraphDestroy(graph));
        exec = nullptr;
        graph = nullptr;
        key.clear();
    }
};

// Captured graphs by key.  A capture costs 0.7 ms, as much as several small passes, so a plan's
// launches do not depend on the tree of one step: leaf and node counts enter as capacities rounded
// up by up to an eighth (capacityOf), the counts themselves come from the control block.  The
// particle arrays alternate between two buffers from one solve to the next (the permutation gathers
// into the alternates and swaps them in), and a tree may sit near a step of its capacity: a few
// entries, least recently used replaced.
struct GraphCache
{
    static constexpr int kEntries = 8;
    LoopGraph e[kEntries];
    unsigned long long clock = 0;
    int captures = 0;

    LoopGraph* find(const std::vector<unsigned long long>& key)
    {
        for (LoopGraph& g : e)
            if (g.exec && g.key == key)
            {
                g.lastUse = ++clock;
                return &g;
            }
        return nullptr;
    }
    LoopGraph& victim()
    {
        LoopGraph* v = &e[0];
        for (LoopGraph& g : e)
        {
            if (!g.exec) return g;
            if (g.lastUse < v->lastUse) v = &g;
        }
        return *v;
    }
};

static GraphCache& graphCache()
{
    static GraphCache* g = new GraphCache();   // lives with the process, as the device state
    return *g;
}

static double wallClockHz()
{
    static double hz = 0.0;
    if (hz == 0.0)
    {
        int dev = 0, khz = 0;
        HIP_CHECK(hipGetDevice(&dev));
        HIP_CHECK(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
        hz = khz > 0 ? 1e3 * khz : 1e8;
    }
    return hz;
}

int deviceLoop(State& s, const DeviceLoopArgs& in, Timings& t)
{
    hipStream_t st = s.stream;
    const int L = s.leafCap, na = s.totalAlive;   // the leaves' capacity; their count is in the control block
    Plan P;
    std::memset(&P, 0, sizeof(P));
    P.L = L;
    P.listCand = in.listCand;
    P.precision = s.precision;
    P.periodic = in.periodic;
    const int logCap = s.maxIter + 4;
    P.ctl = s.passCtl.get<PassCtl>(1);
    // queue head: a heavy item per item at most, plus the sub-items of the split ones
    const size_t qCap = (size_t)std::max(na, s.nLeaves) + 1 + (size_t)kMaxParts;
    int* qOrder = s.qOrder.get<int>(qCap);
    uint8_t* qFlag = s.qFlag.get<uint8_t>(qCap);
    uint32_t* qSub = s.splitLen != 0 ? s.qSub.get<uint32_t>(qCap) : nullptr;
    P.items.maxParts = s.splitParts > 0 ? std::min(s.splitParts, kMaxParts) : kMaxParts;
    double* splitPart = s.splitPart.get<double>((size_t)kMaxParts * kWave * 2);
    uint32_t* splitDone = s.splitDone.get<uint32_t>((size_t)kMaxParts);
    fillU32(splitDone, 0u, (size_t)kMaxParts, st);   // every pass leaves them at 0
    P.jc = s.jCount.get<uint32_t>((size_t)L + 1);
    P.jo = s.jOffset.get<uint32_t>((size_t)L + 2);
    unsigned long long* counters = s.counters.get<unsigned long long>((size_t)kCounterSlots * kCounterStride + 64);
    // ... and these, with the lists handed over to the block walk
    fillU32(reinterpret_cast<uint32_t*>(counters), 0u, 2 * (size_t)kCounterSlots * kCounterStride, st);
    int* heavyN = s.heavyN.get<int>(4);
    fillU32(reinterpret_cast<uint32_t*>(heavyN), 0u, 2, st);
    P.scan = scanReserve(s.scanTmp, std::max(L, 1), st);
    s.ovf.get<int>(4);
    s.heavyList.get<int>((size_t)L + 1);   // the list walks take these: sized before any capture
    s.heavyFlag.get<uint8_t>((size_t)L + 1);
    s.tokPool.get<int2>((size_t)kListTokPool);
    s.tokAt.get<uint2>((size_t)L + 1);
    reserveListSlots(s);
    s.slotN.get<uint32_t>((size_t)L + 1);
    const int instance = s.precision | (in.periodic ? 2 : 0) | (in.da.cull ? 4 : 0) | in.da.tileDepth << 3;
    if (s.loopBlocksFor != instance)
    {
        s.loopBlocks = densityPersistentBlocks(in.da, s.precision, in.periodic);
        s.loopBlocksFor = instance;
    }
    P.blocks = std::max(1, s.loopBlocks * std::max(s.loopBlockScale, 1) / 4);
    P.itemBlocks = std::max(1, std::min(iceil(L, kItemThreads / kWave), 1024));   // a wavefront per leaf where leaves are few

    P.items.C = P.ctl;
    P.items.leaves = in.leaves;
    P.items.layout = s.layout.as<uint32_t>();
    P.items.state = s.active.as<uint8_t>();
    P.items.sparse = in.sparse;
    P.items.itemOff = in.itemOff;
    P.items.jCount = P.jc;
    P.items.itemPos = in.itemPos;
    P.items.itemPart = in.itemPart;
    P.items.qOrder = s.lpt ? qOrder : nullptr;
    P.items.qFlag = s.lpt ? qFlag : nullptr;
    P.items.qSub = s.lpt ? qSub : nullptr;
    P.items.splitLen = s.splitLen;
    P.items.waves = P.blocks * 4;
    P.items.mixed = s.precision == kMixed ? 1 : 0;
    P.items.leafRem = s.leafRem.get<uint32_t>((size_t)L + 1);

    P.compact.C = P.ctl;
    P.compact.leaves = in.leaves;
    P.compact.itemOff = in.itemOff;
    P.compact.leafRem = s.leafRem.as<uint32_t>();
    P.compact.layout = P.items.layout;
    P.compact.state = P.items.state;
    P.compact.h = s.h.as<double>();
    P.compact.hmaxLeaf = s.hmaxLeaf.get<double>((size_t)L + 1);
    P.compact.hRem = s.hRemLeaf.get<double>((size_t)L + 1);
    P.compact.counters = counters;
    P.compact.log = s.passLogDev.get<PassLogDev>((size_t)logCap);
    P.compact.heavyN = heavyN;
    P.compact.qHead = s.qHead.get<uint32_t>((size_t)kQueueHeads * kQueueStride);   // the first compaction clears them
    {
        const int tiles = std::max(iceil(L, kCompactTile), 1);
        const size_t had = s.compactTmp.cap;
        char* sc = s.compactTmp.get<char>(sizeof(ScanHead) + 2 * (size_t)tiles * sizeof(unsigned long long));
        if (s.compactTmp.cap != had)   // a new buffer: no ticket taken, epoch 0, words of no epoch in use
        {
            fillU32(reinterpret_cast<uint32_t*>(sc), ~0u, s.compactTmp.cap / 4, st);
            fillU32(reinterpret_cast<uint32_t*>(sc), 0u, sizeof(ScanHead) / 4, st);
        }
        P.compact.head = reinterpret_cast<ScanHead*>(sc);
        P.compact.words = reinterpret_cast<unsigned long long*>(sc + sizeof(ScanHead));
        P.compact.wordCap = tiles;
    }
    P.compact.logCap = logCap;
    P.compact.sparse = in.sparse;
    P.compact.maxIter = s.maxIter;
    P.compact.tailLeaves = s.tailLeaves;
    P.compact.flat = s.mapping == kMapFlat ? 1 : 0;

    // list capacity: what the buffer holds, at least 16 entries per leaf (or the verification
    // setting, to exercise the overflow path)
    unsigned long long cap = s.jList.cap / sizeof(int);
    cap = std::max<unsigned long long>(cap, 16ull * (unsigned long long)L + 1024ull);
    if (cap > 0xFFFFFFF0ull) cap = 0xFFFFFFF0ull;
    P.jList = s.jList.get<int>((size_t)cap);
    // the capacity the buffer really has (a grown buffer holds more than asked), so that the
    // next solve finds the same value and replays the same graph
    cap = std::min<unsigned long long>(s.jList.cap / sizeof(int), 0xFFFFFFF0ull);
    if (s.loopListCap > 0) cap = std::min<unsigned long long>(cap, (unsigned long long)s.loopListCap);
    P.listCap = cap;

    // byte copies: the graph key covers the Plan's bytes, padding included
    DensArgs da;
    std::memcpy(&da, &in.da, sizeof(da));
    // every buffer sized above is taken here, after its last resize (a pointer taken before a
    // resize would point at freed memory, or at nothing on a process's first solve)
    da.hmaxLeaf = s.hRemLeaf.as<double>();   // FLAT passes: bounds every h evaluated
    da.ctl = P.ctl;
    da.qHead = P.compact.qHead;
    da.qOrder = P.items.qOrder;
    da.qFlag = P.items.qFlag;
    da.qSub = P.items.qSub;
    da.splitPart = splitPart;
    da.splitDone = splitDone;
    da.itemPos = in.itemPos;
    da.itemPart = in.itemPart;
    da.jOffset = P.jo;
    da.jList = P.jList;
    da.counters = counters;
    da.nLeaves = da.nItems = 0;   // not read here, and not part of the plan
    std::memcpy(&P.da, &da, sizeof(da));

    PassCtl h0;
    std::memset(&h0, 0, sizeof(h0));
    h0.nAL = (uint32_t)s.nLeaves;   // every leaf; the first compaction drops those without live particles
    // the first pass's typical list: the last all-leaf lists' (a carried step's h is near the
    // converged h they were built at; the symmetric lists of the gradient sweep, a superset,
    // when no gather lists were built); none for a first solve
    h0.listMean = (unsigned long long)(s.listMeanGather > 0.0 ? s.listMeanGather : s.listMeanSym);
    HIP_CHECK(hipMemcpyAsync(P.ctl, &h0, sizeof(h0), hipMemcpyHostToDevice, st));
    enqueueCompact(s, P, true);

    const int K = std::max(1, s.graphPasses);
    GraphCache& cache = graphCache();
    LoopGraph* G = nullptr;
    auto capture = [&]() {
        if (!G) G = &cache.victim();
        G->drop();
        HIP_CHECK(hipStreamSynchronize(st));
        HIP_CHECK(hipStreamBeginCapture(st, hipStreamCaptureModeRelaxed));
        for (int k = 0; k < K; ++k) enqueuePass(s, P);
        HIP_CHECK(hipStreamEndCapture(st, &G->graph));
        HIP_CHECK(hipGraphInstantiate(&G->exec, G->graph, nullptr, nullptr, 0));
        G->key = planKey(s, P, K);
        G->lastUse = ++cache.clock;
        ++cache.captures;
    };
    if (s.useGraph)
    {
        G = cache.find(planKey(s, P, K));
        if (!G) capture();
    }

    PassCtl hc;
    int replays = 0, overflows = 0;
    // every replay without an overflow completes at least one pass, and a solve has at most
    // maxIter + 1 passes; every overflow grows the buffer past the need it reported: bound
    // both, so that a broken invariant aborts instead of spinning
    const int maxReplays = s.maxIter + 8, maxOverflows = 64;
    for (;;)
    {
        if (replays - overflows > maxReplays || overflows > maxOverflows)
        {
            std::fprintf(stderr, "FATAL: solveDensH: device-driven loop did not finish (%d replays, %d list overflows)\n",
                         replays, overflows);
            std::abort();
        }
        if (s.useGraph) HIP_CHECK(hipGraphLaunch(G->exec, st));
        else
            for (int k = 0; k < K; ++k) enqueuePass(s, P);
        ++replays;
        HIP_CHECK(hipMemcpyAsync(&hc, P.ctl, sizeof(hc), hipMemcpyDeviceToHost, st));
        HIP_CHECK(hipStreamSynchronize(st));
        if (hc.overflow)
        {
            // grow the list buffer and redo the pass that stopped (it changed nothing)
            ++overflows;
            if (hc.listNeed <= P.listCap)
            {
                std::fprintf(stderr, "FATAL: solveDensH: list overflow reported for %llu entries within capacity %llu\n",
                             hc.listNeed, P.listCap);
                std::abort();
            }
            unsigned long long want = hc.listNeed + hc.listNeed / 4 + 1024ull;
            if (hc.listNeed > 0xFFFFFFF0ull)
            {
                std::fprintf(stderr, "FATAL: neighbour-leaf lists hold %llu entries, beyond 32-bit offsets\n",
                             hc.listNeed);
                std::abort();
            }
            want = std::min<unsigned long long>(want, 0xFFFFFFF0ull);
            HIP_CHECK(hipStreamSynchronize(st));
            s.jList.reserve((size_t)want * sizeof(int));
            P.jList = s.jList.as<int>();
            P.listCap = std::min<unsigned long long>(s.jList.cap / sizeof(int), 0xFFFFFFF0ull);
            P.da.jList = P.jList;
            hc.overflow = 0u;
            hc.skip = 0u;
            hc.qBucket[0] = 0u;
            hc.itemCosts = 0ull;
            std::memset(hc.nLong, 0, sizeof(hc.nLong));
            HIP_CHECK(hipMemcpyAsync(P.ctl, &hc, sizeof(hc), hipMemcpyHostToDevice, st));
            fillU32(reinterpret_cast<uint32_t*>(heavyN), 0u, 2, st);   // the count walk runs again
            if (s.useGraph) capture();
            continue;
        }
        if (hc.halt) break;
    }

    // per-pass records -> timings, counters and the pass log
    const int nPass = std::min((int)hc.passes, logCap);
    std::vector<PassLogDev> rec((size_t)std::max(nPass, 1));
    if (nPass > 0)
        HIP_CHECK(hipMemcpyAsync(rec.data(), P.compact.log, (size_t)nPass * sizeof(PassLogDev), hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    const double hz = wallClockHz();
    for (int p = 0; p < nPass; ++p)
    {
        const PassLogDev& r = rec[p];
        const bool ran = r.tKStart != ~0ull && r.tKEnd >= r.tKStart && r.tKStart >= r.tBegin;
        const double tk = ran ? (double)(r.tKEnd - r.tKStart) / hz : 0.0;
        const double tj = ran ? (double)(r.tKStart - r.tBegin) / hz : 0.0;
        const double tc = ran ? (double)(r.tEnd - r.tKEnd) / hz : (double)(r.tEnd - r.tBegin) / hz;
        s.passLog.push_back(PassRecord{(double)r.nAL, (double)r.nItems, (double)r.nIterating, (double)r.cand,
                                       (double)r.pairs, (double)r.closCand, tk, (double)r.perParticle, tj, tc,
                                       (double)r.listTotal, (double)r.maxListLog2, (double)r.heavyItems,
                                       (double)r.splitItems});
        if (r.isNR)
        {
            t.jbuild += tj;
            t.nrkern += tk;
            t.compact += tc;
            t.iters += 1;
            t.kernLaunches += 1;
        }
        else
        {
            t.closure += tj + tk + tc;
        }
        t.pairsAccepted += (double)r.pairs;
        t.pairsCandidate += (double)r.cand;
        t.closurePairs += (double)r.closPairs;
        t.closureCand += (double)r.closCand;
        s.listTotal = (int)std::min<unsigned long long>(r.listTotal, 0x7FFFFFFFull);
    }
    t.graphReplays += replays;
    t.graphCaptures = cache.captures;
    return hc.nIterating > 0ull ? (int)std::min<unsigned long long>(hc.nIterating, 0x7FFFFFFFull) : 0;
}

} // namespace csph
