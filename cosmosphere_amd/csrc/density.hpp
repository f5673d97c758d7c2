/*
 * density.hpp -- launch interface of the Newton-Raphson pass (nr.hip: density kernel,
 * closure, work items, compaction), of the gradient sweep (density.hip) and of the force
 * kernels (force.hip).
 */
#pragma once

#include "state.hpp"

namespace csph
{

// Device-resident state of the Newton-Raphson loop when its passes run without the host
// (loop.hip): every kernel of a pass reads its counts and its go/no-go from here instead of
// from its launch size.  Written by the last block to finish of the list scan and of the
// compaction, by the items kernel's counters and by the work queue's atomics.
struct PassCtl
{
    uint32_t nAL;           // active leaves: positions [0, nAL) of the leaf list
    uint32_t nItems;        // work items of the current pass
    uint32_t iters;         // NR passes completed
    uint32_t passes;        // passes completed (NR and closure-only): next log record
    uint32_t halt;          // the loop is over: no active leaf, or the NR pass cap reached
    uint32_t overflow;      // the current pass needs more list entries than the list buffer holds
    uint32_t skip;          // the current pass does nothing (halt or overflow)
    uint32_t perParticle;   // the current pass uses per-particle items for sparse leaves
    uint32_t isNR;          // the current pass holds NR evaluations (else closures only)
    uint32_t qBucket[2];    // work queue: [0] largest cost bucket, [1] entries at its head (heavy items, split)
    uint32_t nSplit;        // items split over several wavefronts this pass
    uint32_t nParts;        // sub-items of the split items (slots of the partials taken)
    uint32_t nLong[168];    // whole-leaf items with more than kSplitLen list entries, by longBin
    unsigned long long itemCosts;       // cost of all items of the pass (itemCost)
    unsigned long long nIterating;      // particles in state 1 at the start of the pass
    unsigned long long nRem;            // particles in state != 0 at the start of the pass
    unsigned long long accIterating, accRem;   // ... of the next pass, summed by the compaction's blocks
    unsigned long long listNeed;        // list entries of the current pass
    unsigned long long accList;         // ... summed by the scan's blocks (zero between scans)
    unsigned long long tBegin;          // wall clock at the start of the pass
    unsigned long long tStart, tEnd;    // density kernel span (wall clock) of the current pass
    unsigned long long listMean;        // list entries per active leaf of the last pass that built lists (0: none yet)
};

// One record per pass of a device-driven loop (u64 fields, wall-clock ticks for times).
struct PassLogDev
{
    unsigned long long nAL, nItems, nIterating, cand, pairs, closCand, closPairs;
    unsigned long long tBegin, tKStart, tKEnd, tEnd, perParticle, listTotal, isNR, maxListLog2, heavyItems, splitItems;
};

struct DensArgs
{
    const int*      leaves;     // active leaf ids (nullptr: leaf a is leaf a)
    int             nLeaves;
    const int*      itemPos;    // work item -> position in `leaves` (nullptr: item k is position k)
    const int*      itemPart;   // work item -> particle, or -1 for a whole-leaf item (nullptr: all -1)
    int             nItems;
    const uint32_t* jOffset;    // CSR of the lists, indexed by position in `leaves`
    const int*      jList;
    const uint32_t* layout;
    const int*      leafNode;
    const int*      leafSet;
    const double*   cx; const double* cy; const double* cz;
    const double*   sx; const double* sy; const double* sz;
    const double*   lbox;       // tight boxes of the leaves' particles (culling), lboxN apart
    int             lboxN;
    const double*   hmaxLeaf;
    const double*   x; const double* y; const double* z;
    double*         h;
    double*         rho;
    double*         gradh;
    uint8_t*        state;      // 1 iterating, 2 converged with closure pending, 0 done
    const DBox*     boxes;
    double          pmass, tolh, hfact;
    const double*   pmassSet;   // ensemble: particle mass of each set (nullptr: pmass)
    int             closure;    // converged particles pass through state 2
    int             cull;       // whole-leaf items: stage only list entries some particle's support reaches
    int             units;      // mixed whole-leaf items: lanes over work units where that idles fewer lanes
    int             tileDepth;  // device-driven pass: j-slots per LDS tile of whole-leaf items (64 or 128)
    unsigned long long* counters;
    PassCtl*        ctl;        // device-driven pass: persistent waves pull items from a queue
    uint32_t*       qHead;      // ... kQueueHeads counters, kQueueStride words apart, 0 at the start of a pass
    const int*      qOrder;     // ... heavy items qOrder[0, ctl->qBucket[1]) first, then every item
    const uint8_t*  qFlag;      //     not flagged heavy, in item order (nullptr: item order only)
    const uint32_t* qSub;       // ... per head entry: packSub, 0 of an item not split (nullptr: none split)
    double*         splitPart;  // split items: per sub-item (part0 on) and particle, the two partial sums
    uint32_t*       splitDone;  // ... at part0, sub-items finished (the last one resets it)
};

// Counters of the work queue (nr.hip), each in a cache line of its own.
constexpr uint32_t kQueueHeads  = 32;
constexpr uint32_t kQueueStride = 32;

// Split work items: sub-items run by different wavefronts, each summing a part of the item's pairs;
// the last to finish adds the partial sums in sub-item order and ends the particles.  A part is a
// range of the list or (mixed whole leaves, whose FP32 partials have to stay as they are) every
// n-th of the tiles staged from the whole list.  Which items are split: loop.hip; the sub-items of
// a pass always fit their slots (an item cut or not as the slots last would be cut in one run of a solve
// and not in the next, and its sums rounded otherwise).
constexpr int kSplitLen = 2048;         // mixed whole leaves: list ranges beyond this many entries ...
constexpr int kMaxSplit = 256;          // ... of at most this many items a pass
constexpr int kMaxSub   = 32;           // sub-items of an item
constexpr int kMaxParts = 32768;        // sub-items of a pass's split items

// A queue-head entry's sub-item: its number, count, kind and the item's first slot of the partials.
constexpr uint32_t kSubTiles = 1u << 12;
__device__ inline uint32_t packSub(uint32_t sub, uint32_t nSub, bool byTiles, uint32_t part0)
{
    return sub | (nSub << 6) | (byTiles ? kSubTiles : 0u) | (part0 << 16);
}
__device__ inline uint32_t subNumber(uint32_t s) { return s & 63u; }
__device__ inline uint32_t subCount(uint32_t s) { return (s >> 6) & 63u; }
__device__ inline uint32_t subPart0(uint32_t s) { return s >> 16; }

// What an item costs: its list entries, each staged (as much work as kStageCost particles' pairs
// with it) and swept for the particles evaluated.
constexpr uint32_t kStageCost = 8;
__device__ inline uint32_t itemCost(uint32_t len, uint32_t particles)
{
    return (uint32_t)min((unsigned long long)len * (kStageCost + particles), 0x7FFFFFFFull);
}

// Cost bucket of a list of len entries: floor(log2).
__device__ inline int listBucket(uint32_t len) { return 31 - __clz((int)(len | 1u)); }

// Finer ones of lists of at least kSplitLen = 2^11 entries: eight to a power of two.
constexpr int kLongBins = (32 - 11) * 8;
static_assert(kSplitLen == 1 << 11 && kLongBins == sizeof(PassCtl::nLong) / sizeof(uint32_t), "longBin");
__device__ inline int longBin(uint32_t len)
{
    const int b = listBucket(len);
    return (b - 11) * 8 + (int)((len >> (b - 3)) & 7u);
}

// Work items of an active leaf with `remaining` particles still to evaluate.
__device__ inline uint32_t itemsOf(uint32_t remaining, int sparse)
{
    return remaining == 0 ? 0u : (remaining <= (uint32_t)sparse ? remaining : 1u);
}

// Device work counters (u64, summed over the counter slots).
enum Counter
{
    kCtrPairs = 0,        // accepted pairs of NR evaluations
    kCtrCand = 1,         // candidate pairs of NR evaluations
    kCtrIterating = 2,    // particles in state 1 after the pass
    kCtrRemaining = 3,    // particles in state != 0 after the pass
    kCtrItems = 4,        // work items of the next pass
    kCtrClosPairs = 5,    // accepted pairs of closure evaluations
    kCtrClosCand = 6,     // candidate pairs of closure evaluations
    kNumCounters = 7
};

// Work items of a gradient or force sweep, one wavefront each: items [0, nHeavy) are single
// particles (heavy[k] = (leaf, particle)) of the leaves whose lists are long (flag[leaf] != 0);
// item nHeavy + l is leaf l, skipped if flagged.  A whole-leaf wavefront runs the leaf's list
// once per chunk of up to 64 particles; a long list (a leaf whose largest h reaches far, most of
// it beyond the other particles' supports) then keeps one wavefront busy long after the rest of
// the grid has drained.  Its particles spread over wavefronts finish together with the others.
struct SweepItems
{
    int            nHeavy = 0;
    const int2*    heavy = nullptr;
    const uint8_t* flag = nullptr;

    // item k -> leaf a and its particle range [p0, p1); false for a skipped item
    __device__ bool resolve(int k, int nLeaves, const uint32_t* layout, int& a, uint32_t& p0, uint32_t& p1) const
    {
        if (k < nHeavy)
        {
            const int2 it = heavy[k];
            a = it.x;
            p0 = (uint32_t)it.y;
            p1 = p0 + 1u;
            return true;
        }
        a = k - nHeavy;
        if (a >= nLeaves || (flag && flag[a])) return false;
        p0 = layout[a];
        p1 = layout[a + 1];
        return true;
    }
    int count(int nLeaves) const { return nLeaves > 0 ? nHeavy + nLeaves : 0; }
};

// The gradient and force sweeps run one wavefront per block, so that its place is free as soon as it
// ends: in blocks of four a place waits for the longest of four neighbouring items, and only 2,400
// of the chip's 4,096 wavefronts were at work in the middle of a sweep of the 1M-particle mixture.
// Blocks go to the 8 dies (each with its own L2) in turn; the numbers are dealt so that a die gets
// runs of kSweepRun neighbouring items, which share most of their j-particles.  Force pass and
// gradient sweep in blocks of four, of one, of one in runs (16 to 256: within 1%): 4M-particle
// mixture (mixed) 12.3, 10.1, 8.8 and 6.8, 5.8, 5.6 ms; 1M (FP64) 5.0, 3.95, 3.85 and 2.77, 2.37,
// 2.31 ms; periodic box of 369k (FP64) 0.62, 0.58, 0.55 and 0.54, 0.48, 0.43 ms.
constexpr int kXcds = 8, kSweepRun = 32;
__device__ inline int sweepItem(unsigned b)
{
    constexpr unsigned kTurn = kXcds * kSweepRun;
    const unsigned r = b % kTurn;
    return (int)(b - r + (r % kXcds) * kSweepRun + r / kXcds);
}
inline int sweepGrid(int items) { return iceil(items, kXcds * kSweepRun) * kXcds * kSweepRun; }

struct GradArgs
{
    int             nLeaves;
    const uint32_t* jOffset;
    const int*      jList;
    const uint32_t* layout;
    const int*      leafSet;
    const double*   x; const double* y; const double* z;
    const double*   vx; const double* vy; const double* vz;
    const double*   ax; const double* ay; const double* az;
    const double*   h;
    double*         rho; double* gradh; double* divv; double* xi; double* ddivvdt;
    const DBox*     boxes;
    double          pmass;
    const int*      leafNode;                                 // per-particle culling of list entries
    const double*   lbox;                                     // ... against the leaves' tight boxes
    int             lboxN;
    const double*   cx; const double* cy; const double* cz;
    const double*   sx; const double* sy; const double* sz;
    SweepItems      items;                                    // one wavefront per item
};

struct ForceArgs
{
    int             nLeaves;
    const uint32_t* jOffset;
    const int*      jList;
    const uint32_t* layout;
    const int*      leafSet;
    const double*   x; const double* y; const double* z;
    const double*   vx; const double* vy; const double* vz;
    const double*   h;
    const double*   pro2; const double* cs; const double* alpha; const double* u;
    const double*   hsqinv; const double* hinv; const double* rhoh; const double* rho1;
    const double*   grkfac; const double* pres; const double* auterm; const double* divfac;
    double*         fx; double* fy; double* fz; double* f4; double* vsig; double* divv;
    const DBox*     boxes;
    double          pmass, beta, alphau;
    int             pdv, shock;
    unsigned long long* counters;
    const int*      leafNode;                                 // per-particle culling of list entries
    const double*   lbox;                                     // ... against the leaves' tight boxes
    int             lboxN;
    const double*   cx; const double* cy; const double* cz;
    const double*   sx; const double* sy; const double* sz;
    const double*   hmaxLeaf;                                 // reach of a j-leaf's own supports
    const float*    f32;      // mixed form: FP32 copies of hsqinv, hinv, grkfac, rhoh, rho1, pro2, cs,
    size_t          f32Stride; // alpha, pres, auterm (array k at f32 + k f32Stride)
    SweepItems      items;    // one wavefront per item
};

// mode 0: NR on the particles in state != 0 (FLAT_PARTICLE; state 2 = closure only);
// 1: NR on every particle of an active leaf (WARP_PER_LEAF); 2: closure of every particle,
// rho and d(rho)/d(h) at the current h, no update.  a.nItems work items.
void launchDensity(const DensArgs& a, int precision, int mode, bool periodic, hipStream_t st);
// Device-driven pass: both item forms are launched as persistent grids of `blocks` blocks; the
// one ctl->perParticle does not select exits at once.
void launchDensityPersistent(const DensArgs& a, int precision, bool periodic, int blocks, hipStream_t st);
int  densityPersistentBlocks(const DensArgs& a, int precision, bool periodic);
void launchGradients(const GradArgs& a, bool periodic, bool mixed, hipStream_t st);
// Per-particle items of the leaves with more than `entries` list entries (0: none); reads the
// item count back (host-synchronising).
SweepItems buildSweepItems(State& s, int nLeaves, int entries, hipStream_t st);
void launchDeadGradients(int first, int n, double* divv, double* xi, double* ddivvdt, hipStream_t st);
// Per active leaf: flag (has a particle in state != 0) and its work-item count (1 whole-leaf
// item, or one item per remaining particle when at most `sparse` remain); counters 2-4.
// List candidates of a pass: for each active leaf position a (n of them, or ctl->nAL), the
// particle counts of its list's leaves summed (entries [jOffset[a], jOffset[a] + jCount[a]), or
// to jOffset[a + 1] without jCount), times the leaf's particles in state 1 into out[0] and in
// state 2 into out[1]; without state, times all its particles into out[0].
void launchListCand(const PassCtl* ctl, int n, const int* leaves, const uint32_t* jOffset, const uint32_t* jCount,
                    const int* jList, const uint32_t* layout, const uint8_t* state, unsigned long long* out,
                    hipStream_t st);
void launchLeafFlags(const int* leaves, int nLeaves, const uint32_t* layout, const uint8_t* state, int sparse,
                     uint32_t* flag, uint32_t* itemCount, unsigned long long* counters, hipStream_t st);
// Compaction: out[pos[a]] = leaves[a], outCount[pos[a]] = count[a] for flagged a.
void launchLeafScatter(const int* leaves, const uint32_t* count, int nLeaves, const uint32_t* flag,
                       const uint32_t* pos, int* out, uint32_t* outCount, hipStream_t st);
// Work items of the active leaves from their counts' exclusive scan `off`.
void launchItemFill(const int* leaves, int nLeaves, const uint32_t* layout, const uint8_t* state, int sparse,
                    const uint32_t* off, int* itemPos, int* itemPart, hipStream_t st);
void launchInitActive(uint8_t* active, int nAlive, int n, double* rho, double* gradh, hipStream_t st);
void launchIota(int* v, int n, hipStream_t st);
void launchMaxH(const double* h, int n, unsigned long long* out, hipStream_t st);
int  counterSlots();
int  counterStride();

void launchForcePrep(const double* h, const double* gradh, const double* pro2, double* hsqinv, double* hinv,
                     double* rhoh, double* rho1, double* grkfac, double* pres, double* auterm, double* divfac, int n,
                     double pmass, double alphau, double hfact, hipStream_t st);
// rounds: the mixed form with each tile's accepted pairs shared evenly over the lanes
// (forceKernelMixedRounds, the default), else lanes that keep their own slots (forceKernelMixed)
void launchForce(const ForceArgs& a, bool periodic, bool disc, bool full, bool mixed, bool rounds, hipStream_t st);
// FP32 copies of the force factors for the mixed form (ForceArgs::f32 layout), n particles.
void launchForceF32(const ForceArgs& a, int n, float* dst, hipStream_t st);
void launchDeadForce(int first, int n, double* fx, double* fy, double* fz, double* f4, double* vsig, double* divv,
                     hipStream_t st);

} // namespace csph
