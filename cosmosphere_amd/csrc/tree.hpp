/*
 * tree.hpp -- tree build, neighbour-leaf lists and the physics passes (host entry points
 * into the kernels of tree.hip, jlist.hip, density.hip and force.hip).
 */
#pragma once

#include "prims.hpp"

namespace csph
{

struct PassCtl;

// Block walks of long lists: tokens the count pass keeps for the fill pass (16M, 128 MiB).
constexpr int kListTokPool = 1 << 24;
constexpr int kListSlotTok = 256;  // light lists: tokens the count walk keeps per list for the fill, at least
constexpr int kListSlotMax = 2048; // ... at most
constexpr size_t kListSlotWords = size_t(1) << 30;   // ... of all lists together, beyond the least (4 GiB)

// Tokens kept per list: a list with more is walked twice, which takes several times as long as
// copying its tokens, so a slot is as long as the leaves' number allows (the first passes of a solve
// have the longest lists: 1,900 entries on the 8M-particle mixture).  Lists of a solve with slots of
// 256, 512, 1024, 2048 tokens: 250k-particle disc 5.2, 4.1, 3.7, 3.7 ms; 2M-particle mixture 19.1,
// 18.4, 15.9, 14.5; 8M 75, 75, 73, 45; 12 sets of 10k-53k 2.7, 2.3, 2.3, 2.3.
inline int listSlotTokens(int leafCap)
{
    int n = kListSlotMax;
    while (n > kListSlotTok && (size_t)n * ((size_t)leafCap + 1) > kListSlotWords) n /= 2;
    return n;
}

// The slots of the present leafCap: s.slotTok, and their length in s.slotCap.  More than the least length
// is taken only out of a sixteenth of the card's free memory, and where the allocation succeeds: it
// saves time, and must not fail a solve, or a later allocation, that fits without it.  Called before
// any capture.
void reserveListSlots(State& s);

// Box, keys, sort, permutation (x, y, z, h and, if withVelAcc, v and a), leaf tree, node
// geometry, layout and particle -> leaf map for the sets described in s.
// periodicBox: nullptr (open, fitted boxes) or 6 doubles per set.
// incremental: the inputs are in the previous solve's order (x, y, z, h and, with withVelAcc,
// v and a), and the previous tree is still in s; the keys are then re-sorted incrementally
// (resort.hip) with the same result as the full sort.
void buildTree(State& s, bool withVelAcc, const double* periodicBox, SortScratch& sc, bool incremental = false);

// Incremental re-sort of keys given in the previous solve's order (s.order, the previous
// tree's leaves and particle -> leaf map): sorted keys, the input position of each sorted
// entry and its caller index (the new order).  Returns the number of particles that left
// their previous leaf's key range (sorted from scratch).
int resortIncremental(State& s, const uint64_t* keys, uint64_t* keysOut, uint32_t* idxOut, int* orderOut,
                      SortScratch& sc);

// hmax of the given leaves (leaves == nullptr: all of them); with `state`, also the max h of
// their particles in state != 0 into s.hRemLeaf (the reach of tight lists).
void hmaxLeaves(State& s, const int* leaves, int nLeaves, const uint8_t* state = nullptr);

// hmax per node, leaves first then internal levels deepest first (force upsweep).
void hmaxUpsweep(State& s);

// CSR neighbour-leaf lists of the given leaves (leaves == nullptr: all leaves) into
// s.jCount / s.jOffset / s.jList, indexed by position in the leaf list.  Returns the
// total number of entries.  tight: gather lists trimmed to s.hRemLeaf (same order, same
// accepted pairs for the particles in state != 0).
long long buildLists(State& s, const int* leaves, int nLeaves, bool symmetric, bool tight = false);

// Device-driven pass: the count walk (jList == nullptr: counts into jCount) or the fill walk
// (into jList at jOffset) of the tight gather lists of ctl->nAL leaves; nothing when
// ctl->skip.  nCap bounds ctl->nAL.
void launchGatherListsDevice(State& s, const int* leaves, int nCap, uint32_t* jCount, const uint32_t* jOffset,
                             int* jList, PassCtl* ctl);

} // namespace csph
