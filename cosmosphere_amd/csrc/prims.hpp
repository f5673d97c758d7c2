/*
 * prims.hpp -- device-wide scan and radix sort (prims.hip).
 */
#pragma once

#include "state.hpp"

namespace csph
{

struct PassCtl;

struct SortScratch
{
    DevBuf words;           // digit counts, tile counters and look-back words of the running sort
    int*   err = nullptr;   // device counter of out-of-range scatters (must stay 0)
};


// The scratch of scans of up to n entries, sized and (when it had to grow) set up.  It carries state
// from one scan to the next: scans that share it run on one stream.
char* scanReserve(DevBuf& scratch, int n, hipStream_t st);

// out[0..n] = exclusive prefix sums of in[0..n), out[n] = total.  If total64 is given,
// the total is also added to it as a 64-bit sum (overflow check).
void scanExclusive(const uint32_t* in, uint32_t* out, int n, DevBuf& scratch, unsigned long long* total64,
                   hipStream_t st);

// Device-driven pass: the offsets of the ctl->nAL lists from their counts (n: their capacity),
// the longest list's cost bucket, and the check of the total against cap entries (prims.hip); with
// the lists' particles still to evaluate in leafRem also the cost of the pass's items and its long lists.
// Nothing when ctl->skip.  scratch: scanReserve'd for n before the capture.
void scanLists(const uint32_t* counts, uint32_t* offsets, int n, char* scratch, PassCtl* ctl, unsigned long long cap,
               hipStream_t st, const uint32_t* leafRem = nullptr, int sparse = 0);

// Stable ascending sort of (keys, vals) by the 8-bit digits that hold a bit of `varying`; the
// other digits must be shared by all keys, or in order already among keys that the sorted digits
// leave equal.  Returns true when the sorted result sits in keysAlt / valsAlt rather than keys /
// vals.
bool radixSortPairs(uint64_t* keys, uint64_t* keysAlt, uint32_t* vals, uint32_t* valsAlt, int n, uint64_t varying,
                    SortScratch& sc, hipStream_t st);

// The bits in which the integers 0 .. n - 1 can differ.
inline uint64_t bitsBelow(uint64_t n) { return n <= 1 ? 0 : ~uint64_t(0) >> __builtin_clzll(n - 1); }

// Fill with a kernel rather than hipMemsetAsync, so the call is safe inside graph capture.
void fillU32(uint32_t* p, uint32_t v, size_t n, hipStream_t st);

} // namespace csph
