/*
 * lookback.hpp -- the pieces of single-launch scans (decoupled look-back: Merrill and Garland,
 * "Single-pass Parallel Prefix Scan with Decoupled Look-back", 2016), shared by the scan
 * (prims.hip) and the compaction of the device-driven loop (loop.hip).
 *
 * A block's tile is taken from a counter, in the order the blocks start.  It publishes its tile's
 * own sum in the tile's word and finds the sum of the tiles before it by looking back over their
 * words.  It waits only for tiles whose blocks have started, which publish before they wait
 * themselves: every wait ends.  A word is (epoch, state, value), state 1 = the tile's own sum, 2 =
 * the sum up to and with the tile.  The words need no clearing: each launch has its own epoch, and
 * the launch's last block to finish moves counter and epoch on for the next one (launches that share
 * the scratch are ordered by the stream).
 */
#pragma once

#include "common.hpp"

namespace csph
{

struct ScanHead
{
    uint32_t ticket, done, epoch, pad;
};

constexpr unsigned long long kWordSum = 1ull << 32, kWordPrefix = 2ull << 32;   // state bits; the epoch above them

__device__ inline unsigned long long wordOf(uint32_t epoch, unsigned long long state, uint32_t value)
{
    return ((unsigned long long)(epoch & 0x3FFFFFFFu) << 34) | state | value;
}

__device__ inline void publish(unsigned long long* w, unsigned long long v)
{
    __hip_atomic_store(w, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ inline unsigned long long published(const unsigned long long* w)
{
    return __hip_atomic_load(w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Called by one wavefront: publishes tile's own sum and returns the sum of the tiles before it (in
// every lane): windows of 64 words, newest first, up to the nearest one that carries a prefix.
__device__ inline uint32_t tilePrefix(unsigned long long* words, int tile, uint32_t epoch, uint32_t own)
{
    uint32_t sum = 0;
    if (tile > 0)
    {
        if (laneId() == 0) publish(words + tile, wordOf(epoch, kWordSum, own));
        const unsigned long long tag = wordOf(epoch, 0, 0) >> 34;
        for (int t = tile - 1 - laneId();; t -= kWave)
        {
            unsigned long long w = kWordPrefix;   // before the first tile: an empty prefix
            if (t >= 0)
                do w = published(words + t);
                while ((w >> 34) != tag || !(w & (kWordSum | kWordPrefix)));
            const uint64_t isPrefix = ballot64((w & kWordPrefix) != 0);
            const int stop = isPrefix ? __builtin_ctzll(isPrefix) : kWave - 1;
            sum += waveReduceSum(laneId() <= stop ? (uint32_t)w : 0u);
            if (isPrefix) break;
        }
    }
    if (laneId() == 0) publish(words + tile, wordOf(epoch, kWordPrefix, sum + own));
    return sum;
}

} // namespace csph
