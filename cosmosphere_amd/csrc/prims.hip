/*
 * prims.hip -- device-wide primitives written for gfx950: exclusive scan, a stable LSD
 * radix sort of (u64 key, u32 value) pairs that skips the digits the caller knows to be
 * shared by all keys.  These replace the Thrust calls of the reference
 * (sequence + sort_by_key, src/tree.cu:90-91; the inclusive scans of tree.cu:151 and
 * tree.cuh:385).
 *
 * Sort: 8-bit digits, one launch per digit after one that counts every digit.  Each 256-thread
 * block owns a tile of 4096 keys; each wavefront a contiguous 1024 of them, visited in 16 rounds of
 * 64 coalesced loads.  Wave-level multisplit: 8 ballots give each lane the mask of lanes with
 * its digit, the rank is the popcount below it, and a per-wave LDS counter carries ranks across
 * rounds -- so the order within a digit is the input order, which is what makes the sort stable.
 * The base of (digit, tile) comes from looking back over the earlier tiles' published counts
 * (the scheme of Adinets and Merrill, "Onesweep: A Faster Least Significant Digit Radix Sort for
 * GPUs", 2022).
 */
#include "density.hpp"
#include "lookback.hpp"
#include "prims.hpp"

#include <algorithm>

namespace csph
{

// ---------------------------------------------------------------------------------------
// Exclusive scan
// ---------------------------------------------------------------------------------------
// One launch by look-back (lookback.hpp) over tiles of 2048.  The tile / top / add / total launches
// this replaces took 13-20 us per scan where the data take 1-2.
constexpr int kScanThreads = 256;
constexpr int kScanItems   = 8;
constexpr int kScanTile    = kScanThreads * kScanItems;

// Count of a device-driven scan: entries from nEff on read as zero.
__device__ inline int scanCount(const PassCtl* ctl, int n) { return ctl ? min(n, (int)ctl->nAL) : n; }

// LISTS: the offsets of a device-driven pass's lists.  The largest list's cost bucket goes to
// ctl->qBucket[0], and the last block to finish checks the total against the list buffer's
// capacity: a pass that does not fit stops here with nothing changed.  Totals are summed in 64 bits:
// the offsets of lists of more than 2^32 entries wrap, and must not look as if they fitted.
template<bool LISTS>
__global__ __launch_bounds__(kScanThreads) void scanKernel(const uint32_t* __restrict__ in, uint32_t* __restrict__ out,
                                                           int n, ScanHead* __restrict__ head,
                                                           unsigned long long* __restrict__ words,
                                                           unsigned long long* __restrict__ total64,
                                                           PassCtl* __restrict__ ctl, unsigned long long cap,
                                                           const uint32_t* __restrict__ leafRem, int sparse)
{
    __shared__ uint32_t longLists[LISTS ? kLongBins : 1];
    __shared__ unsigned long long waveCost[LISTS ? kScanThreads / kWave : 1];
    __shared__ uint32_t waveTot[kScanThreads / kWave];
    __shared__ unsigned long long waveTot64[kScanThreads / kWave];
    __shared__ uint32_t waveMax[kScanThreads / kWave];
    __shared__ uint32_t shTile, shEpoch, shBefore;
    if (ctl && ctl->skip) return;
    const int nEff = scanCount(ctl, n);
    const int tiles = nEff / kScanTile + 1;   // entries 0 .. nEff
    if ((int)blockIdx.x >= tiles) return;     // the rest of a capacity's grid
    if (threadIdx.x == 0)
    {
        shTile = tiles > 1 ? atomicAdd(&head->ticket, 1u) : 0u;
        shEpoch = head->epoch;
    }
    if constexpr (LISTS)
        if (threadIdx.x < kLongBins) longLists[threadIdx.x] = 0u;
    __syncthreads();
    const int tile = (int)shTile;
    const int base = tile * kScanTile + threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t sum = 0, most = 0;
    unsigned long long sum64 = 0, cost = 0;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
    {
        const int i = base + k;
        v[k] = (i < nEff) ? in[i] : 0u;
        sum += v[k];
        sum64 += v[k];
        if constexpr (LISTS)
        {
            most = max(most, v[k]);
            if (leafRem && i < nEff)
            {
                const uint32_t rem = leafRem[i];
                const bool parts = ctl->perParticle && rem <= (uint32_t)sparse;   // an item for each particle
                cost += parts ? (unsigned long long)rem * itemCost(v[k], 1u) : (unsigned long long)itemCost(v[k], rem);
                if (!parts && v[k] > (uint32_t)kSplitLen) atomicAdd(&longLists[longBin(v[k])], 1u);
            }
        }
    }
    // block-wide exclusive scan of the per-thread sums
    const uint32_t incl = waveInclusiveScan(sum);
    const int w = threadIdx.x / kWave;
    if (laneId() == kWave - 1) waveTot[w] = incl;
    if (LISTS || total64)
    {
        sum64 = waveReduceSum(sum64);
        if (laneId() == 0) waveTot64[w] = sum64;
    }
    if constexpr (LISTS)
    {
        most = waveReduceMax(most);
        cost = waveReduceSum(cost);
        if (laneId() == 0)
        {
            waveMax[w] = most;
            waveCost[w] = cost;
        }
    }
    __syncthreads();
    uint32_t waveOff = 0, blockTot = 0;
#pragma unroll
    for (int j = 0; j < kScanThreads / kWave; ++j)
    {
        if (j < w) waveOff += waveTot[j];
        blockTot += waveTot[j];
    }
    if (w == 0)
    {
        const uint32_t before = tiles > 1 ? tilePrefix(words, tile, shEpoch, blockTot) : 0u;
        if (laneId() == 0) shBefore = before;
    }
    __syncthreads();
    uint32_t run = shBefore + waveOff + incl - sum;
#pragma unroll
    for (int k = 0; k < kScanItems; ++k)
    {
        const int i = base + k;
        if (i <= nEff) out[i] = run;   // out[nEff]: the total
        run += v[k];
    }
    if constexpr (LISTS)
        if (threadIdx.x < kLongBins && longLists[threadIdx.x]) atomicAdd(&ctl->nLong[threadIdx.x], longLists[threadIdx.x]);
    if (threadIdx.x != 0) return;
    unsigned long long blockTot64 = 0;
    if (LISTS || total64)
        for (int j = 0; j < kScanThreads / kWave; ++j) blockTot64 += waveTot64[j];
    if (total64 && blockTot64) atomicAdd(total64, blockTot64);
    if constexpr (LISTS)
    {
        const unsigned long long c = waveCost[0] + waveCost[1] + waveCost[2] + waveCost[3];
        if (c) atomicAdd(&ctl->itemCosts, c);
        if (tiles > 1 && blockTot64) atomicAdd(&ctl->accList, blockTot64);
        const uint32_t m = max(max(waveMax[0], waveMax[1]), max(waveMax[2], waveMax[3]));
        if (m > 1u) atomicMax(&ctl->qBucket[0], (uint32_t)listBucket(m));
        __threadfence();
    }
    if (tiles > 1 && atomicAdd(&head->done, 1u) != (uint32_t)tiles - 1u) return;
    if (tiles > 1)
    {
        head->ticket = 0u;
        head->done = 0u;
        head->epoch = shEpoch + 1u;
    }
    if constexpr (LISTS)
    {
        const unsigned long long tot = tiles > 1 ? published(&ctl->accList) : blockTot64;
        ctl->accList = 0ull;
        ctl->listNeed = tot;
        if (nEff > 0) ctl->listMean = tot / (unsigned long long)nEff;
        if (tot > cap)
        {
            ctl->overflow = 1u;
            ctl->skip = 1u;
        }
    }
}

static size_t scanTiles(int n) { return (size_t)iceil((long long)n + 1, kScanTile); }   // out[n] is written too

char* scanReserve(DevBuf& scratch, int n, hipStream_t st)
{
    const size_t had = scratch.cap;
    char* sc = scratch.get<char>(sizeof(ScanHead) + scanTiles(n) * sizeof(unsigned long long));
    if (scratch.cap != had)   // a new buffer: no ticket taken, epoch 0, words of no epoch in use
    {
        fillU32(reinterpret_cast<uint32_t*>(sc), ~0u, scratch.cap / 4, st);
        fillU32(reinterpret_cast<uint32_t*>(sc), 0u, sizeof(ScanHead) / 4, st);
    }
    return sc;
}

void scanExclusive(const uint32_t* in, uint32_t* out, int n, DevBuf& scratch, unsigned long long* total64,
                   hipStream_t st)
{
    char* sc = scanReserve(scratch, n, st);
    scanKernel<false><<<(int)scanTiles(n), kScanThreads, 0, st>>>(
        in, out, n, reinterpret_cast<ScanHead*>(sc), reinterpret_cast<unsigned long long*>(sc + sizeof(ScanHead)), total64,
        nullptr, 0ull, nullptr, 0);
    LAUNCH_CHECK();
}

void scanLists(const uint32_t* counts, uint32_t* offsets, int n, char* scratch, PassCtl* ctl, unsigned long long cap,
               hipStream_t st, const uint32_t* leafRem, int sparse)
{
    scanKernel<true><<<(int)scanTiles(n), kScanThreads, 0, st>>>(
        counts, offsets, n, reinterpret_cast<ScanHead*>(scratch),
        reinterpret_cast<unsigned long long*>(scratch + sizeof(ScanHead)), nullptr, ctl, cap, leafRem, sparse);
    LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------------------
// Radix sort
// ---------------------------------------------------------------------------------------
constexpr int kSortThreads = 256;
constexpr int kSortWaves   = kSortThreads / kWave;
constexpr int kSortRounds  = 16;
constexpr int kSortTile    = kSortThreads * kSortRounds;   // 4096
constexpr int kSortPasses  = 8;
constexpr int kSortLook    = 16;   // earlier tiles read per round trip of the look-back (4: 0.21 ms a pass
                                   // over 8M keys, the first tiles' look-backs one chain)

// Scratch of one sort, cleared before it: the digit counts of every pass, a tile counter per pass,
// then a word per pass, tile and digit: 2 state bits (1 = the tile's count, 2 = the count up to
// and with the tile) above 30 bits of count (2^30 particles are beyond the card's memory).
constexpr uint32_t kDigitSum = 1u << 30, kDigitPrefix = 2u << 30, kDigitValue = kDigitSum - 1u;

// Digit counts of the passes in `mask` (bit p: digit p), all of them in one read of the keys.
__global__ __launch_bounds__(kSortThreads) void radixCountKernel(const uint64_t* __restrict__ keys, int n,
                                                                 uint32_t mask, uint32_t* __restrict__ counts)
{
    __shared__ uint32_t h[kSortPasses][256];
    for (int p = 0; p < kSortPasses; ++p) h[p][threadIdx.x] = 0;
    __syncthreads();
    for (int i = blockIdx.x * kSortThreads + threadIdx.x; i < n; i += gridDim.x * kSortThreads)
    {
        const uint64_t k = keys[i];
#pragma unroll
        for (int p = 0; p < kSortPasses; ++p)
            if ((mask >> p) & 1u) atomicAdd(&h[p][(k >> (8 * p)) & 0xFF], 1u);
    }
    __syncthreads();
    for (int p = 0; p < kSortPasses; ++p)
    {
        const uint32_t c = h[p][threadIdx.x];
        if (c) atomicAdd(&counts[p * 256 + threadIdx.x], c);
    }
}

// One digit pass in one launch.  A block takes the next tile of 4096 keys (so that the tiles before
// it belong to blocks that have started), ranks them by wave-level multisplit, publishes its digit
// counts, and thread d looks back over the earlier tiles' words of digit d for the tile's base,
// kSortLook tiles a round trip.  Nobody waits before publishing, so every wait ends.  Keys and
// values leave through LDS in digit order (written straight from the ranks, a wavefront's stores
// hit up to 64 lines).  8M pairs: 93 us a pass, 2.1 TB/s of its 24 bytes a pair (count, scan and
// scatter launches before: 200 us); 180k pairs: 5 us (45 us in 5 launches).
__global__ __launch_bounds__(kSortThreads) void radixPassKernel(const uint64_t* __restrict__ keysIn,
                                                                const uint32_t* __restrict__ valsIn,
                                                                uint64_t* __restrict__ keysOut,
                                                                uint32_t* __restrict__ valsOut, int n, int shift,
                                                                const uint32_t* __restrict__ counts,
                                                                uint32_t* __restrict__ ticket,
                                                                uint32_t* __restrict__ words, int* __restrict__ err)
{
    __shared__ uint32_t cnt[kSortWaves][256];
    __shared__ uint32_t toOut[256];
    __shared__ uint32_t waveTot[2][kSortWaves];
    __shared__ uint32_t shTile;
    __shared__ uint64_t sKey[kSortTile];
    uint32_t* const sVal = reinterpret_cast<uint32_t*>(sKey);
    for (int d = threadIdx.x; d < kSortWaves * 256; d += kSortThreads) (&cnt[0][0])[d] = 0;
    if (threadIdx.x == 0) shTile = gridDim.x > 1 ? atomicAdd(ticket, 1u) : 0u;
    __syncthreads();

    const int tile = (int)shTile;
    const int w = threadIdx.x / kWave, lane = laneId();
    const int base = tile * kSortTile + w * (kSortRounds * kWave);
    uint64_t k[kSortRounds];
    uint32_t v[kSortRounds];
    uint32_t rank[kSortRounds];

#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
    {
        const int  i     = base + r * kWave + lane;
        const bool valid = i < n;
        k[r] = valid ? keysIn[i] : 0;
        v[r] = valid ? valsIn[i] : 0;
    }
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
    {
        const bool valid = base + r * kWave + lane < n;
        const uint32_t d = (uint32_t)(k[r] >> shift) & 0xFF;
        uint64_t peers = ballot64(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b)
        {
            const bool     bit = (d >> b) & 1u;
            const uint64_t m   = ballot64(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t below = (uint32_t)__popcll(peers & lanemaskLt());
        uint32_t pre = 0;
        if (valid) pre = cnt[w][d];
        waveLdsSync();
        if (valid && below == 0) cnt[w][d] = pre + (uint32_t)__popcll(peers);
        waveLdsSync();
        rank[r] = pre + below;
    }
    __syncthreads();
    {
        const int d = threadIdx.x;   // 256 threads, one digit each
        uint32_t mine = 0;
#pragma unroll
        for (int ww = 0; ww < kSortWaves; ++ww) mine += cnt[ww][d];
        uint32_t before = 0;   // keys of digit d in the earlier tiles
        if (gridDim.x > 1)
        {
            uint32_t* word = words + (size_t)tile * 256 + d;
            if (tile > 0)
            {
                __hip_atomic_store(word, kDigitSum | mine, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                for (int t = tile - 1; t >= 0;)
                {
                    uint32_t q[kSortLook];
#pragma unroll
                    for (int u = 0; u < kSortLook; ++u)
                        q[u] = __hip_atomic_load(word - (size_t)(tile - max(t - u, 0)) * 256, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int u = 0; u < kSortLook; ++u)
                    {
                        if (t < 0 || q[u] == 0u) break;   // not published yet: read again from there
                        before += q[u] & kDigitValue;
                        t = (q[u] & kDigitPrefix) ? -1 : t - 1;
                    }
                }
            }
            __hip_atomic_store(word, kDigitPrefix | (before + mine), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // exclusive scans over the digits: of the pass's counts (where the digit starts in the output)
        // and of the tile's (where it starts in the tile); then each wave's first place of the digit
        const uint32_t c = counts[d];
        const uint32_t inclAll = waveInclusiveScan(c), inclMine = waveInclusiveScan(mine);
        if (lane == kWave - 1)
        {
            waveTot[0][w] = inclAll;
            waveTot[1][w] = inclMine;
        }
        __syncthreads();
        uint32_t out = inclAll - c + before, run = inclMine - mine;
        for (int ww = 0; ww < w; ++ww)
        {
            out += waveTot[0][ww];
            run += waveTot[1][ww];
        }
        toOut[d] = out - run;
#pragma unroll
        for (int ww = 0; ww < kSortWaves; ++ww)
        {
            const uint32_t x = cnt[ww][d];
            cnt[ww][d] = run;
            run += x;
        }
    }
    __syncthreads();
    // through LDS in the tile's digit order, so that neighbouring lanes write neighbouring places
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
        if (base + r * kWave + lane < n)
        {
            rank[r] += cnt[w][(uint32_t)(k[r] >> shift) & 0xFF];
            sKey[rank[r]] = k[r];
        }
    __syncthreads();
    const int held = min(kSortTile, n - tile * kSortTile);
    uint32_t dst[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
    {
        const int i = r * kSortThreads + threadIdx.x;
        dst[r] = 0xFFFFFFFFu;
        if (i < held)
        {
            const uint64_t key = sKey[i];
            dst[r] = toOut[(uint32_t)(key >> shift) & 0xFF] + (uint32_t)i;
            if (dst[r] < (uint32_t)n) keysOut[dst[r]] = key;
            else                      atomicAdd(err, 1);
        }
    }
    __syncthreads();   // sKey becomes sVal
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
        if (base + r * kWave + lane < n) sVal[rank[r]] = v[r];
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r)
        if (dst[r] < (uint32_t)n) valsOut[dst[r]] = sVal[r * kSortThreads + threadIdx.x];
}

__global__ void fillU32Kernel(uint32_t* __restrict__ p, uint32_t v, size_t n)
{
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

void fillU32(uint32_t* p, uint32_t v, size_t n, hipStream_t st)
{
    if (n == 0) return;
    fillU32Kernel<<<(int)std::min<size_t>((n + 255) / 256, 4096), 256, 0, st>>>(p, v, n);
    LAUNCH_CHECK();
}

bool radixSortPairs(uint64_t* keys, uint64_t* keysAlt, uint32_t* vals, uint32_t* valsAlt, int n, uint64_t varying,
                    SortScratch& sc, hipStream_t st)
{
    if (n <= 1) return false;
    uint32_t mask = 0;
    int passes = 0;
    for (int p = 0; p < kSortPasses; ++p)
        if ((varying >> (8 * p)) & 0xFF)
        {
            mask |= 1u << p;
            ++passes;
        }
    const int nb = iceil(n, kSortTile);
    const size_t head = (size_t)kSortPasses * 256 + kSortPasses;
    const size_t perPass = nb > 1 ? (size_t)nb * 256 : 0;
    uint32_t* counts = sc.words.get<uint32_t>(head + perPass * passes);
    uint32_t* tickets = counts + (size_t)kSortPasses * 256;
    uint32_t* words = counts + head;
    fillU32(counts, 0u, head + perPass * passes, st);
    radixCountKernel<<<std::min(iceil(n, 4 * kSortThreads), 1024), kSortThreads, 0, st>>>(keys, n, mask, counts);
    LAUNCH_CHECK();
    bool flipped = false;
    uint64_t* kin = keys;  uint64_t* kout = keysAlt;
    uint32_t* vin = vals;  uint32_t* vout = valsAlt;
    for (int p = 0; p < kSortPasses; ++p)
    {
        if (!((mask >> p) & 1u)) continue;
        radixPassKernel<<<nb, kSortThreads, 0, st>>>(kin, vin, kout, vout, n, 8 * p, counts + p * 256, tickets + p, words,
                                                     sc.err);
        LAUNCH_CHECK();
        words += perPass;
        std::swap(kin, kout);
        std::swap(vin, vout);
        flipped = !flipped;
    }
    return flipped;   // true: the result is in keysAlt / valsAlt
}

} // namespace csph
