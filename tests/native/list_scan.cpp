// The scan of the device-driven pass's list counts (scanLists) and the host-driven one's
// (scanExclusive), on their own: totals around 2^32 entries, where the 32-bit offsets wrap.  Nothing but the
// offsets is written.  Prints a line per case; exit code 1 where a total or an overflow flag is wrong.
#include "../../cosmosphere_amd/csrc/density.hpp"
#include "../../cosmosphere_amd/csrc/prims.hpp"

#include <cstdio>
#include <cstring>
#include <vector>

using namespace csph;

int main()
{
    hipStream_t st;
    HIP_CHECK(hipStreamCreate(&st));
    const unsigned long long cap = 0xFFFFFFF0ull;
    struct Case { int n; uint32_t each; uint32_t last; };
    const Case cases[] = {
        {1000, 7u, 3u},                              // one tile, fits
        {100000, 40000u, 5u},                        // 4.0e9, fits
        {5000, 1u << 20, 1u},                        // 5.2e9 over several tiles: wraps to 9.5e8
        {1000, 5000000u, 1u},                        // 5.0e9 in one tile
        {4097, 1u << 20, 0u},                        // 4096 * 2^20 = 2^32 exactly: wraps to 0
        {300000, 14317u, 0u},                        // just above the capacity
        {300000, 14316u, 4294967280u - 299999u * 14316u},   // the capacity exactly
        {2048, 2097152u, 4294967295u},
    };
    DevBuf scratch, counts, offsets, ctlBuf, total;
    int bad = 0;
    for (int round = 0; round < 2; ++round)          // the second on used scratch
        for (const Case& c : cases)
        {
            std::vector<uint32_t> h((size_t)c.n, c.each);
            h.back() = c.last ? c.last : c.each;
            if (c.n == 4097) h.back() = 0u;
            unsigned long long want = 0;
            for (uint32_t v : h) want += v;
            uint32_t* d = counts.get<uint32_t>((size_t)c.n);
            uint32_t* o = offsets.get<uint32_t>((size_t)c.n + 1);
            char* sc = scanReserve(scratch, c.n, st);
            PassCtl ctl;
            std::memset(&ctl, 0, sizeof(ctl));
            ctl.nAL = (uint32_t)c.n;
            PassCtl* dc = ctlBuf.get<PassCtl>(1);
            unsigned long long* t64 = total.get<unsigned long long>(1);
            HIP_CHECK(hipMemcpyAsync(d, h.data(), h.size() * 4, hipMemcpyHostToDevice, st));
            HIP_CHECK(hipMemcpyAsync(dc, &ctl, sizeof(ctl), hipMemcpyHostToDevice, st));
            fillU32(reinterpret_cast<uint32_t*>(t64), 0u, 2, st);
            scanLists(d, o, c.n, sc, dc, cap, st);
            scanExclusive(d, o, c.n, scratch, t64, st);
            unsigned long long got = 0;
            HIP_CHECK(hipMemcpyAsync(&ctl, dc, sizeof(ctl), hipMemcpyDeviceToHost, st));
            HIP_CHECK(hipMemcpyAsync(&got, t64, sizeof(got), hipMemcpyDeviceToHost, st));
            HIP_CHECK(hipStreamSynchronize(st));
            const bool over = want > cap;
            const bool ok = ctl.listNeed == want && (ctl.overflow != 0u) == over && (ctl.skip != 0u) == over &&
                            ctl.listMean == want / (unsigned long long)c.n && ctl.accList == 0ull && got == want;
            std::printf("%d lists, %llu entries: %llu, overflow %u, total %llu%s\n", c.n, want, ctl.listNeed, ctl.overflow,
                        got, ok ? "" : "  WRONG");
            std::fflush(stdout);
            bad += ok ? 0 : 1;
        }
    return bad ? 1 : 0;
}
