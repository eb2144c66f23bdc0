// host_pages.h -- presence of a result buffer's pages before the device copies
// into it.  Plain C++: the CPU tests compile it on its own.
#pragma once

#include <sys/mman.h>

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <initializer_list>
#include <thread>
#include <utility>
#include <vector>

namespace cupf {

constexpr size_t kHostPage = 4096;

// Whether the first, the middle or the last page of [lo, hi) (whole pages) is
// not present.  A fresh mapping has none, a reused block of a heap may lack its
// end.  Where the kernel does not say, the copy faults what it has to.
inline bool pages_absent(uintptr_t lo, uintptr_t hi)
{
    const uintptr_t looks[] = {lo, lo + (hi - lo) / 2 / kHostPage * kHostPage, hi - kHostPage};
    for (uintptr_t at : looks) {
        unsigned char there = 1;
        if (mincore((void*)at, kHostPage, &there) != 0) return false;
        if (!(there & 1)) return true;
    }
    return false;
}

// Makes the pages of large result buffers present while the device still works
// on what goes there.  A fresh array's pages are zeroed one fault at a time,
// inside the copy otherwise, which then runs at 10 GB/s instead of 25.  The
// contents stay; where the kernel or the mapping does not take the advice, the
// copy faults as before.  Small buffers, and those whose pages are there, are
// left to the copy (advice for pages that are there cost 7 % of collecting two
// fields of 9 MB and 17 MB: 1042 -> 1119 us, 1981 -> 2130; with the look 1070 and
// 2004).  Returns the threads it took.
inline int make_present(std::initializer_list<std::pair<void*, size_t>> bufs)
{
    constexpr size_t kSmall = 8u << 20, kThreads = 4;
    std::vector<std::thread> pool;
    try {
        for (auto [p, bytes] : bufs) {
            if (!p || bytes < kSmall) continue;
            const uintptr_t lo = ((uintptr_t)p + kHostPage - 1) / kHostPage * kHostPage;
            const uintptr_t hi = ((uintptr_t)p + bytes) / kHostPage * kHostPage;
            if (!pages_absent(lo, hi)) continue;
            const size_t part = ((hi - lo) / kThreads + kSmall - 1) / kSmall * kSmall;
            for (uintptr_t q = lo; q < hi; q += part)
                pool.emplace_back([=] { (void)madvise((void*)q, std::min<size_t>(part, hi - q), 23 /* MADV_POPULATE_WRITE */); });
        }
    } catch (...) {  // no thread to be had: the copy does the rest
    }
    for (auto& t : pool) t.join();
    return (int)pool.size();
}

}  // namespace cupf
