// host_copy.h -- host copies into memory the caller has not touched yet.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstring>
#include <thread>

namespace custen {

// Such a copy is bound by page faults (2 MB take 0.9 ms), which the kernel serves
// in parallel: it is split over up to 8 of the machine's `hw` threads, with 512 KB
// each at least.  What no thread can be had for (std::system_error, or no memory
// for one) is copied here.
inline void copyOut(double* dst, const double* src, size_t count,
                    unsigned hw = std::thread::hardware_concurrency())
{
    constexpr size_t kSplitBytes = size_t(512) << 10;
    const size_t parts = std::min({count * sizeof(double) / kSplitBytes, (size_t)hw, (size_t)8});
    if (parts <= 1) {
        std::memcpy(dst, src, count * sizeof(double));
        return;
    }
    const size_t chunk = (count + parts - 1) / parts;
    std::thread workers[8];
    size_t rest = count;  // where the workers' parts begin
    try {
        for (size_t t = parts - 1; t > 0; t--) {
            const size_t b = t * chunk, e = rest;
            if (b >= e) continue;
            workers[t] = std::thread([=]() { std::memcpy(dst + b, src + b, (e - b) * sizeof(double)); });
            rest = b;
        }
    } catch (...) {
    }
    std::memcpy(dst, src, rest * sizeof(double));
    for (std::thread& w : workers)
        if (w.joinable()) w.join();
}

}  // namespace custen
