// Copies between host buffers on a few threads.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

namespace tah {

// bytes from one host buffer to another, sliced over a few threads when large (one thread copies to pages it touches
// for the first time at about 10 GB/s, less than the card delivers them). Never throws: where a thread cannot be had
// (its start allocates as well, so either std::system_error or std::bad_alloc), its slice and the rest are copied here,
// and the threads that run are waited for.
inline void host_copy(uint8_t *dst, const uint8_t *src, size_t bytes) {
    constexpr size_t SLICE = 2 << 20;
    const size_t n = std::min<size_t>(8, bytes / SLICE);
    if (n < 2) {
        std::memcpy(dst, src, bytes);
        return;
    }
    const size_t step = (bytes / n + 4095) & ~size_t(4095);
    std::vector<std::thread> threads;
    size_t at = step;  // the first slice is this thread's
    try {
        threads.reserve(n);
        for (; at < bytes; at += step) {
            const size_t k = std::min(step, bytes - at);
            threads.emplace_back([=] { std::memcpy(dst + at, src + at, k); });
        }
    } catch (...) {
        std::memcpy(dst + at, src + at, bytes - at);
    }
    std::memcpy(dst, src, std::min(step, bytes));
    for (auto &t : threads) t.join();
}

}  // namespace tah
