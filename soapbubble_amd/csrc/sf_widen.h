// Downloaded fields on their way to the caller's array (host only).
#pragma once

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <exception>
#include <thread>
#include <vector>

namespace sfh {

// Values widened from a staging buffer to the caller's FP64 array once
// `arrived` returns. The caller's array is usually fresh memory, whose first
// touch (a page fault and its clearing, 0.5 ms for the 16 MB of a 1024x2048
// field) costs more than the copy (0.2 ms over PCIe) and the conversion: large
// arrays are cut among a few threads, which touch their part's pages while
// the copy runs and convert it when it has arrived. A field, against a pageable
// copy into a cleared temporary and one thread: 1024x2048 1.03 -> 0.28 ms, in FP64
// 1.9-4.8 -> 0.5, 2048x4096 12 -> 2.0, 64x128 in FP64 0.038 -> 0.014.
constexpr size_t kWidenSerial = (size_t)1 << 20;   // values below which one thread does it
template <typename X, typename Arrived>
void widen(const X* src, size_t n, double* dst, Arrived&& arrived) {
    const size_t cpus = std::max(1u, std::thread::hardware_concurrency());
    const size_t parts = n < kWidenSerial ? 1 : std::min<size_t>(8, cpus);
    auto convert = [&](size_t a, size_t b) {
        for (size_t k = a; k < b; ++k) dst[k] = (double)src[k];
    };
    if (parts == 1) {
        arrived();
        convert(0, n);
        return;
    }
    const size_t each = ((n + parts - 1) / parts + 511) / 512 * 512;
    std::atomic<int> state{0};   // 1: arrived, 2: the copy failed
    auto part = [&](size_t a, size_t b) {
        for (size_t k = a; k < b; k += 512) dst[k] = 0.0;
        while (state.load(std::memory_order_acquire) == 0) std::this_thread::yield();
        if (state.load(std::memory_order_relaxed) == 1) convert(a, b);
    };
    std::vector<std::thread> crew;
    size_t own = each;   // the parts from here on are this thread's
    try {
        // (room for all first: no growth, which can fail, beside running threads)
        crew.reserve(parts);
        for (size_t a = each; a < n; a += each) {
            crew.emplace_back(part, a, std::min(n, a + each));
            own = std::min(n, a + each);
        }
    } catch (const std::exception&) {
        // no thread or no memory for one: what is left is this thread's
    }
    auto finish = [&](int how) {
        state.store(how, std::memory_order_release);
        if (how == 1) {
            convert(0, std::min(each, n));
            if (own < n) convert(own, n);
        }
        for (std::thread& t : crew) t.join();
    };
    try {
        for (size_t k = 0; k < std::min(each, n); k += 512) dst[k] = 0.0;
        arrived();
    } catch (...) {
        finish(2);
        throw;
    }
    finish(1);
}

}  // namespace sfh
