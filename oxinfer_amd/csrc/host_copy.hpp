// Copies between host buffers by several threads (the results of the host surface on their way out of page-locked memory).
#pragma once
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <exception>
#include <thread>

namespace oxhip {

struct HostCopy {
    void* dst;
    const void* src;
    size_t bytes;
};

constexpr size_t COPY_THREADS = 8, COPY_PER_THREAD = (size_t)2 << 20;

// Copies the pieces, large ones by several threads: a thread moves some 10 GB/s between page-locked and ordinary memory, a
// fifth of what the host link does. Every piece of work is done when it returns, also where no thread could be started. Pieces whose
// destinations overlap go one after the other, by the caller: what a later one writes stays.
inline void host_copy(const HostCopy* pieces, size_t n) {
    size_t total = 0;
    for (size_t i = 0; i < n; i++) total += pieces[i].bytes;
    auto range = [pieces, n](size_t lo, size_t hi) {  // bytes lo .. hi of the pieces in a row
        size_t at = 0;
        for (size_t i = 0; i < n && at < hi; at += pieces[i++].bytes) {
            const size_t a = lo > at ? lo - at : 0, b = hi - at < pieces[i].bytes ? hi - at : pieces[i].bytes;
            if (a < b) std::memcpy(static_cast<char*>(pieces[i].dst) + a, static_cast<const char*>(pieces[i].src) + a, b - a);
        }
    };
    bool overlap = false;
    for (size_t i = 1; i < n; i++)
        for (size_t j = 0; j < i; j++) {
            const uintptr_t a = reinterpret_cast<uintptr_t>(pieces[i].dst), b = reinterpret_cast<uintptr_t>(pieces[j].dst);
            overlap |= a < b + pieces[j].bytes && b < a + pieces[i].bytes;
        }
    size_t parts = overlap ? 1 : total / COPY_PER_THREAD;
    parts = parts < 1 ? 1 : parts > COPY_THREADS ? COPY_THREADS : parts;
    const size_t per = ((total + parts - 1) / parts + 4095) / 4096 * 4096;
    std::thread th[COPY_THREADS];
    size_t k = 1;  // part 0 is the caller's
    try {
        for (; k < parts; k++) th[k] = std::thread(range, k * per < total ? k * per : total, (k + 1) * per < total ? (k + 1) * per : total);
    } catch (const std::exception&) {  // no more threads, or no memory for one's state: the caller does the rest
    }
    range(0, per < total ? per : total);
    if (k < parts) range(k * per < total ? k * per : total, total);
    for (size_t i = 1; i < k; i++) th[i].join();
}

}  // namespace oxhip
