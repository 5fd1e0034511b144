// Copies between host buffers by several threads (the results of the host surface on their way out of page-locked memory).
#pragma once
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

namespace oxhip {

struct HostCopy {
    void* dst;
    const void* src;
    size_t bytes;
};

constexpr size_t COPY_THREADS = 8, COPY_PER_THREAD = (size_t)2 << 20, COPY_SHARE = (size_t)256 << 10;

// Copies the pieces while their bytes arrive: chunk c of `chunks` ends at byte ends[c] of all of them in a row (the last one at their
// end). wait(c), called by the caller's thread for c = 0, 1, ... in order, returns once chunk c is there, or false if it never will be
// (then what is not copied yet stays as it was, and the result is false). Large chunks go by several threads, each its share of every
// chunk: a thread moves some 10 GB/s between page-locked and ordinary memory, a fifth of what the host link does. The threads start
// when the first chunk has come and sleep until the next one: what it takes before (the kernels that make the bytes) costs no core.
// Every piece of work is done when it returns, also where no thread could be started. Pieces whose destinations overlap go one after
// the other, by the caller: what a later one writes stays.
template <class Wait>
inline bool host_copy_arriving(const HostCopy* pieces, size_t n, const size_t* ends, size_t chunks, size_t per_thread, Wait wait) {
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
    size_t parts = overlap ? 1 : ends[chunks - 1] / chunks / per_thread;
    parts = parts < 1 ? 1 : parts > COPY_THREADS ? COPY_THREADS : parts;
    auto share = [=](size_t k, size_t c) {  // thread k's share of chunk c
        const size_t lo = c ? ends[c - 1] : 0, hi = ends[c], per = ((hi - lo + parts - 1) / parts + 4095) / 4096 * 4096;
        range(lo + k * per < hi ? lo + k * per : hi, lo + (k + 1) * per < hi ? lo + (k + 1) * per : hi);
    };
    if (!wait(0)) return false;
    std::mutex mu;
    std::condition_variable more;
    size_t arrived = 1;  // chunks (guarded by mu)
    bool never = false;  // no more will come (guarded by mu)
    auto work = [&](size_t k) {
        for (size_t c = 0; c < chunks; c++) {
            {
                std::unique_lock<std::mutex> lk(mu);
                more.wait(lk, [&] { return arrived > c || never; });
                if (arrived <= c) return;
            }
            share(k, c);
        }
    };
    std::thread th[COPY_THREADS];
    size_t k = 1;  // share 0 is the caller's
    try {
        for (; k < parts; k++) th[k] = std::thread(work, k);
    } catch (const std::exception&) {  // no more threads, or no memory for one's state: the caller does the rest
    }
    bool ok = true;
    for (size_t c = 0; ok; c++) {
        share(0, c);
        for (size_t i = k; i < parts; i++) share(i, c);
        if (c + 1 == chunks) break;
        ok = wait(c + 1);
        {
            std::lock_guard<std::mutex> lk(mu);
            if (ok) arrived++;
            else never = true;
        }
        more.notify_all();
    }
    for (size_t i = 1; i < k; i++) th[i].join();
    return ok;
}

// The same for bytes that are there.
inline void host_copy(const HostCopy* pieces, size_t n) {
    size_t total = 0;
    for (size_t i = 0; i < n; i++) total += pieces[i].bytes;
    (void)host_copy_arriving(pieces, n, &total, 1, COPY_PER_THREAD, [](size_t) { return true; });
}

}  // namespace oxhip
