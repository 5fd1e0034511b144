// Copies between host buffers by several threads (the results of the host surface on their way out of page-locked memory).
#pragma once
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>

#include <emmintrin.h>

namespace oxhip {

struct HostCopy {
    void* dst;
    void* src;  // (staging: where bytes come in several chunks it holds others afterwards)
    size_t bytes;
};

constexpr size_t COPY_THREADS = 8, COPY_PER_THREAD = (size_t)2 << 20, COPY_SHARE = (size_t)256 << 10;

// `dst` receives the bytes of `src` and `src` those that `dst` held. What goes to `src` is written past the caches: left dirty there, it
// would meet the next transfer (59 MB of results, half a dozen runs: a call takes 1.60 to 1.71 ms if they are only copied, 1.71 to 1.90
// exchanged through the caches, 1.69 to 1.87 this way; copied after the last chunk has come, 2.01).
inline void host_exchange(char* dst, char* src, size_t n) {
    auto few = [&](size_t at, size_t len) {  // up to 64 bytes
        char old[64];
        std::memcpy(old, dst + at, len);
        std::memcpy(dst + at, src + at, len);
        std::memcpy(src + at, old, len);
    };
    const size_t head = (64 - reinterpret_cast<uintptr_t>(src) % 64) % 64;
    size_t at = head < n ? head : n;
    few(0, at);
    for (; at + 64 <= n; at += 64) {
        __m128i was[4], is[4];
        for (int i = 0; i < 4; i++) {
            was[i] = _mm_loadu_si128(reinterpret_cast<const __m128i*>(dst + at) + i);
            is[i] = _mm_load_si128(reinterpret_cast<const __m128i*>(src + at) + i);
        }
        for (int i = 0; i < 4; i++) _mm_storeu_si128(reinterpret_cast<__m128i*>(dst + at) + i, is[i]);
        for (int i = 0; i < 4; i++) _mm_stream_si128(reinterpret_cast<__m128i*>(src + at) + i, was[i]);
    }
    few(at, n - at);
    _mm_sfence();
}

// Copies the pieces while their bytes arrive: chunk c of `chunks` ends at byte ends[c] of all of them in a row (the last one at their
// end). wait(c), called by the caller's thread for c = 0, 1, ... in order, returns once chunk c is there, or false if it never will be:
// then the result is false and every destination holds what it held before. (Up to the last chunk, whose coming ends all doubt,
// destination and staging exchange their bytes, so that what was overwritten can be put back.) Large chunks go by several threads,
// each its share of every chunk: a thread moves some 10 GB/s between page-locked and ordinary memory, a fifth of what the host link
// does. The threads start when the first chunk has come and sleep until the next one: what it takes before (the kernels that make
// the bytes) costs no core. Every piece of work is done when it returns, also where no thread could be started. Pieces whose
// destinations overlap go one after the other, by the caller: what a later one writes stays.
template <class Wait>
inline bool host_copy_arriving(const HostCopy* pieces, size_t n, const size_t* ends, size_t chunks, size_t per_thread, Wait wait) {
    enum { COPY, EXCHANGE, PUT_BACK };
    auto range = [pieces, n](size_t lo, size_t hi, int how) {  // bytes lo .. hi of the pieces in a row (put back: the last piece first)
        auto part = [&](size_t i, size_t at) {
            const size_t a = lo > at ? lo - at : 0, b = hi - at < pieces[i].bytes ? hi - at : pieces[i].bytes;
            if (a >= b) return;
            char *dst = static_cast<char*>(pieces[i].dst) + a, *src = static_cast<char*>(pieces[i].src) + a;
            if (how == COPY) std::memcpy(dst, src, b - a);
            else host_exchange(dst, src, b - a);
        };
        size_t i = 0, at = 0;
        for (; i < n && at < hi; at += pieces[i++].bytes)
            if (how != PUT_BACK) part(i, at);
        while (how == PUT_BACK && i-- > 0) part(i, at -= pieces[i].bytes);
    };
    bool overlap = false;
    for (size_t i = 1; i < n; i++)
        for (size_t j = 0; j < i; j++) {
            const uintptr_t a = reinterpret_cast<uintptr_t>(pieces[i].dst), b = reinterpret_cast<uintptr_t>(pieces[j].dst);
            overlap |= a < b + pieces[j].bytes && b < a + pieces[i].bytes;
        }
    size_t parts = overlap ? 1 : ends[chunks - 1] / chunks / per_thread;
    parts = parts < 1 ? 1 : parts > COPY_THREADS ? COPY_THREADS : parts;
    auto share = [=](size_t k, size_t c, int how) {  // thread k's share of chunk c
        const size_t lo = c ? ends[c - 1] : 0, hi = ends[c], per = ((hi - lo + parts - 1) / parts + 4095) / 4096 * 4096;
        range(lo + k * per < hi ? lo + k * per : hi, lo + (k + 1) * per < hi ? lo + (k + 1) * per : hi, how);
    };
    auto bring = [=](size_t k, size_t c) { share(k, c, c + 1 == chunks ? COPY : EXCHANGE); };
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
            bring(k, c);
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
        bring(0, c);
        for (size_t i = k; i < parts; i++) bring(i, c);
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
    if (!ok)  // every thread has brought all that came
        for (size_t c = arrived; c-- > 0;)
            for (size_t i = 0; i < parts; i++) share(i, c, PUT_BACK);
    return ok;
}

// The same for bytes that are there.
inline void host_copy(const HostCopy* pieces, size_t n) {
    size_t total = 0;
    for (size_t i = 0; i < n; i++) total += pieces[i].bytes;
    (void)host_copy_arriving(pieces, n, &total, 1, COPY_PER_THREAD, [](size_t) { return true; });
}

}  // namespace oxhip
