"""The threaded copy of the host surface's results (csrc/host_copy.hpp), compiled for the CPU."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oxinfer_amd", "csrc")

PROGRAM = r"""
#include "host_copy.hpp"
#include <cstdlib>
#include <new>
#include <vector>

// allocations that still succeed (-1: all of them); std::thread allocates its state
static long left = -1;
void* operator new(size_t n) {
    if (left == 0) throw std::bad_alloc();
    if (left > 0) left--;
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, size_t) noexcept { std::free(p); }

int main(int argc, char** argv) {
    const long threads = std::atol(argv[1]);  // that may start
    std::vector<size_t> sizes;
    for (int i = 2; i < argc; i++) sizes.push_back((size_t)std::atoll(argv[i]));
    std::vector<std::vector<unsigned char>> src, dst;
    std::vector<oxhip::HostCopy> pieces;
    for (size_t i = 0; i < sizes.size(); i++) {
        src.emplace_back(sizes[i]);
        for (size_t k = 0; k < sizes[i]; k++) src[i][k] = (unsigned char)(k * 31 + (k >> 12) + i);
        dst.emplace_back(sizes[i] + 1, 0xEE);
    }
    for (size_t i = 0; i < sizes.size(); i++) pieces.push_back({dst[i].data(), src[i].data(), sizes[i]});
    left = threads;
    oxhip::host_copy(pieces.data(), pieces.size());
    left = -1;
    for (size_t i = 0; i < sizes.size(); i++)
        if (std::memcmp(dst[i].data(), src[i].data(), sizes[i]) || dst[i][sizes[i]] != 0xEE) return 1;
    return 0;
}
"""


@pytest.fixture(scope="module")
def build(tmp_path_factory):
    def build(program):
        d = tmp_path_factory.mktemp("host_copy")
        (d / "main.cpp").write_text(program)
        subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", CSRC, str(d / "main.cpp"), "-o", str(d / "main")], check=True)
        return str(d / "main")
    return build


def test_every_byte_arrives_whatever_threads_start(build):
    exe = build(PROGRAM)
    for sizes in ((0,), (1,), (4096, 0, 5), (3 << 20, 1, (5 << 20) + 77), (40 << 20,), tuple([1000003] * 20)):
        for threads in (-1, 0, 1, 3):  # all, none for want of memory, one, three
            r = subprocess.run([exe, str(threads), *map(str, sizes)], timeout=60)
            assert r.returncode == 0, (sizes, threads, r.returncode)


OVERLAP = r"""
#include "host_copy.hpp"
#include <algorithm>
#include <vector>

int main() {
    // two results to one place, and one that begins in the middle of another (both ways round in address order): the later job's stay
    const size_t n = 24 << 20;
    std::vector<unsigned char> a(n, 1), b(n, 2), y(2 * n);
    for (int k = 0; k < 3; k++) {
        std::fill(y.begin(), y.end(), 0);
        unsigned char *first = y.data() + (k == 2 ? n / 2 : 0), *second = y.data() + (k == 1 ? n / 2 : 0);
        const oxhip::HostCopy pieces[] = {{first, a.data(), n}, {second, b.data(), n}};
        oxhip::host_copy(pieces, 2);
        for (size_t i = 0; i < 2 * n; i++) {
            const unsigned char* p = y.data() + i;
            const unsigned char want = p >= second && p < second + n ? 2 : p >= first && p < first + n ? 1 : 0;
            if (*p != want) return 1;
        }
    }
    return 0;
}
"""


def test_overlapping_results_keep_the_order_of_the_jobs(build):
    exe = build(OVERLAP)
    for _ in range(3):
        assert subprocess.run([exe], timeout=60).returncode == 0


ARRIVING = r"""
#include "host_copy.hpp"
#include <algorithm>
#include <cstdlib>
#include <vector>

static unsigned char old_byte(size_t k) { return (unsigned char)(k * 7 + (k >> 11) + 5); }
static unsigned char new_byte(size_t k) { return (unsigned char)(k * 31 + (k >> 12) + 1); }

// argv: the chunk that never comes (-1: all come), bytes by which the second piece's destination lies inside the first's, the chunks'
// ends; two pieces, the second a third of the bytes
int main(int argc, char** argv) {
    const long never = std::atol(argv[1]);
    std::vector<size_t> ends;
    for (int i = 3; i < argc; i++) ends.push_back((size_t)std::atoll(argv[i]));
    const size_t total = ends.back(), first = total - total / 3, back = std::min((size_t)std::atoll(argv[2]), first);
    const size_t at2 = first + 1 - (back ? back + 1 : 0);  // (one byte lies between them where they do not overlap)
    std::vector<unsigned char> src(total + 1, 0), dst(total + 2), want;
    for (size_t k = 0; k < dst.size(); k++) dst[k] = old_byte(k);
    want = dst;
    if (never < 0) {
        for (size_t k = 0; k < first; k++) want[k] = new_byte(k);
        // overlapping ranges are written chunk by chunk, the later piece's bytes of a chunk last
        for (size_t c = 0; back && c < ends.size(); c++)
            for (size_t k = c ? ends[c - 1] : 0; k < ends[c]; k++) want[k < first ? k : at2 + k - first] = new_byte(k);
        for (size_t k = first; !back && k < total; k++) want[at2 + k - first] = new_byte(k);
    }
    const oxhip::HostCopy pieces[2] = {{dst.data(), src.data(), first}, {dst.data() + at2, src.data() + first, total - first}};
    size_t told = 0;
    const bool ok = oxhip::host_copy_arriving(pieces, 2, ends.data(), ends.size(), 4096, [&](size_t c) {
        if (c != told++ || (long)c == never) return false;
        for (size_t k = c ? ends[c - 1] : 0; k < ends[c]; k++) src[k] = new_byte(k);
        return true;
    });
    if (ok != (never < 0) || told != (never < 0 ? ends.size() : (size_t)never + 1)) return 1;
    return dst == want ? 0 : 2;
}
"""


def test_all_chunks_are_copied_or_nothing_is(build):
    """Each chunk by all threads once it has come, in order; after one that never comes every destination is as it was, also where
    destinations overlap."""
    exe = build(ARRIVING)
    for ends in ((1,), (4096,), (3000, 3000, 9001), (5 << 20, 9 << 20, 12 << 20, 14 << 20, (15 << 20) - 3)):
        for never in (-1, *range(len(ends))):
            for back in (0, ends[-1] // 4):
                r = subprocess.run([exe, str(never), str(back), *map(str, ends)], timeout=60)
                assert r.returncode == 0, (ends, never, back)


WAITING = r"""
#include "host_copy.hpp"
#include <chrono>
#include <filesystem>
#include <sys/resource.h>
#include <vector>

static long threads() {
    long n = 0;
    for (const auto& e : std::filesystem::directory_iterator("/proc/self/task")) n += e.path().filename() != ".";
    return n;
}
static double cpu_seconds() {
    rusage u{};
    getrusage(RUSAGE_SELF, &u);
    return u.ru_utime.tv_sec + u.ru_stime.tv_sec + 1e-6 * (u.ru_utime.tv_usec + u.ru_stime.tv_usec);
}

int main() {
    std::vector<size_t> ends = {1 << 20, 2 << 20, 3 << 20};
    std::vector<unsigned char> src(ends.back(), 1), dst(ends.back(), 0);
    const oxhip::HostCopy piece{dst.data(), src.data(), ends.back()};
    const double before = cpu_seconds();
    bool early = false;
    const bool ok = oxhip::host_copy_arriving(&piece, 1, ends.data(), ends.size(), 4096, [&](size_t c) {
        std::this_thread::sleep_for(std::chrono::milliseconds(200));
        early |= c == 0 && threads() != 1;
        return true;
    });
    return !ok || early || cpu_seconds() - before > 0.15 || dst != std::vector<unsigned char>(ends.back(), 1);  // (a thread that spins through the waits alone takes 0.6 s)
}
"""


def test_waiting_for_chunks_costs_no_core(build):
    """No thread before the first chunk has come, and none that spins until the next one."""
    assert subprocess.run([build(WAITING)], timeout=60).returncode == 0
