"""The conversion of a downloaded field by several threads (sf_widen.h, host only),
in a program of its own whose allocations fail one after another: whatever fails,
every value arrives and no thread is left behind; a copy that fails is
reported."""
import os
import subprocess

from conftest import ROOT

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <stdexcept>

#include "sf_widen.h"

static std::atomic<long> left{-1};   // allocations until they fail; -1: never
static std::atomic<bool> all_after{false};
void* operator new(std::size_t n) {
    const long k = left.load();
    if (k == 0) {
        if (!all_after) left = -1;
        throw std::bad_alloc();
    }
    if (k > 0) left = k - 1;
    if (void* p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

template <typename X>
int run(std::size_t n, int fail, bool after) {
    std::vector<X> src(n);
    std::vector<double> dst(n, -1.0);
    for (std::size_t k = 0; k < n; ++k) src[k] = (X)(k * 0.5);
    all_after = after;
    left = fail;
    sfh::widen(src.data(), n, dst.data(), [] { std::this_thread::yield(); });
    left = -1;
    for (std::size_t k = 0; k < n; ++k)
        if (dst[k] != (double)src[k]) {
            std::printf("n %zu fail %d: value %zu\n", n, fail, k);
            return 1;
        }
    return 0;
}

int main() {
    int bad = 0;
    for (std::size_t n : {(std::size_t)1, sfh::kWidenSerial - 1, sfh::kWidenSerial, sfh::kWidenSerial + 77})
        for (int fail = -1; fail < 24; ++fail)
            for (bool after : {false, true}) bad += run<float>(n, fail, after) + run<double>(n, fail, after);
    for (int fail = -1; fail < 24; ++fail) {
        std::vector<float> src(sfh::kWidenSerial + 5);
        std::vector<double> dst(src.size());
        all_after = false;
        bool thrown = false;
        left = fail;
        try {
            sfh::widen(src.data(), src.size(), dst.data(), [] { throw std::range_error("copy"); });
        } catch (const std::range_error&) {
            thrown = true;
        } catch (const std::bad_alloc&) {
            thrown = true;   // (the failure fell on the error's own text)
        }
        left = -1;
        bad += !thrown;
    }
    std::printf("%d\n", bad);
    return bad != 0;
}
"""


def test_every_failing_allocation(tmp_path):
    src, exe = tmp_path / "widen.cpp", tmp_path / "widen"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-pthread", "-I",
                    os.path.join(ROOT, "soapbubble_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, (r.returncode, r.stdout[-500:], r.stderr[-500:])
