"""The radix sort's scratch covers every sort that a handle of that capacity
can run: histogram table, digit totals and ping-pong halves of each particle
count up to the capacity, on both sides of the counts where the digits change
width, for every key width.  Host code only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include <cstdio>
#include <vector>
#include "mpm_radix_plan.hpp"
using namespace mpm;
int main() {
    std::vector<uint32_t> counts;  // around every change of the digit width, and far beyond
    for (uint64_t nb : {1, 2, 63, 64, 65, 74, 127, 128, 129, 255, 256, 257, 511, 512, 513, 700, 2048, 262144})
        for (int64_t d : {-4095, -1, 0, 1, 2048})
            if (int64_t(nb) * SORT_TILE + d > 0 && int64_t(nb) * SORT_TILE + d < (1ll << 30))
                counts.push_back(uint32_t(int64_t(nb) * SORT_TILE + d));
    long bad = 0, seen = 0;
    for (uint32_t cap : counts)
        for (uint32_t n : counts) {
            if (n > cap) continue;
            for (int bits = 1; bits <= 26; ++bits, ++seen) {
                const RadixPlan p = radix_plan(n, bits);
                const size_t digits = size_t(1) << p.width;
                const size_t used = 2 * size_t(n) + digits * sort_blocks(n) + digits;
                if (p.passes * p.width < bits || p.width > MAX_DIGIT || used > radix_scratch_words(cap)) {
                    if (bad++ < 5)
                        std::printf("cap %u n %u bits %d: %zu words used, %zu there\n", cap, n, bits, used,
                                    radix_scratch_words(cap));
                }
            }
        }
    std::printf("%ld plans, %ld too large\n", seen, bad);
    return bad != 0;
}
"""


def test_scratch_of_a_capacity_covers_every_smaller_sort(tmp_path):
    src, exe = tmp_path / "check.cpp", tmp_path / "check"
    src.write_text(CHECK)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(ROOT, "molla_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
