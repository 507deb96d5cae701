"""The dynamic-LDS limit of a kernel is one per process: no planner lowers what another launch relies on."""
import glob
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "fusekit_amd", "csrc")

PROGRAM = r"""
#include <atomic>
#include <cstdio>
#include <thread>
#include <vector>
#include "lds_limit.hpp"

static std::atomic<uint32_t> runtime_limit[3];   // what the runtime holds
static fk::LdsLimits limits;

static int raise(int kernel, uint32_t bytes) {
    return limits.raise(&runtime_limit[kernel], bytes, [&](uint32_t b) {
        if (b > 160u * 1024u) return 1;
        runtime_limit[kernel] = b;
        return 0;
    });
}

int main() {
    // two shapes of a kernel in turn, the wider one planned once
    if (raise(0, 80000) || raise(0, 56000) || runtime_limit[0] != 80000) return 1;
    // refused: nothing is taken as allowed, the next one asks again
    if (raise(1, 200000) != 1 || raise(1, 60000) || runtime_limit[1] != 60000) return 2;
    // threads that plan different shapes: each launch finds what it asked for, or more
    std::atomic<int> low{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; ++t)
        threads.emplace_back([&, t] {
            for (uint32_t i = 0; i < 2000; ++i) {
                const uint32_t bytes = 49152u + (i * 7919u + (uint32_t)t * 104729u) % 100000u;
                if (raise(2, bytes) || runtime_limit[2] < bytes) ++low;
            }
        });
    for (auto& t : threads) t.join();
    return low ? 3 : 0;
}
"""


def test_limits_only_rise(tmp_path):
    src, exe = tmp_path / "limits.cpp", tmp_path / "limits"
    src.write_text(PROGRAM)
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-pthread", "-Wall", "-Wextra", "-I", CSRC, str(src), "-o", str(exe)])
    assert subprocess.run([str(exe)], timeout=60).returncode == 0


def test_every_planner_goes_through_the_limits():
    users = {os.path.basename(f): open(f).read().count("hipFuncSetAttribute(") for f in glob.glob(os.path.join(CSRC, "*.h*"))}
    assert {f: n for f, n in users.items() if n} == {"capi.hip": 1}
