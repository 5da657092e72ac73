"""LdsLimit (gsd_lds_limit.h) with threads whose launches need different sizes,
on the CPU: once raise() has returned, the limit set is never below its size."""
import os
import shutil
import subprocess

from gsdlq import build

PROGRAM = r"""
#include "gsd_lds_limit.h"
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>

// the runtime's side of it: the limit last set, after a while of its own
static std::atomic<size_t> runtime{0};
static int set(size_t n) {
    std::this_thread::sleep_for(std::chrono::microseconds(50 * (1 + n % 3)));
    runtime = n;
    return 0;
}

int main() {
    int bad = 0;
    for (int round = 0; round < 200; round++) {
        gsd::LdsLimit limit;
        std::atomic<int> wrong{0}, ready{0};
        runtime = 0;
        std::vector<std::thread> threads;
        for (size_t i = 0; i < 4; i++)
            threads.emplace_back([&, i] {
                ready++;
                while (ready < 4) {}
                for (size_t n : {1000 + i, 1007 - i, 1000 + i})   // (up, and down again)
                    for (int k = 0; k < 20; k++) {
                        if (limit.raise(n, set)) wrong++;
                        if (runtime < n) wrong++;
                    }
            });
        for (auto& t : threads) t.join();
        bad += wrong != 0;
    }
    // what could not be set is not taken for set
    gsd::LdsLimit limit;
    int calls = 0;
    auto fails = [&](size_t) { calls++; return 7; };
    if (limit.raise(5, fails) != 7 || limit.raise(5, fails) != 7 || calls != 2) bad++;
    if (limit.raise(5, set) || limit.raise(4, fails)) bad++;
    std::printf("%d\n", bad);
    return bad != 0;
}
"""


def test_limit_of_two_threads(tmp_path):
    src, exe = tmp_path / "limit.cpp", tmp_path / "limit"
    src.write_text(PROGRAM)
    cxx = shutil.which("g++") or "g++"
    subprocess.run([cxx, "-O2", "-std=c++17", "-pthread", "-I", os.fspath(build.CSRC), os.fspath(src), "-o", os.fspath(exe)],
                   check=True, timeout=120)
    r = subprocess.run([os.fspath(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, f"rounds with a limit below a launch's size: {r.stdout}"
