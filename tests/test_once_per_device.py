"""once.h on the CPU: the dynamic LDS limit of a kernel is asked for on every device, once, and again after a failure."""
import os
import subprocess

from conftest import ROOT

SRC = r"""
#include <cstdio>
#include <thread>
#include <vector>
#include "once.h"
static int check(bool ok, int line) { if (!ok) std::printf("line %d\n", line); return ok ? 0 : 1; }
int main() {
    std::atomic<uint64_t> done{0};
    int calls[70] = {}, bad = 0, fail = 0;
    auto on = [&](int d) { return lstk::once_per_device(done, d, [&] { calls[d]++; return fail; }); };
    for (int i = 0; i < 3; i++) for (int d : {0, 1, 63}) bad += check(on(d) == 0, __LINE__);
    bad += check(calls[0] == 1 && calls[1] == 1 && calls[63] == 1, __LINE__);
    fail = 7;
    bad += check(on(5) == 7 && on(0) == 0, __LINE__); // a failure on one device is that device's own
    fail = 0;
    bad += check(on(5) == 0 && on(5) == 0 && calls[5] == 2, __LINE__);
    bad += check(on(64) == 0 && on(64) == 0 && calls[64] == 2, __LINE__); // past the bits: every time
    std::atomic<uint64_t> d2{0};
    std::atomic<int> n{0};
    std::vector<std::thread> ts;
    for (int i = 0; i < 8; i++) ts.emplace_back([&, i] { for (int r = 0; r < 1000; r++) lstk::once_per_device(d2, i % 4, [&] { n++; return 0; }); });
    for (auto &t : ts) t.join();
    bad += check(n >= 4 && n <= 8 && d2 == 15, __LINE__);
    return bad;
}
"""


def test_once_per_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-pthread", "-I", os.path.join(ROOT, "localstack_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, timeout=100)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout
