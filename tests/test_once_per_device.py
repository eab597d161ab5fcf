"""The once-per-device helper behind the kernels' LDS allowance (mdx_once.h), compiled for the CPU:
an action runs once on each device, not once in the process; a failure is tried again; devices past
the table and calls from several threads are served."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include <cassert>
#include <thread>
#include <vector>
#include "mdx_once.h"
int main() {
    static mdx::OncePerDevice once;
    int runs[3] = {0, 0, 0};
    auto act = [&](int dev, int result) { return once.run(dev, [&] { ++runs[dev]; return result; }); };
    assert(act(0, 0) == 0 && act(0, 0) == 0 && runs[0] == 1);
    assert(act(1, 0) == 0 && runs[1] == 1);   // a second device has its own
    assert(act(2, 7) == 7 && act(2, 0) == 0 && act(2, 0) == 0 && runs[2] == 2);
    int far = 0;
    for (int q = 0; q < 2; ++q) assert(once.run(64, [&] { ++far; return 0; }) == 0);
    assert(far == 2 && once.run(-1, [] { return 5; }) == 5);
    std::atomic<int> n{0};
    std::vector<std::thread> th;
    for (int q = 0; q < 4; ++q) th.emplace_back([&] { for (int r = 0; r < 1000; ++r) once.run(9, [&] { ++n; return 0; }); });
    for (auto &t : th) t.join();
    assert(n >= 1 && n <= 4);
    return 0;
}
"""


def test_runs_once_on_every_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I", os.path.join(ROOT, "mobydiff_amd", "csrc"),
                    str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True, timeout=60)
