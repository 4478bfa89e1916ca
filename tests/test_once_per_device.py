"""What a launch tells a kernel once (how much LDS it asks for): once for every device, by one thread, and nobody launches before
it is done. csrc/once_per_device.h is plain C++ and runs here on the CPU."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "llm-inference-engine-v6_amd", "csrc")
PROGRAM = r"""
#include "once_per_device.h"
#include <chrono>
#include <cstdio>
#include <thread>
#include <vector>
static llme::OncePerDevice told;
int main() {
    constexpr int N = 3;
    std::atomic<int> calls[N] = {}, done[N] = {}, early{0};
    std::vector<std::thread> threads;
    for (int i = 0; i < 24; ++i)
        threads.emplace_back([&, i] {
            const int device = i % N;
            const int status = told(device, 1000, [&] {
                ++calls[device];
                std::this_thread::sleep_for(std::chrono::milliseconds(30));
                done[device] = 1;
                return 0;
            });
            if (status != 0 || !done[device]) ++early;
        });
    for (auto& t : threads) t.join();
    if (early) return std::puts("a thread went on before it was done"), 1;
    for (int d = 0; d < N; ++d)
        if (calls[d] != 1) return std::printf("device %d: %d calls\n", d, calls[d].load()), 1;
    int more = 0;
    if (told(0, 900, [&] { return ++more, 0; }) || more != 0) return std::puts("told again for less"), 1;
    if (told(0, 2000, [&] { return ++more, 0; }) || more != 1) return std::puts("not told of more"), 1;
    if (told(9, 10, [] { return 7; }) != 7) return std::puts("a failure is lost"), 1;
    if (told(9, 10, [&] { return ++more, 0; }) || more != 2) return std::puts("not tried again behind a failure"), 1;
    if (told(-1, 10, [&] { return ++more, 0; }) || told(1000, 10, [&] { return ++more, 0; }) || more != 4)
        return std::puts("devices out of range are told every time"), 1;
    std::puts("ok");
}
"""


def test_once_per_device(tmp_path):
    cxx = shutil.which(os.environ.get("CXX", "g++")) or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    (tmp_path / "main.cpp").write_text(PROGRAM)
    exe = str(tmp_path / "once")
    built = subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", "-I", CSRC, "-o", exe, str(tmp_path / "main.cpp")],
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    assert built.returncode == 0, built.stdout
    run = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=60)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout


def test_every_kernel_is_told_through_it():
    """(a flag of the launching function's own is one for the whole process, and two threads race on it)"""
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".h")) and name != "common.h":
            with open(os.path.join(CSRC, name)) as f:
                assert "hipFuncSetAttribute(" not in f.read(), name
