"""State kept per device (csrc/per_device.h) and not per process."""
import os
import re
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "alpaca_amd", "csrc")

PROGRAM = r"""
#include "per_device.h"
#include <cassert>
#include <thread>
#include <vector>

int main() {
    OncePerDevice once;
    int calls[70] = {};
    auto set = [&](int dev, int result) { return once(dev, [&] { calls[dev]++; return result; }); };
    assert(set(0, 0) == 0 && set(0, 0) == 0 && calls[0] == 1);    // once on a device
    assert(set(1, 0) == 0 && set(63, 0) == 0 && calls[1] == 1 && calls[63] == 1);  // and on each of them
    assert(set(2, 7) == 7 && set(2, 7) == 7 && calls[2] == 2);    // a failure is not kept
    assert(set(2, 0) == 0 && set(2, 7) == 0 && calls[2] == 3);
    assert(set(64, 0) == 0 && set(64, 0) == 0 && calls[64] == 2);  // past the bits: every call
    OncePerDevice shared;
    std::atomic<int> n{0};
    std::vector<std::thread> t;
    for (int i = 0; i < 8; i++)
        t.emplace_back([&] { for (int d = 0; d < 64; d++) assert(shared(d, [&] { n++; return 0; }) == 0); });
    for (auto& x : t) x.join();
    assert(n >= 64 && n <= 8 * 64);
    const int before = n;
    for (int d = 0; d < 64; d++) shared(d, [&] { n++; return 0; });
    assert(n == before);
    return 0;
}
"""


def test_once_per_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    subprocess.run([str(exe)], check=True, timeout=60)


def test_function_attributes_are_set_per_device():
    """An attribute set through a function-local static holds for the device that was current first,
    and a first failure for good."""
    for name in sorted(os.listdir(CSRC)):
        text = open(os.path.join(CSRC, name)).read()
        assert not re.search(r"static\s+(const\s+)?hipError_t\s+\w+\s*=", text), name
