"""CPU check of csrc/per_device.h, by which a kernel's LDS limit is raised on every device it runs on."""

import os
import subprocess

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quasi-linear-kernel-attention_amd",
                    "csrc")

PROGRAM = r"""
#include "per_device.h"
#include <cstdio>
int main() {
    qlka::PerDevice once;
    int ran[70] = {}, fail = 0;
    auto at = [&](int d) { return once(d, [&] { ++ran[d]; return fail; }); };
    if (at(0) || at(0) || ran[0] != 1) return 1;               // once on a device
    if (at(1) || at(1) || ran[1] != 1 || ran[0] != 1) return 2;     // and once on the next
    fail = 7;
    if (at(2) != 7 || at(2) != 7 || ran[2] != 2) return 3;     // an error is reported and tried again
    fail = 0;
    if (at(2) || at(2) || ran[2] != 3) return 4;
    if (at(63) || at(63) || ran[63] != 1) return 5;
    if (at(64) || at(64) || ran[64] != 2) return 6;            // beyond the tracked ones: every time
    qlka::PerDevice other;
    if (other(0, [&] { ++ran[0]; return 0; }) || ran[0] != 2) return 7;     // each kernel has its own
    std::puts("ok");
    return 0;
}
"""


def test_once_per_device(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.strip() == "ok"


def test_every_raised_lds_limit_goes_through_it():
    # more than 64 KB of LDS needs the attribute, which belongs to one device's copy of the kernel
    for name in sorted(os.listdir(CSRC)):
        if name.endswith(".hip"):
            text = open(os.path.join(CSRC, name)).read()
            assert text.count("hipFuncSetAttribute(") == text.count("once(dev, [&] {"), name
            assert "static const hipError_t" not in text, name
