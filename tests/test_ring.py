"""The ring of staging slots (geode_amd/csrc/ring.hpp) stays within its slots and in turn past 2^32 uses, where a count of
the uses would have wrapped twice. CPU: the header alone, built with g++."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include "ring.hpp"
int main() {
    gv::Ring<8> ring;
    for (unsigned long long i = 0; i < (1ull << 32) + 64; ++i) {
        const int s = ring.take();
        if (s < 0 || s >= 8 || s != static_cast<int>(i % 8)) return 1;
    }
    return 0;
}
"""


def test_slots_past_the_range_of_an_int(tmp_path):
    src, exe = tmp_path / "ring.cpp", tmp_path / "ring"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(ROOT, "geode_amd", "csrc"), str(src),
                    "-o", str(exe)], check=True, timeout=60)
    assert subprocess.run([str(exe)], timeout=100).returncode == 0
