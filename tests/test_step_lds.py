"""The LDS that a step asks for: 40 bytes a body for worlds the level form
takes, and no more than their state's 32 for larger ones, which would fit fewer
worlds to a CU for nothing."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "layout.hpp"
int main() {
    std::printf("%d %d\n", prx::kLevelMaxBodies, prx::kStageFloat4 * 16);
    for (int nb = 0; nb <= 2000; ++nb) std::printf("%d\n", prx::StepLdsBytes(nb));
}
"""


def test_lds_of_worlds_beyond_the_level_form(tmp_path):
    src, exe = tmp_path / "lds.cpp", tmp_path / "lds"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "playrho_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    lines = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.split("\n")
    most, stage = (int(x) for x in lines[0].split())
    got = [int(x) for x in lines[1:2002]]
    assert most == 576
    for nb, lds in enumerate(got):
        assert lds == stage + nb * (40 if nb <= most else 32), nb
    per_cu = [160 * 1024 // -(-lds // 256 * 256) for lds in got]
    # Worlds of 1100 and 1500 bodies: four and three to a CU.
    assert (per_cu[1100], per_cu[1500]) == (4, 3)
