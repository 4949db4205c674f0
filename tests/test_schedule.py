"""The sweep thresholds that the schedule search times: where the level form
takes every island of a batch, those that it sweeps alike are timed once."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <cstdio>
#include "schedule.hpp"
int main() {
    for (int level = 0; level < 2; ++level)
        for (std::uint32_t cur : {0u, 1u, 3u, 4u, 8u, 32u, 200u, 0x40000000u, 0x7fffffffu, 0xffffffffu}) {
            std::printf("%d %u:", level, cur);
            for (std::uint32_t k : prx::CoopCandidates(level != 0))
                if (!prx::SameSweeps(k, cur, level != 0)) std::printf(" %u", k);
            std::printf("\n");
        }
}
"""
MOST = 0xffffffff


def test_sweep_threshold_candidates(tmp_path):
    src, exe = tmp_path / "schedule.cpp", tmp_path / "schedule"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "playrho_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    got = {}
    for line in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines():
        key, trials = line.split(":")
        got[tuple(int(x) for x in key.split())] = [int(x) for x in trials.split()]
    every = [8, 16, 32, 64, 128, MOST]
    for cur in (0, 1, 3, 4, 8, 32, 200, 0x40000000, 0x7fffffff, MOST):
        assert got[0, cur] == [k for k in every if k != cur], cur
    # Lanes only: the level form; the level form: lanes; smaller islands too: both.
    assert got[1, MOST] == got[1, 0x7fffffff] == [32]
    assert got[1, 4] == got[1, 8] == got[1, 32] == got[1, 200] == got[1, 0x40000000] == [MOST]
    assert got[1, 0] == got[1, 1] == got[1, 3] == [32, MOST]
