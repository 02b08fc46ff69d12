"""CPU check of the windows in which the minimizer's bonded terms pass through LDS
(csrc/bonded_windows.h, compiled here by the host compiler): with the LDS that a launch reserves,
down to molecules of one atom, every window holds at least one term and no more than the LDS does,
and together they hold every 64-term task once and whole."""
from __future__ import annotations

import subprocess
from pathlib import Path

import numpy as np

CSRC = Path(__file__).resolve().parent.parent / "mlxmolkit_archive_amd" / "csrc"

MAIN = r"""
#include <cstdio>
#include "bonded_windows.h"
// reads lines "words c1 .. c5 max_n" (words 0: the LDS words of a launch of max_n); prints the
// words and the window ends of each, and "stall" where one does not move on
int main() {
  int words, c[5], mn;
  while (std::scanf("%d %d %d %d %d %d %d", &words, c, c + 1, c + 2, c + 3, c + 4, &mn) == 7) {
    if (words == 0) words = mmff::lbfgs_eb_floats(mn);
    std::printf("%d", words);
    for (int s = 0; s < c[4];) {
      const int e = mmff::bonded_window_end({0, c[0], c[1], c[2], c[3], c[4]}, s, words);
      if (e <= s) {
        std::printf(" stall");
        break;
      }
      std::printf(" %d", s = e);
    }
    std::printf("\n");
  }
}
"""


def _run(tmp_path, cases):
    exe = tmp_path / "windows"
    (tmp_path / "windows.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-unknown-pragmas", "-I", str(CSRC), str(tmp_path / "windows.cpp"),
                    "-o", str(exe)], check=True)
    text = "".join(" ".join(str(int(v)) for v in c) + "\n" for c in cases)
    out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout
    return [line.split() for line in out.splitlines()]


def test_windows_move_on_and_hold_every_task_once(tmp_path):
    rng = np.random.default_rng(1)
    cases = []
    for mn in (4, 8, 12, 16, 20, 48, 96):
        for _ in range(200):
            hi = int(rng.choice([2, 20, 100, 400]))
            c = np.cumsum(rng.integers(0, hi + 1, 5) * (rng.random(5) < 0.8))
            cases.append([0, *c, mn])
    for case, line in zip(cases, _run(tmp_path, cases)):
        words, ends = int(line[0]), line[1:]
        assert "stall" not in ends, (case, line)
        assert words >= max(64, 4 * case[6])
        ends = [int(e) for e in ends]
        base = np.array([0, *case[1:6]])
        assert (ends[-1] if ends else 0) == base[5]
        starts = [0, *ends[:-1]] if ends else []
        for s, e in zip(starts, ends):
            assert 0 < e - s <= words
        # a task is 64 consecutive terms of one type: no window ends inside one
        for k in range(5):
            for s in range(base[k], base[k + 1], 64):
                assert not any(s < e < min(s + 64, base[k + 1]) for e in ends), (case, ends)


def test_less_than_one_task_of_room_would_not_move_on(tmp_path):
    """Why the LDS has a minimum: twelve words per atom alone do not hold one task of
    a two-atom launch's 100 bonds, nor of a four-atom one's 100 torsions."""
    lines = _run(tmp_path, [[4 * 8, 100, 100, 100, 100, 100, 8], [4 * 12, 6, 18, 30, 42, 142, 12]])
    assert lines[0] == ["32", "stall"] and lines[1][-1] == "stall"
