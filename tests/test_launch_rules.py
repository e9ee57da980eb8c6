"""Launch shapes chosen from a level's sizes (csrc/pmg_rules.h, compiled here
for the host): over cubes, flat and long grids up to 4 * 10^9 points every
choice fits what the solver allocates and what the kernels assume."""
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "pamr_amrd_amd" / "csrc"

HEAD = r"""
#include <cstdio>
#include "pmg_rules.h"
using namespace pmg;
// all shapes of the given sides with at most 4e9 points
template <typename F> void shapes(F f) {
  const int side[] = {3, 4, 5, 9, 17, 18, 31, 33, 34, 35, 49, 50, 65, 66, 97, 113, 129, 130, 161, 257, 258, 513, 1025, 1026,
                      2049, 4097, 8209, 16385, 131073, 666667, 2097153, 16777217};
  for (int x : side) for (int y : side) for (int z : side)
    if ((double)x * y * z <= 4e9) { const int n[3] = {x, y, z}; f(n); }
}
"""


def run(tmp_path, body):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(HEAD + "int main() { long bad = 0, all = 0;\n" + body + '\nprintf("%ld %ld\\n", all, bad); }\n')
    r = subprocess.run(["g++", "-O1", "-std=c++17", f"-I{CSRC}", str(src), "-o", str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    every, bad = map(int, subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()[-2:])
    assert every > 1000 and bad == 0, (every, bad)


def test_residual_fits_the_norm_workspace(tmp_path):
    """on the finest level and on any coarser one, which is no larger along any side"""
    run(tmp_path, r"""
  shapes([&](const int *n) {
    const int cap = norm_room(n);
    int c[3] = {n[0], n[1], n[2]};
    for (int l = 0; l < 12; l++) {
      const int z = residual_planes(c, cap);
      all++;
      if (z < 1 || z > RZC || residual_blocks(c, z) > cap || residual_blocks(c, z) < 1) bad++;
      for (int d = 0; d < 3; d++) c[d] = std::max(3, (c[d] - 1) / 2 + 1);
    }
  });""")


def test_resid_restrict_march(tmp_path):
    """one plane a block only where two make fewer than 500 blocks"""
    run(tmp_path, r"""
  shapes([&](const int *n) {
    if (n[0] % 2 == 0 || n[1] % 2 == 0 || n[2] % 2 == 0) return;
    const int c[3] = {(n[0] + 1) / 2, (n[1] + 1) / 2, (n[2] + 1) / 2};
    for (int pi = 0; pi < 2; pi++) {
      const int z = resid_restrict_planes(c, pi);
      all++;
      if (z < 1 || (z == 1) != (c[2] < 257 && rr_blocks(c, pi, 2) < 500)) bad++;
    }
  });""")


def test_default_sweeps_fit_the_norm_workspace(tmp_path):
    """both operators and types, on the finest level and the coarser ones"""
    run(tmp_path, r"""
  shapes([&](const int *n) {
    const int cap = norm_room(n);
    int c[3] = {n[0], n[1], n[2]};
    for (int l = 0; l < 12; l++) {
      for (int op = 0; op < 2; op++)
        for (int pi = 0; pi < 2; pi++) {
          int v, z;
          default_sweep(c, op, pi, &v, &z);
          all++;
          const long long tx = v == 2 ? 32 : v == 1 ? 64 : 128, ty = v == 11 ? 8 : 16;
          if ((v != 1 && v != 2 && v != 5 && v != 11) || z < 1 ||
              (c[0] - 2 + tx - 1) / tx * ((c[1] - 2 + ty - 1) / ty) * ((c[2] - 2 + z - 1) / z) > cap)
            bad++, bad == 1 ? printf("%d %d %d op %d type %d: variant %d z %d\n", c[0], c[1], c[2], op, pi, v, z) : 0;
        }
      for (int d = 0; d < 3; d++) c[d] = std::max(3, (c[d] - 1) / 2 + 1);
    }
  });""")
