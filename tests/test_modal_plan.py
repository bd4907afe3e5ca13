"""Extents of the eigenvector solve (csrc/f2d_modal_plan.hpp, compiled for the
host): for every size, kind of direction and tile, the whole tiles of columns
and whole chunks of rows that a pass loads lie inside its matrix, and every
input index that it forms lies inside its row."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include "f2d_modal_plan.hpp"
using namespace f2d;

// one pass: K x LJ matrix, nj output pairs; returns 0 when in bounds
static int outside(int K, int LJ, int nk, int nj) {
  for (const ModalTile& t : MODAL_TILES) {
    if (K % t.kc || K < nk) return 1;
    for (int j0 = 0; j0 < nj; j0 += t.b)
      if (j0 + t.b > LJ) return 2;
  }
  return 0;
}

// mirror pairs (p, refl - p) of a row of npts points, as k_modal clamps them
static int unfolds(int nk, int refl, int npts) {
  for (int p = 0; p < nk; p++) {
    const int q = std::min(refl - p, npts - 1);
    if (p >= npts || q < 0) return 3;
  }
  return 0;
}

int main() {
  int used[3] = {0, 0, 0};
  for (int n = 8; n <= 4096; n++)
    for (int bc = 0; bc < 3; bc++) {
      const ModalSizes d = modal_sizes(bc, n);
      int e = outside(d.KF, d.LF, d.nh, d.ne);
      if (!e) e = outside(d.KB, d.LB, d.ne, d.nh);
      if (!e && bc != BC_EVEN) e = outside(d.KC, d.LF, d.cnh, d.ne);
      if (!e) e = unfolds(d.nh, d.refl, d.pts);
      if (!e) e = unfolds(d.cnh, d.crefl, d.cpts);
      if (!e && (d.no < 1 || d.ne + d.no != d.pts)) e = 4;
      if (e) {
        std::printf("n %d kind %d: %d\n", n, bc, e);
        return 1;
      }
      for (int m = 8; m <= 4096; m = m * 5 / 4 + 1) used[modal_tile(m, d.nh)]++;
    }
  std::printf("in bounds %d %d %d\n", used[0] > 0, used[1] > 0, used[2] > 0);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_passes_stay_inside_their_matrices(tmp_path):
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I",
                    os.path.join(ROOT, "fluids2d_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.split() == ["in", "bounds", "1", "1", "1"], r.stdout
