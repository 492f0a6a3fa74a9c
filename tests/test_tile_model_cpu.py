"""The grouped contractions' cost model and its tuning (host code, compiled
here): shapes that take what the model says are left at the model's costs, and a
shape that takes longer is made dearer by that factor, whatever the operands'
orders and however the tiles are cut into units."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

PROGRAM = """
#include <cstdio>
#include "tile_model.h"
using namespace tenet;
int main() {
  // the tuned problem: 256 x 256 x 1024, column-major A and B
  std::vector<int64_t> rowA, kA, kB, colB;
  for (int i = 0; i < 256; ++i) rowA.push_back(i), colB.push_back(1024 * i);
  for (int k = 0; k < 1024; ++k) kA.push_back(256 * k), kB.push_back(k);
  for (int dtype = 0; dtype < 2; ++dtype) {
    const double a = gather_cycles(rowA, kA, false), b = gather_cycles(colB, kB, dtype == TENET_C64);
    double c[3], cycles[3], eff[3];
    tile_step_cycles(dtype, b, a, c);
    for (int v = 0; v < 3; ++v) cycles[v] = tile_cycles(c[v], 64 * (256 / TILE_EDGE[v]) * (256 / TILE_EDGE[v]), 64, 1 + v);
    const double ms[3] = {cycles[0] * 1e-6, cycles[1] * 1e-6, cycles[2] * 1.5e-6};
    tile_efficiency(ms, cycles, eff);
    std::printf("%d %g %g %.15g %.15g %.15g\\n", dtype, a, b, eff[0], eff[1], eff[2]);
  }
}
"""


def test_tuning_keeps_what_the_model_predicts(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "model.cpp", tmp_path / "model"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-I" + os.path.join(ROOT, "tenet.jl_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True, capture_output=True)
    lines = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.splitlines()
    rows = [list(map(float, x.split())) for x in lines]
    # rows of A adjacent; B read along K, 16 lines a load, two K steps each in complex64
    assert [r[:3] for r in rows] == [[0, 24, 48], [1, 24, 24]]
    for r in rows:
        assert r[3:] == pytest.approx([1.0, 1.0, 1.5], rel=1e-12)
