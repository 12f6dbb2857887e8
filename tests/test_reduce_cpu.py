"""dr_reduce.hpp on the host: a NaN anywhere in a reduction by max_nan stays to
the end, as a sequence and as a tree."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include "dualres_amd/csrc/dr_reduce.hpp"
#include <cmath>
#include <cstdio>
#include <vector>
static double seq(const std::vector<double>& x) {
  double v = 0.0;
  for (double b : x) v = drh::max_nan(v, b);
  return v;
}
static double tree(std::vector<double> x) {
  for (size_t s = x.size() / 2; s > 0; s /= 2)
    for (size_t i = 0; i < s; ++i) x[i] = drh::max_nan(x[i], x[i + s]);
  return x[0];
}
int main() {
  const double inf = INFINITY, nan = NAN;
  std::vector<double> x = {1.0, 3.0, 2.0, 0.5, 7.0, 6.0, 7.0, 0.0};
  if (seq(x) != 7.0 || tree(x) != 7.0) return 1;
  for (size_t i = 0; i < x.size(); ++i) {
    std::vector<double> y = x;
    y[i] = nan;
    if (!std::isnan(seq(y)) || !std::isnan(tree(y))) return 2;
    y[i] = inf;
    if (seq(y) != inf || tree(y) != inf) return 3;
    y[(i + 3) % 8] = nan;
    if (!std::isnan(seq(y)) || !std::isnan(tree(y))) return 4;
  }
  std::puts("ok");
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_max_keeps_a_nan(tmp_path):
    src, exe = tmp_path / "t.cpp", tmp_path / "t"
    src.write_text(SRC)
    r = subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + ROOT, str(src),
                        "-o", str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.returncode
