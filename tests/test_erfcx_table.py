"""The erfcx table and evaluation of the Ewald direct sum
(gse_amd/csrc/erfcx_table.h), compiled for the host and compared with
erfc(x) exp(x^2) in extended precision: every interval at its ends, its
middle and between, the step from intervals of 1/4 to intervals of 1 at 8, and
the last one up to 27; from there on, and for a NaN, the value is finite."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "gse_amd", "csrc")

CHECK = r"""
#include <cstdio>
#include "erfcx_table.h"
int main() {
  const std::vector<double> t = gse::make_erfcx_table();
  double worst = 0, at = 0;
  auto test = [&](double x) {
    if (!(x >= 0.0 && x < 27.0)) return;
    const long double ref = erfcl((long double)x) * expl((long double)x * x);
    const double e = (double)fabsl((gse::ew_erfcx(t.data(), x) - ref) / ref);
    if (!(e <= worst)) { worst = e; at = x; }
  };
  for (int i = 0; i <= 27 * 4; i++) {
    const double c = 0.25 * i;
    test(c); test(std::nextafter(c, 0.0)); test(std::nextafter(c, 100.0));
  }
  for (int i = 0; i < 270000; i++) test(i * 1e-4 + 3.3e-5);
  std::printf("worst %.3e at %.6f\n", worst, at);
  for (double x : {27.0, 27.5, 30.0, 1e3, 1e300, (double)INFINITY, (double)NAN})
    if (!(gse::ew_erfcx(t.data(), x) > 0.0 && gse::ew_erfcx(t.data(), x) < 0.03)) return 2;
  return worst <= 3.3e-16 ? 0 : 1;
}
"""


def test_erfcx_table_against_long_double(tmp_path):
    """Half a unit in the last place (2.2e-16 of the value at most) from the
    last multiply-add, half from the constant coefficient, and half for the
    other terms, which the interval's half width scales down."""
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    src, exe = tmp_path / "c.cpp", tmp_path / "c"
    src.write_text(CHECK)
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout
