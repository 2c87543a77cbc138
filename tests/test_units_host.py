"""The constants of the odd-radix butterflies (csrc/sgpe_units.h, plain C++):
compiled with g++ and compared, bit for bit, with cos and sin of 2 pi m / R
taken in extended precision and rounded to double; symmetric entries are equal
and opposite. One unit in the last place would be wrong alike in every pass."""

import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), 'spinor-gpe_amd', 'csrc')

SRC = r'''
#include <cmath>
#include <cstdio>
#include "sgpe_units.h"
template <int R> int check() {
  const auto& u = sgpe::MixUnitTable<R>::u;
  int bad = 0;
  for (int m = 0; m < R; ++m) {
    const int h = 2 * m > R ? R - m : m;  // the same angle mirrored: symmetric by construction
    const long double a = 6.283185307179586476925286766559005768L * h / R;
    const double c = (double)cosl(a), s = (2 * m > R ? -1 : 1) * (double)sinl(a);
    if (u.c[m] != c || u.s[m] != s) {
      std::printf("R=%d m=%d: %.17g %.17g, want %.17g %.17g\n", R, m, u.c[m], u.s[m], c, s);
      ++bad;
    }
  }
  return bad;
}
int main() { return check<3>() + check<5>() + check<7>() + check<9>() + check<11>() + check<13>() ? 1 : 0; }
'''


@pytest.mark.skipif(shutil.which('g++') is None, reason='no g++')
def test_units_are_correctly_rounded(tmp_path):
    src = tmp_path / 'units.cpp'
    src.write_text(SRC)
    exe = tmp_path / 'units'
    subprocess.run(['g++', '-std=c++17', '-O1', f'-I{CSRC}', str(src), '-o', str(exe)], check=True, timeout=120)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
