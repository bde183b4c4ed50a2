"""Host-side checks of arithmetic that the kernels rest on, compiled from the
kernels' own sources with the system compiler.

The Schur chase divides and takes square roots by Newton iterations from the
hardware's seeds (csrc/schur_math.hpp), whose results have to be the correctly
rounded ones: here the seeds are the exact values off by up to 2^-23 (the
documented error is 2^29 units in the last place, 2^-24), over random operands
of the whole range that the kernel admits, quotients as near to the middle between
two doubles as there are, and roots near it.

The Gabor bound counts on the row and column factors (gabor_factors) being
within 4e-16 of each filter's taps, added over the taps."""
import os
import subprocess

import numpy as np
import pytest

from helpers import ROOT

CSRC = os.path.join(ROOT, 'wnd-charm_amd', 'csrc')

ROUNDING = r'''
#define __device__
#define __forceinline__ inline
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include "schur_math.hpp"
static uint64_t s[2] = {SEED, 0x9E3779B97F4A7C15ull};
static uint64_t next() {  // xorshift128+
  uint64_t a = s[0], b = s[1];
  s[0] = b;
  a ^= a << 23;
  s[1] = a ^ b ^ (a >> 17) ^ (b >> 26);
  return s[1] + b;
}
static double mantissa() { return 1.0 + (next() >> 12) * 0x1p-52; }
static double sign() { return next() & 1 ? -1.0 : 1.0; }
static double off() { return 1.0 + ((double)(int64_t)next() * 0x1p-63) * 0x1p-23; }
static int scale(int lo, int hi) { return lo + (int)(next() % (unsigned)(hi - lo + 1)); }
static uint64_t mulmod(uint64_t a, uint64_t b, uint64_t m) { return (unsigned __int128)a * b % m; }
// A with A / D as near to the middle between two doubles as it can be: A 2^53 =
// (D +- 1) / 2 modulo the odd D
static uint64_t hardest(uint64_t D, uint64_t plus) {
  uint64_t inv = 1, half = (D + 1) / 2;
  for (int k = 0; k < 53; k++) inv = mulmod(inv, half, D);
  return mulmod(plus ? (D + 1) / 2 : (D - 1) / 2, inv, D);
}
int main() {
  long bad = 0, hard = 0;
  for (int k = 0; k < 3000000; k++) {
    double d = sign() * ldexp(mantissa(), scale(-350, 341));
    double a = sign() * ldexp(mantissa(), scale(-350, 341));
    if (k % 8 == 1) {
      const uint64_t D = (1ull << 52) | (next() >> 12) | 1, A = hardest(D, k & 8 ? 1 : 0);
      if (2 * A >= D) {
        const int e = scale(-300, 250);
        d = ldexp((double)D, e);
        a = ldexp((double)A, e);
        hard++;
      }
    }
    const double y = wnd::recip(d, 1.0 / d * off());
    bad += wnd::quot(a, d, y) != a / d;
    double r = ldexp(mantissa(), scale(-700, 682));
    if (k & 1) {  // its root near a midpoint
      const long double g = (long double)mantissa() + 0x1p-53L;
      r = ldexp((double)(g * g), 2 * scale(-340, 340));
    }
    bad += wnd::root(r, 1.0 / sqrt(r) * off()) != sqrt(r);
  }
  printf("%ld %d\n", bad, hard > 100000);
}
'''

FACTORS = r'''
#include <cstdio>
#include <vector>
#include "tables.hpp"
int main() {
  const int n = 38;
  const std::vector<double> g = wnd::gabor_kernels(), f = wnd::gabor_factors();
  for (int k = 0; k < 8; k++) {
    const double *F = &f[k * 6 * n], *G = &g[(size_t)k * n * n * 2];
    long double err = 0, sum = 0;
    for (int y = 0; y < n; y++)
      for (int x = 0; x < n; x++)
        for (int c = 0; c < 2; c++) {
          const long double v = G[(y * n + x) * 2 + c];
          const long double w = (long double)F[(2 + c) * n + y] * F[x] + (long double)F[(4 + c) * n + y] * F[n + x];
          err += v > w ? v - w : w - v;
          sum += v > 0 ? v : -v;
        }
    printf("%.6Le\n", err / sum);
  }
}
'''


def run(tmp_path, source, *files):
    (tmp_path / 'check.cpp').write_text(source)
    exe = str(tmp_path / 'check')
    subprocess.run(['g++', '-O2', '-std=c++17', '-ffp-contract=off', '-I' + CSRC, '-o', exe, str(tmp_path / 'check.cpp')] +
                   [os.path.join(CSRC, f) for f in files], check=True)
    return subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()


@pytest.mark.parametrize('seed', [1, 2])
def test_schur_quotients_and_roots_are_correctly_rounded(tmp_path, seed):
    assert run(tmp_path, '#define SEED %dull\n' % (seed * 0x1234567) + ROUNDING) == ['0', '1']


def test_gabor_factors_are_the_taps(tmp_path):
    err = np.array([float(v) for v in run(tmp_path, FACTORS, 'tables.cpp')])
    assert err.shape == (8,) and (err < 4e-16).all(), err
