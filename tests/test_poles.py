"""The table of poles behind M^-1/2 (oak_amd/csrc/poles.hpp), compiled for the host
with g++ and evaluated in quadruple precision: for every bound on the spectrum
that the kernels can find, the blocks that they choose give x^-1/2 on all of
[1, bound] to rounding, or no block is chosen (no GPU)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <stdio.h>
#include "poles.hpp"
typedef __float128 q;
static q qsqrt(q x) {
  q r = (q)sqrtl((long double)x);
  for (int i = 0; i < 3; ++i) r = (r + x / r) / 2;
  return r;
}
int main() {
  const std::vector<double>& t = oakg::pole_table();
  for (int ex = 0; ex <= 1025; ++ex) {
    const oakg::PoleBlocks b = oakg::pole_blocks(ex);
    q worst = 0, sum = 0;
    int zeros = 0;
    if (b.count && (size_t)(b.first + b.count) * oakg::kPoleBlock <= t.size()) {
      const double* p = &t[b.first * oakg::kPoleBlock];
      for (int g = 0; g <= 600; ++g) {
        const q x = (q)powl(2.0L, (long double)ex * g / 600);
        q f = 0;
        for (int c = 0; c < b.count; ++c)
          for (int j = 0; j < 32; ++j) f += (q)p[64 * c + 32 + j] / (x + (q)p[64 * c + j]);
        q e = f * qsqrt(x) - 1;
        if (e < 0) e = -e;
        if (e > worst) worst = e;
      }
      for (int c = 0; c < b.count; ++c)
        for (int j = 0; j < 32; ++j) {
          zeros += p[64 * c + j] == 0.0 && p[64 * c + 32 + j] == 0.0 && c == 0 && j == 31;
          if (p[64 * c + j] < 0 || p[64 * c + 32 + j] < 0) worst = 1;
          sum += p[64 * c + 32 + j];
        }
    }
    printf("%d %d %d %d %.3e\n", ex, b.first, b.count, zeros, (double)worst);
  }
  return 0;
}
"""


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    d = tmp_path_factory.mktemp("poles")
    src, exe = d / "poles.cpp", d / "poles"
    src.write_text(DRIVER)
    subprocess.check_call(["g++", "-O2", "-std=gnu++17", "-I", os.path.join(ROOT, "oak_amd", "csrc"),
                           str(src), "-o", str(exe)])
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    return [tuple(float(v) for v in l.split()) for l in out.splitlines()]


def test_every_bound_to_rounding(rows):
    # the approximation to 4.3e-16 (see the header), and the rounding of the poles
    # and weights to doubles, half an ulp each
    for ex, first, count, zeros, err in rows:
        if count:
            assert zeros == 1, ex
            assert err < 4.3e-16 + 2.3e-16, (ex, err)


def test_blocks_up_to_the_last_bound(rows):
    n = {int(ex): int(count) for ex, _, count, _, _ in rows}
    assert all(n[ex] == 1 for ex in range(0, 21))
    assert all(n[ex] == 2 for ex in range(21, 45))
    # beyond 2^44 the eigenvalues are taken (rounding may have left M indefinite)
    assert all(n[ex] == 0 for ex in range(45, 1026))
