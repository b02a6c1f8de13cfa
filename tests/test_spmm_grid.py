"""The launch of the observation operator on the members (oak_amd/csrc/spmm_grid.hpp),
compiled for the host with g++: every row and member is some workgroup's, once,
and no launch exceeds the device's limits (no GPU)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

DRIVER = r"""
#include <stdio.h>
#include <stdlib.h>
#include <vector>
#include "spmm_grid.hpp"
int main(int, char** a) {
  const int64_t m = atoll(a[1]);
  const int N = atoi(a[2]);
  const oakg::SpmmGrid g = oakg::spmm_grid(m, N);
  // blocks of 256 rows: workgroups that take them (x and z decide), by XCD
  std::vector<unsigned char> row((m + 255) / 256, 0);
  int64_t twice = 0, missed = 0, off = 0;
  for (unsigned z = 0; z < g.z; ++z)
    for (unsigned x = 0; x < g.x; ++x) {
      const int64_t r = oakg::spmm_row(x, z);
      off += r % 256 != 0 || r < 0;
      if (r < 0 || r >= m) continue;
      unsigned char& c = row[r / 256];
      twice += (c >> (x & 7)) & 1;
      c |= 1u << (x & 7);
    }
  for (unsigned char c : row) missed += c != 255;
  std::vector<int> mem(N, 0);
  for (unsigned y = 0; y < g.y; ++y)
    for (unsigned x = 0; x < 8; ++x)
      for (int q = 0; q < oakg::kSpmmMembers; ++q) {
        const int k = oakg::spmm_member(x, y) + 8 * q;
        if (k < N) ++mem[k];
      }
  for (int c : mem) missed += c != 1;
  printf("%u %u %u %lld %lld %lld\n", g.x, g.y, g.z, (long long)twice, (long long)missed, (long long)off);
}
"""


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    d = tmp_path_factory.mktemp("spmm")
    (d / "driver.cpp").write_text(DRIVER)
    subprocess.run(["g++", "-std=c++17", "-O2", "-I", os.path.join(ROOT, "oak_amd", "csrc"),
                    str(d / "driver.cpp"), "-o", str(d / "driver")], check=True)
    return str(d / "driver")


@pytest.mark.parametrize("m", [1, 255, 256, 257, 201_000, 67_200_000, 2 ** 28 - 1, 2 ** 28 + 1,
                               2 ** 29 + 300, 2 ** 31 - 1])
@pytest.mark.parametrize("N", [1, 8, 31, 33, 100, 256])
def test_every_row_and_member_once(driver, m, N):
    out = subprocess.run([driver, str(m), str(N)], check=True, capture_output=True, text=True).stdout
    x, y, z, twice, missed, off = map(int, out.split())
    assert (twice, missed, off) == (0, 0, 0)
    assert x * 256 < 2 ** 32 and y <= 65535 and z <= 65535 and x % 8 == 0
    assert z == 1 or m > 2 ** 28
