"""Offsets of the ghost images (csrc/rk_ghost.h) on lattices of 2^31 nodes and
more, where a step along x is past what an int holds: compiled for the host,
every signed overflow an error, and compared with 64-bit arithmetic modulo 2^32."""

import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHECK = r"""
#include "rk_ghost.h"
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
using namespace rk;
int main(int, char** v)
{
  const int H = GHOST_LAYERS, N[3] = {atoi(v[1]), atoi(v[2]), atoi(v[3])};
  const int L[3] = {N[0] + 2 * H, N[1] + 2 * H, N[2] + 2 * H};
  const int64_t row[3] = {int64_t(L[1]) * L[2], L[2], 1};
  auto step = [&](int c, int a) { return c < 2 * H ? int64_t(N[a]) : (c >= N[a] ? -int64_t(N[a]) : 0); };
  for(int i : {H, 2 * H - 1, 2 * H, N[0] - 1, N[0], N[0] + H - 1})
    for(int j : {H, 2 * H - 1, 2 * H, N[1] - 1, N[1], N[1] + H - 1})
      for(int k : {H, 2 * H - 1, 2 * H, N[2] - 1, N[2], N[2] + H - 1})
        for(int n = 0; n < 8; ++n) {
          const int64_t s[3] = {step(i, 0), step(j, 1), step(k, 2)};
          const uint32_t d0 = ghost_row(N, L, i, 0), d1 = ghost_row(N, L, j, 1), d2 = ghost_step(k, N[2]);
          int64_t off = 0;
          bool there = true;
          for(int a = 0; a < 3; ++a)
            if(n & (4 >> a)) {
              off += s[a] * row[a];
              there = there && s[a] != 0;
            }
          if(there != ghost_there(n, d0, d1, d2) || (there && ghost_image(n, d0, d1, d2) != uint32_t(uint64_t(off)))) {
            printf("node %d %d %d image %d\n", i, j, k, n);
            return 1;
          }
        }
  return 0;
}
"""


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    d = tmp_path_factory.mktemp("ghost")
    (d / "check.cpp").write_text(CHECK)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-fsanitize=signed-integer-overflow",
                    "-fno-sanitize-recover=all", "-I", os.path.join(ROOT, "runko_amd", "csrc"), "-o", str(d / "check"),
                    str(d / "check.cpp")], check=True)
    return str(d / "check")


@pytest.mark.parametrize("N", [(6, 6, 6), (7, 64, 9), (2042, 1018, 1018), (2024, 1024, 1024), (4090, 1018, 1018)])
def test_ghost_offsets(check, N):
    r = subprocess.run([check, *map(str, N)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
