"""CPU walk of the launch plan of the small-tile FP8 product (fp8_mid.hpp): tokens and scale blocks covered,
no empty token tile, no split without a block, weight tiles that divide N."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferret_amd", "csrc")

CHECKER = r"""
#include <cstdio>
#include <initializer_list>
#include "fp8_mid.hpp"
using namespace ferret::mid;
#define BAD(what) do { std::printf("%s M=%d N=%d nkb=%d\n", what, M, N, nkb); return 1; } while (0)
int main() {
  long long plans = 0;
  for (int M = 1; M <= 300; ++M)
    for (int nkb = 1; nkb <= 128; ++nkb)
      for (int N : {128, 384, 1024, 4096, 7168, 24576}) {
        const Plan p = plan(M, N, nkb * 128, 256);
        if (p.ok != (M > 16 && M <= 256)) BAD("taken");
        if (!p.ok) continue;
        ++plans;
        const Tile& t = kTiles[p.tile];
        if (p.tok_tiles * t.tt * 16 < M || (p.tok_tiles - 1) * t.tt * 16 >= M) BAD("tokens");
        if (N % (16 * t.rt) != 0 || 128 % (16 * t.rt) != 0) BAD("rows");
        int at = 0;
        for (int s = 0; s < p.splits; ++s) {
          const int b = (int)((long long)s * nkb / p.splits), e = (int)((long long)(s + 1) * nkb / p.splits);
          if (b != at || e <= b) BAD("ranges");
          at = e;
        }
        if (at != nkb) BAD("cover");
      }
  for (int M : {1, 256, 257, 320, 511, 512, 513, 1000, 4096, 16384, 16385, 1000000})
    for (int nkb : {1, 3, 4, 19, 56, 128, 129})
      for (int N : {128, 384, 1024, 4096, 7168, 16384, 24576}) {
        const Plan p = unsplit_plan(M, N, nkb * 128, 256);
        const bool fits = M > 256 && nkb <= 128 && (long long)((M + 63) / 64) * (N / 64) <= 256;
        if (fits && !p.ok) BAD("not taken");
        if (!p.ok) continue;
        if (M <= 256 || nkb > 128 || p.splits != 1) BAD("taken");
        const Tile& t = kTiles[p.tile];
        if (p.tok_tiles * t.tt * 16 < M || (p.tok_tiles - 1) * t.tt * 16 >= M) BAD("tokens");
        if (p.tok_tiles * (N / (16 * t.rt)) > 256) BAD("rounds");
      }
  std::printf("plans %lld\n", plans);
  return 0;
}
"""


def test_plans_cover_tokens_and_blocks(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(CHECKER)
    subprocess.run([gxx, "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split()[1]) > 10000
