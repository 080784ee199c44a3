"""CPU walk of the launch plan of the LDS-tiled bf16 product (bf16_tiled.hpp).

Compiled with g++ and swept over shapes: the token and row tiles cover the
product with none empty, the K splits cover every stage once, the partials of
a run of 128 weight rows fit the 4 MiB array of the allocation-free entry, and
the estimate never picks a split for a product whose row tiles fill the CUs.
"""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferret_amd", "csrc")

CHECKER = r"""
#include <cstdio>
#include <initializer_list>
#include "bf16_tiled.hpp"
using namespace ferret::bt;
#define BAD(what) do { std::printf("%s M=%d N=%d K=%d ncu=%d\n", what, M, N, 128 * nkb, ncu); return 1; } while (0)
int main() {
  long long plans = 0;
  for (int M : {1, 16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 100, 128, 129, 200, 256, 257, 1000, 4096, 8192, 8193})
    for (int nkb = 1; nkb <= 128; ++nkb)
      for (int N : {16, 48, 64, 80, 96, 1024, 4096, 5008, 6144, 24576, 153600})
        for (int ncu : {80, 256}) {
          const Plan p = plan(M, N, nkb * 128, ncu);
          if (!p.ok) BAD("no plan");
          ++plans;
          const Tile& t = kTiles[p.tile];
          if ((long long)p.tok_tiles * t.tt * 16 < M || (long long)(p.tok_tiles - 1) * t.tt * 16 >= M) BAD("tokens");
          const int stages = nkb * 128 / t.ks;
          if (p.splits < 1 || p.splits > 8) BAD("splits");
          int at = 0;
          for (int s = 0; s < p.splits; ++s) {
            const int b = (int)((long long)s * stages / p.splits), e = (int)((long long)(s + 1) * stages / p.splits);
            if (b != at) BAD("ranges");
            at = e;
          }
          if (at != stages) BAD("cover");
          if (p.splits > 1 && (long long)p.splits * M * 128 * 4 > (4 << 20)) BAD("partials of 128 rows");
          const long long tiles = (long long)p.tok_tiles * ((N + 16 * t.rt - 1) / (16 * t.rt));
          if (p.splits > 1 && tiles >= 2 * ncu) BAD("split of a full grid");
        }
  std::printf("plans %lld\n", plans);
  return 0;
}
"""


def test_plans_cover_tokens_rows_and_k(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(CHECKER)
    subprocess.run([gxx, "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
    assert int(res.stdout.split()[1]) > 50000
