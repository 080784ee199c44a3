"""CPU checks of the bf16 linear's dispatch rules (ferret_amd/csrc/linear_plan.hpp), compiled with g++."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ferret_amd", "csrc")


def run_rules(tmp_path, body, header="linear_plan.hpp"):
    """Compile `body` (the statements of main) against a header of rules, run it and return its output."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "route.cpp", tmp_path / "route"
    src.write_text('#include <cstdio>\n#include <initializer_list>\n#include "' + header + '"\n'
                   "using namespace ferret;\n#define CHECK(c) do { if (!(c)) { std::printf(\"%s\\n\", #c); return 1; } } "
                   "while (0)\nint main() {\n" + body + "\n  return 0;\n}\n")
    subprocess.run([gxx, "-std=c++17", "-O2", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, res.stdout
    return res.stdout


def test_tiled_kernel_takes_aligned_tensors_only(tmp_path):
    run_rules(tmp_path, r"""
  alignas(64) static char buf[5][128];
  for (int which = 0; which < 5; ++which)  // x, w, residual, y, workspace
    for (int off = 0; off <= 32; off += 2) {
      char* p[5];
      for (int i = 0; i < 5; ++i) p[i] = buf[i] + (i == which ? off : 0);
      const int bound = which == 2 || which == 3 ? 8 : 16;
      CHECK(lin::tiled_aligned(p[0], p[1], p[2], p[3], p[4]) == (off % bound == 0));
    }
  CHECK(lin::tiled_aligned(buf[0], buf[1], nullptr, buf[3], nullptr));""")


def test_allocation_free_entry_shares_its_array_only_where_16_token_tiles_split(tmp_path):
    """Shapes that ran unsplit before the tiled kernel took them must not write to the library's one array."""
    run_rules(tmp_path, r"""
  const int shared[][3] = {{16, 6144, 4096}, {5, 4096, 12288}, {48, 4096, 12288}, {16, 1536, 4096}};
  for (auto& s : shared) CHECK(lin::noalloc_shares_array(s[0], s[1], s[2], 256));
  const int own[][3] = {{64, 4096, 4096}, {20, 4096, 4096}, {64, 6144, 4096}, {8, 1536, 9984}, {100, 2144, 1408}};
  for (auto& s : own) {
    const bt::Plan p = lin::tiled_plan(s[0], s[1], s[2], 256);
    CHECK(p.ok && p.splits > 1 && !lin::noalloc_shares_array(s[0], s[1], s[2], 256));
  }""")


def test_each_kernel_asks_for_its_own_partials(tmp_path):
    """A workspace of the 16-token split, or tensors off the tiled kernel's bounds, keep that split."""
    run_rules(tmp_path, r"""
  alignas(64) static char b[5][64];
  const auto route = [](const int* s, size_t bytes, int off = 0, bool ws = true) {
    return lin::route(s[0], s[1], s[2], 256, b[0] + off, b[1], b[2], b[3], ws ? b[4] : nullptr, bytes);
  };
  // M, N, K, splits of the tiled plan and of the 16-token kernels
  const int shapes[][5] = {{48, 4096, 12288, 4, 3}, {64, 1536, 12288, 8, 6}, {24, 6144, 4096, 4, 1}, {16, 4096, 12288, 0, 3}};
  for (auto& s : shapes) {
    const size_t one = (size_t)s[0] * s[1] * 4, tiled = one * s[3], units = s[4] > 1 ? one * s[4] : 0;
    if (s[3]) {
      CHECK(route(s, tiled).tiled.ok && route(s, tiled).tiled.splits == s[3]);
      CHECK(!route(s, tiled - 1).tiled.ok && route(s, tiled - 1).splits == s[4]);
      CHECK(!route(s, tiled, 8).tiled.ok && route(s, tiled, 8).splits == s[4]);
    }
    CHECK(!route(s, units).tiled.ok && route(s, units).splits == s[4]);
    if (units) CHECK(route(s, units - 1).splits == 1);
    CHECK(!route(s, 1 << 30, 0, false).tiled.ok && route(s, 1 << 30, 0, false).splits == 1);
  }
  const int unsplit[3] = {64, 24576, 4096};  // needs no workspace and looks at none
  CHECK(route(unsplit, 0, 0, false).tiled.ok && lin::route(64, 24576, 4096, 256, b[0], b[1], b[2], b[3], b[4] + 1, 8).tiled.ok);""")


def test_reported_workspace_serves_tensors_on_and_off_the_bounds(tmp_path):
    """Where the tiled plan splits less than the 16-token kernels, unaligned tensors find their split all the same."""
    run_rules(tmp_path, r"""
  alignas(64) static char b[5][64];
  // M, N, K, splits of the tiled plan and of the 16-token kernels
  const int shapes[][5] = {{512, 4096, 12288, 2, 3}, {2048, 8192, 6144, 1, 3}, {1036, 4432, 16384, 4, 8}, {48, 4096, 12288, 4, 3}};
  for (auto& s : shapes) {
    const int M = s[0], N = s[1], K = s[2];
    const size_t any = lin::workspace(M, N, K, 256), on = lin::aligned_workspace(M, N, K, 256);
    CHECK(lin::stream_splits(M, N, K, 256) == s[4] && on == lin::partial_bytes(s[3], M, N));
    CHECK(any == lin::partial_bytes(s[3] > s[4] ? s[3] : s[4], M, N));
    CHECK(lin::route(M, N, K, 256, b[0], b[1], b[2], b[3], b[4], on).tiled.splits == s[3]);
    CHECK(lin::route(M, N, K, 256, b[0] + 8, b[1], b[2], b[3], b[4], any).splits == s[4]);
  }""")


def test_oracle_shapes_reach_every_tile(tmp_path):
    """The shapes that the GPU tests hold to the oracle run every tile of the plan, unsplit and split."""
    from tests.test_gpu_bf16_tiled import EVERY_TILE
    shapes = ", ".join("{%d, %d, %d, %d, %d}" % s for s in EVERY_TILE)
    run_rules(tmp_path, "const int shapes[][5] = {" + shapes + r"""};
  bool seen[bt::kNumTiles][2] = {};
  for (auto& s : shapes) {
    const bt::Plan p = lin::tiled_plan(s[0], s[1], s[2], 256);
    CHECK(p.ok && p.tile == s[3] && p.splits == s[4]);
    CHECK(s[1] % (16 * bt::kTiles[p.tile].rt) != 0 && s[0] % 16 != 0);
    seen[p.tile][p.splits > 1] = true;
  }
  for (auto& t : seen) CHECK(t[0] && t[1]);""")


def test_few_tokens_split_a_short_k_only_from_a_larger_product_on(tmp_path):
    run_rules(tmp_path, r"""
  const int left[][3] = {{1, 6352, 1664}, {1, 4256, 2688}, {3, 7056, 1536}, {2, 3760, 2944}, {1, 3168, 3328},
    {4, 6464, 1664}, {7, 6288, 1792}};
  for (auto& s : left) CHECK(!lin::tiled_plan(s[0], s[1], s[2], 256).ok);
  const int taken[][3] = {{4, 6352, 2560}, {16, 4400, 2432}, {13, 6032, 1920}, {1, 1536, 9984}, {1, 9200, 1152}, {1, 8016, 1664}, {3, 5232, 2432}};
  for (auto& s : taken) CHECK(lin::tiled_plan(s[0], s[1], s[2], 256).ok);""")
