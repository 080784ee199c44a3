"""CPU checks of the FP8 product's dispatch rules past 16 tokens (ferret_amd/csrc/fp8_plan.hpp), compiled with g++."""
from tests.test_linear_route import run_rules


def kernel(tmp_path, M, N, K, workspace=True):
    """The kernel and K splits of a call with all the workspace it can use, or with none: ("small", splits) for the
    small-tile kernel, ("128x128", splits) and ("256x128", 1) for the tiled one."""
    out = run_rules(tmp_path, f"const int M = {M}, N = {N}, K = {K}, mb = (M + 127) / 128, t256 = (N + 255) / 256 * mb;"
                              f"const f8::Route r = f8::route(M, N, K, false, {'f8::workspace(M, N, K)' if workspace else 0});"
                              r"""
  const bool half = r.splits > 1 || (2 * t256 <= f8::kRound && N / 128 * mb <= f8::kRound);
  std::printf("%s %d", r.mid.ok ? "small" : half ? "128x128" : "256x128", r.mid.ok ? r.mid.splits : r.splits);""",
                    "fp8_plan.hpp").split()
    return out[0], int(out[1])


def test_each_kernel_asks_for_its_own_partials(tmp_path):
    """A workspace of the 128 x 128 tiles' split keeps that split where the small tiles' is larger, with either
    matrix instruction, and the UE8M0 entry takes it."""
    run_rules(tmp_path, r"""
  // M, N, K, splits of the small tiles and of the 128 x 128 tiles
  const int shapes[][5] = {{17, 128, 1408, 8, 4}, {100, 512, 1664, 8, 4}, {200, 640, 1664, 4, 4}, {128, 4096, 512, 1, 2}};
  for (auto& s : shapes) {
    const int M = s[0], N = s[1], K = s[2];
    const size_t small = f8::partial_bytes(s[3], M, N), tiles = f8::partial_bytes(s[4], M, N);
    const size_t need = small > tiles ? small : tiles, sc = f8::ue8m0_scale_bytes(M, N, K);
    CHECK(f8::mid_plan(M, N, K).splits == s[3] && f8::tile_splits(M, N, K) == s[4] && f8::workspace(M, N, K) == need);
    CHECK(f8::route(M, N, K, false, need).mid.splits == s[3] && f8::route(M, N, K, false, need).mid.ok);
    CHECK(!f8::route(M, N, K, true, tiles).mid.ok && f8::route(M, N, K, true, tiles).splits == s[4]);
    CHECK(f8::route(M, N, K, true, tiles - 1).splits == 1);
    if (small > tiles) {
      CHECK(!f8::route(M, N, K, false, small - 1).mid.ok && f8::route(M, N, K, false, tiles).splits == s[4]);
      CHECK(f8::route(M, N, K, false, tiles - 1).splits == 1 && f8::route(M, N, K, false, 0).splits == 1);
    }
    CHECK(f8::ue8m0_workspace(M, N, K) == sc + need && f8::ue8m0_least_workspace(M, N, K) == sc + tiles);
  }
  for (int M : {17, 100, 256}) for (int N : {128, 4096, 24576}) for (int K : {128, 1536, 7168, 16384})
    CHECK(f8::ue8m0_least_workspace(M, N, K) <= f8::ue8m0_workspace(M, N, K));""", "fp8_plan.hpp")


def test_small_tiles_take_one_round(tmp_path):
    """Past one round of work-groups, or a single K block past 64 tokens, the larger tiles are the faster."""
    run_rules(tmp_path, r"""
  for (int M = 17; M <= 256; ++M)
    for (int N = 128; N <= 40960; N += 128)
      for (int nkb : {1, 2, 7, 8, 16, 24, 56, 96, 128}) {
        const mid::Plan p = f8::mid_plan(M, N, nkb * 128);
        if (!p.ok) continue;
        CHECK((long long)p.tok_tiles * (N / (16 * mid::kTiles[p.tile].rt)) * p.splits <= f8::kRound);
        CHECK(nkb > 1 || M <= 64);
      }
  const int taken[][3] = {{24, 4096, 7168}, {32, 7168, 2048}, {64, 14720, 128}, {100, 4096, 512}, {256, 4096, 2048}};
  for (auto& s : taken) CHECK(f8::mid_plan(s[0], s[1], s[2]).ok);
  const int left[][3] = {{23, 34944, 1024}, {24, 36608, 5376}, {20, 10624, 11904}, {172, 5248, 128}, {100, 4096, 7168}};
  for (auto& s : left) CHECK(!f8::mid_plan(s[0], s[1], s[2]).ok);""", "fp8_plan.hpp")


def test_oracle_shapes_reach_every_small_tile(tmp_path):
    """One shape per tile of the small-tile kernel, unsplit and split, of those the GPU tests hold to the oracle."""
    run_rules(tmp_path, r"""
  const int shapes[][4] = {{17, 128, 128, 0}, {24, 4096, 7168, 0}, {48, 1152, 128, 1}, {33, 256, 2432, 1}, {33, 8320, 128, 2},
    {33, 1152, 1664, 2}, {129, 1024, 256, 3}, {65, 128, 3072, 3}, {65, 8320, 256, 4}, {65, 1152, 1408, 4}};
  for (int i = 0; i < 2 * mid::kNumTiles; ++i) {
    const mid::Plan p = f8::mid_plan(shapes[i][0], shapes[i][1], shapes[i][2]);
    CHECK(p.ok && p.tile == i / 2 && shapes[i][3] == i / 2 && (p.splits > 1) == (i % 2 == 1));
  }""", "fp8_plan.hpp")
