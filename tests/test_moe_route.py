"""CPU checks of the decode MoE products' dispatch rules (ferret_amd/csrc/moe_plan.hpp), compiled with g++."""
from tests.test_linear_route import run_rules


def test_w2_stream_kernel_takes_aligned_weights_and_many_units_where_another_kernel_is_left(tmp_path):
    run_rules(tmp_path, r"""
  alignas(64) static char buf[64];
  for (int nkb = 1; nkb <= 128; ++nkb) {
    const bool four = nkb == 8 || nkb == 16 || nkb == 28 || nkb == 32, more = nkb == 12 || nkb == 4 || nkb == 6 || nkb == 14;
    const int least = nkb == 12 ? 256 : nkb == 4 ? 2048 : 768;  // units
    for (int off = 0; off <= 16; ++off)
      for (int units : {1, least - 1, least, 100000})
        CHECK(moe::w2_streams(nkb, buf + off, units, 256) == (four || (more && off % 16 == 0 && units >= least)));
  }""", "moe_plan.hpp")


def test_two_tiles_per_unit_only_where_the_units_fill_the_cus(tmp_path):
    """Few units, or hardly an expert with a second tile, keep one tile per unit."""
    run_rules(tmp_path, r"""
  // num_pairs, E, N, K / 128, taken
  const int w13[][5] = {{5600, 256, 4096, 56, 1}, {1612, 256, 4096, 56, 1}, {1500, 256, 4096, 56, 0}, {260, 16, 512, 56, 0},
    {600, 64, 512, 56, 0}, {480, 32, 1280, 56, 1}, {1904, 256, 512, 16, 0}, {194, 8, 256, 16, 0}, {416, 16, 256, 56, 0},
    {6000, 256, 512, 16, 1}, {404, 32, 1280, 16, 0}};
  for (auto& s : w13) CHECK(moe::w13_pairs(s[0], s[1], s[2], s[3], 256) == (s[4] != 0));
  const int w2[][5] = {{4000, 256, 7168, 16, 1}, {2406, 256, 7168, 16, 0}, {1348, 128, 768, 16, 0}, {764, 64, 1536, 8, 0},
    {362, 16, 1024, 8, 0}, {432, 16, 896, 28, 0}, {360, 32, 1152, 16, 0}, {6400, 256, 7168, 8, 1}, {4000, 256, 7168, 12, 1},
    {4000, 256, 7168, 6, 1}, {4000, 256, 7168, 14, 1}};
  for (auto& s : w2) CHECK(moe::w2_pairs(s[0], s[1], s[2], s[3], 256) == (s[4] != 0));""", "moe_plan.hpp")


def test_int4_checkpoint_layout_asks_for_whole_rounds_at_large_k(tmp_path):
    run_rules(tmp_path, r"""
  // num_pairs, E, N, K / 128, taken with the checkpoint layout (the tiled one takes them all)
  const int shapes[][5] = {{2128, 128, 1792, 56, 0}, {4096, 64, 1280, 56, 0}, {3456, 96, 2816, 56, 0}, {1984, 64, 2304, 56, 0},
    {7084, 128, 768, 32, 0}, {6400, 128, 4096, 56, 1}, {8192, 128, 1024, 56, 1}, {4096, 384, 4096, 56, 0},
    {2128, 128, 1792, 16, 1}};
  for (auto& s : shapes) {
    CHECK(i4::takes(s[0], s[1], s[2], s[3], 4096, 256, true, false) == (s[4] != 0));
    CHECK(s[0] < 14 * s[1] || i4::takes(s[0], s[1], s[2], s[3], 4096, 256, true, true));
  }""", "int4_moe.hpp")
