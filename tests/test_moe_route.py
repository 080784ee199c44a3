"""CPU checks of the decode MoE products' dispatch rules (ferret_amd/csrc/moe_plan.hpp), compiled with g++."""
from tests.test_linear_route import run_rules


def test_w2_stream_kernel_takes_aligned_weights_only_where_another_kernel_is_left(tmp_path):
    run_rules(tmp_path, r"""
  alignas(64) static char buf[64];
  for (int nkb = 1; nkb <= 128; ++nkb) {
    const bool four = nkb == 8 || nkb == 16 || nkb == 28 || nkb == 32, more = nkb == 12 || nkb == 4 || nkb == 6 || nkb == 14;
    for (int off = 0; off <= 16; ++off) CHECK(moe::w2_streams(nkb, buf + off) == (four || (more && off % 16 == 0)));
  }""", "moe_plan.hpp")
