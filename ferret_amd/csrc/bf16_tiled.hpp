// Launch plan and arguments of the LDS-tiled bf16 product (bf16_tiled.hip).
// Plain C++17 without HIP, so that a CPU test walks it over shapes.
#pragma once

#include <cstddef>
#include <cstdint>

namespace ferret {
namespace bt {

struct Args {
  const uint8_t* w;          // bf16 [N, K]
  const uint8_t* x;          // bf16 [M, K]
  const uint16_t* residual;  // bf16 [M, ldo] or null
  uint16_t* out;             // bf16 [M, ldo]
  float* partial;            // splits > 1: fp32 [splits, M, N]
  int M, N, K, ldo;
  int splits;                // K splits
  int tok_tiles;             // token tiles
  int rt0;                   // row tiles before this launch's first (its place in the K rotation)
  bool nt;                   // stream the weights past the caches
  int rot_rows;              // serial form: rows of the plan's tiles (a place in the K rotation each)
};

// The tiles the kernel is built for: rt x 16 weight rows by tt x 16 tokens,
// ks of K per stage, ns stages in LDS.
struct Tile {
  int rt, tt, ks, ns;
};
constexpr Tile kTiles[] = {
    {4, 1, 128, 4}, {6, 1, 128, 5}, {4, 2, 128, 5}, {6, 2, 128, 5}, {4, 3, 128, 5}, {6, 3, 128, 4},
    {4, 4, 128, 4}, {6, 4, 128, 4}, {4, 6, 128, 4}, {6, 6, 128, 3}, {4, 8, 128, 3}, {8, 8, 64, 4}};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

struct Plan {
  bool ok = false;
  int tile = 0;
  int splits = 1;
  int tok_tiles = 1;
};

// Most tokens x splits of a plan, so that the partials of a run of 128 weight
// rows fit 4 MiB.
constexpr int kMaxTokenSplits = 8192;

// The tile and K split with the least estimated time.  A stage takes what its
// weights take at 25 B/ns per CU (6.4 TB/s from HBM over 256 CUs) or, where
// larger, what all its bytes take through a CU's loads (46 B/ns); a round of
// work-groups adds 1.5 us of pipeline fill and epilogue, a split the reduce launch
// and the fp32 partials' way out and back.
// Measured against the model: 4096 x 12288 at 64 tokens 24.2 / 25.3 us, 24576 x
// 4096 at 64 tokens 34.2 / 35.9 us, at 128 tokens 51.6 / 52.1 us.
inline Plan plan(int M, int N, int K, int ncu) {
  Plan best;
  if (M <= 0 || N <= 0 || K <= 0 || K % 128 != 0 || ncu <= 0) return best;
  const int blocks = (M + 15) / 16;
  double best_t = 0;
  for (int i = 0; i < kNumTiles; ++i) {
    const Tile& t = kTiles[i];
    const long long tok_tiles = (blocks + t.tt - 1) / t.tt;
    if (tok_tiles > 1 && t.tt < 6) continue;
    const long long tiles = tok_tiles * ((N + 16 * t.rt - 1) / (16 * t.rt));
    const double wb = t.rt * 32.0 * t.ks, xb = t.tt * 32.0 * t.ks;  // bytes of a stage
    const double stage_w = wb / 25e3, stage_all = (wb + xb) / 46e3;
    const double stage = stage_w > stage_all ? stage_w : stage_all;  // us
    for (int s = 1; s <= 8; ++s) {
      if (s > 1 && ((long long)s * M > kMaxTokenSplits || tiles >= 2LL * ncu)) break;
      const long long steps = (K / t.ks + s - 1) / s;
      const long long rounds = (tiles * s + ncu - 1) / ncu;
      const double us = rounds * (steps * stage + 1.5) + (s > 1 ? 3.0 + (double)s * M * N * 8 / 4e6 : 0.0);
      if (tiles * s < (1LL << 31) && (!best.ok || us < best_t)) {
        best_t = us;
        best.ok = true;
        best.tile = i;
        best.splits = s;
        best.tok_tiles = (int)tok_tiles;
      }
    }
  }
  return best;
}

}  // namespace bt
}  // namespace ferret
