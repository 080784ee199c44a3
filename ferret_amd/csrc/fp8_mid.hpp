// Launch plan and arguments of the mid-M FP8 product (fp8_mid.hip).  Plain
// C++17 without HIP, so that a CPU test walks it over shapes.
#pragma once

#include <cstddef>
#include <cstdint>

namespace ferret {
namespace mid {

struct Args {
  const uint8_t* a;   // e4m3 tokens [M, K]
  const float* sa;    // [M, K/128]
  const uint8_t* b;   // e4m3 weights [N, K]
  const float* sb;    // [N/128, K/128]
  uint16_t* out;      // bf16 [M, N]
  float* partial;     // splits > 1: fp32 [splits, M, N]
  int M, N, K;
  int splits, tok_tiles;
};

// The tiles the kernel is built for: rt x 16 weight rows by tt x 16 tokens, ns
// stages in LDS; `us` is what a stage of 256 K takes a CU (measured).
struct Tile {
  int rt, tt, ns;
  double us;
};
constexpr Tile kTiles[] = {{4, 2, 5, 0.78}, {2, 4, 3, 0.80}, {4, 4, 4, 1.05}, {2, 8, 2, 1.15}, {4, 8, 2, 1.50}};
constexpr int kNumTiles = sizeof(kTiles) / sizeof(kTiles[0]);

struct Plan {
  bool ok = false;
  int tile = 0;
  int splits = 1;
  int tok_tiles = 1;
};

// The tile and K split with the least estimated time: rounds of work-groups x
// stages, 3.3 us of launch, first stage and epilogue, and for a split the
// reduce launch (3.5) and the fp32 partials' way out and back (4 TB/s).
inline Plan plan(int M, int N, int K, int ncu) {
  Plan best;
  if (M <= 16 || M > 256 || N <= 0 || N % 128 != 0 || K <= 0 || K % 128 != 0 || ncu <= 0) return best;
  const int nkb = K / 128, blocks = (M + 15) / 16;
  double best_us = 0;
  for (int i = 0; i < kNumTiles; ++i) {
    const Tile& t = kTiles[i];
    const int tok_tiles = (blocks + t.tt - 1) / t.tt;
    if (tok_tiles > 1 && t.tt < 8) continue;
    const long long tiles = (long long)tok_tiles * (N / (16 * t.rt));
    for (int s = 1; s <= 8 && s <= nkb; s *= 2) {
      const int stages = ((nkb + s - 1) / s + 1) / 2;
      const long long rounds = (tiles * s + ncu - 1) / ncu;
      const double us = 3.3 + rounds * stages * t.us + (s > 1 ? 3.5 + (double)s * M * N * 8 / 4e6 : 0.0);
      if (!best.ok || us < best_us) {
        best_us = us;
        best.ok = true;
        best.tile = i;
        best.splits = s;
        best.tok_tiles = tok_tiles;
      }
    }
  }
  return best;
}

// Past 256 tokens, where K is not split: the tile with the least estimated time
// of those whose work-groups fit one round.  64 x 128 only from K = 512 on: its
// epilogue outlasts one or two stages (3072 x 128 at 583 tokens 5.2 us against
// 4.5 with 128 x 128 tiles; 4096 x 384 at 400 6.8 / 6.6, 4096 x 512 at 368 6.7 /
// 7.5).
inline Plan unsplit_plan(int M, int N, int K, int ncu) {
  Plan best;
  if (M <= 256 || N <= 0 || N % 128 != 0 || K <= 0 || K % 128 != 0 || K > 16384) return best;
  double best_us = 0;
  for (int i = 0; i < kNumTiles; ++i) {
    const Tile& t = kTiles[i];
    const long long tok_tiles = ((long long)M + 16 * t.tt - 1) / (16 * t.tt);
    if (tok_tiles * (N / (16 * t.rt)) > ncu || (K < 512 && t.rt * t.tt > 16)) continue;
    const double us = (K / 128 + 1) / 2 * t.us;
    if (best.ok && us >= best_us) continue;
    best_us = us;
    best.ok = true;
    best.tile = i;
    best.tok_tiles = (int)tok_tiles;
  }
  return best;
}

}  // namespace mid
}  // namespace ferret
