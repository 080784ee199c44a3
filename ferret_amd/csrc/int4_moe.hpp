// LDS layout and range of the two-tile INT4 w13 kernel (int4_moe.hip).  Plain
// C++17 with no HIP dependency.
#pragma once

#include <cstdint>

namespace ferret {
namespace i4 {

constexpr int kWaves = 4;
constexpr int BW = 2;                                // pairs of 16-row blocks (gate, up) per wave
constexpr int kItemRows = kWaves * BW * 32;          // weight rows of an item, half of them gate rows
constexpr int kNS = 3;                               // stages of 128 K
constexpr int kTB = 2;                               // 16-token tiles per item
constexpr int kScaleOff = 2 * BW * 1024;             // a wave's weights of a stage, then their scales
constexpr int kWaveBytes = kScaleOff + BW * 256;
constexpr int kXOff = kWaves * kWaveBytes;           // a stage's tokens: 32 rows of 256 B
constexpr int kStage = kXOff + kTB * 16 * 256;
constexpr int kXLoads = kTB * 16 * 256 / 1024 / kWaves;
constexpr int kOps = 2 * BW + BW + kXLoads;          // loads per wave and stage
constexpr int kMaxTiles = 4096;                      // rows of the tile table: 64 words of group-start bits
constexpr int kBitsOff = kNS * kStage;
constexpr int kBeforeOff = kBitsOff + kMaxTiles / 8;
constexpr int kCountOff = kBeforeOff + kMaxTiles / 64 * 4;
constexpr int kLds = kCountOff + 16;
static_assert(kLds <= 80 * 1024, "two work-groups share a CU's LDS");

// The rule, for num_pairs routed rows over E experts on ncu CUs (the results
// are the same bits either way).
//
// stream: the persistent stream kernel takes this K.  It is the faster of the
// two while most experts have one tile; the line lies where enough have two.
// Rows per expert and time, stream / this kernel (us), N = 1024, K = 7168, 384
// experts: tiled weights 13: 373 / 359, 14: 385 / 361, 16: 448 / 372 (48 experts
// of N = 4096: 188 / 188, 196 / 185, 222 / 187; N = 4096, K = 7168, 384 experts at
// 13: 1385 / 1434); checkpoint layout, whose half cache lines the shorter ring
// fetches later, 14: 428 / 464, 16: 495 / 481.
// From K = 4096 on the checkpoint layout gains less, and items that come out a
// little over a whole number of rounds (two work-groups per CU) cost more: at least
// 3 rounds if every expert had one group or by the 32-row groups there must be, and
// 20 rows per expert, or 2 and 40.  N = 1792, 128 experts at 17 rows 293 / 355, N =
// 1280, 64 experts at 64 rows 273 / 336, N = 2816, 96 experts at 36 rows 545 / 639;
// past the line 1.17 times as fast (82 shapes, none slower), below it 1.05 (94).
// Other K run on the per-unit kernel, a tile and 16 gate rows per work-group and
// nothing in flight at its ends: N = 2048, K = 5120, 64 experts 2 / 4 / 8 / 16 rows
// 108 / 120 / 134 / 199 against 82 / 83 / 84 / 91 us; N = 1024, K = 1024, 128
// experts 18.8 / 21.6 / 24.7 / 37.1 against 20.5 / 20.2 / 20.1 / 23.3.
// And the items have to fill the CUs: both work-groups of each if every expert
// had one, or three quarters of them by the 32-row groups there must be.  48
// experts of 512 rows are 96 items of one group (18 rows per expert: 48 / 71 us),
// 16 experts of 2048 rows 128 (31 / 43); by groups, 16 experts of 2048 rows, K =
// 4096 reach the line at 96 rows per expert (24 / 64 / 96 / 256 rows: 32 / 73 / 99 /
// 244 against 46 / 69 / 71 / 167), 48 experts of 512 at 128 (48 / 64 / 128 rows: 79 /
// 96 / 176 against 80 / 82 / 127).
inline bool takes(long long num_pairs, int E, int N, int nkb, int max_tiles, int ncu, bool stream, bool tiled) {
  const long long least_rows = stream ? (tiled ? 14 : 16) : 4, nb = N / kItemRows;
  if (stream && !tiled && nkb >= 32) {
    const long long items = (E > num_pairs / 32 ? E : num_pairs / 32) * nb;
    if (items < (num_pairs >= 40LL * E ? 4LL : 6LL) * ncu || num_pairs < 20LL * E) return false;
  }
  return N % kItemRows == 0 && max_tiles <= kMaxTiles && num_pairs >= least_rows * E &&
         (E * nb >= 2LL * ncu || num_pairs / 32 * nb >= ncu + ncu / 2);
}

}  // namespace i4
}  // namespace ferret
