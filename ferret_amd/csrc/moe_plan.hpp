// Dispatch rules of the decode-sized MoE products (skinny.hip).  Plain C++17
// without HIP, so that CPU tests compile the rules themselves.
#pragma once

#include <cstdint>

namespace ferret {
namespace moe {

// K / 128 = nkb of the w2 (down) projection on the stream kernel: 4 waves of 2,
// 4, 7 or 8 K-steps.
inline bool w2_four_waves(int nkb) { return nkb == 8 || nkb == 16 || nkb == 28 || nkb == 32; }

// Whether the stream kernel takes the w2 projection.  K / 128 = 12 (3 K-steps
// per wave) and 4, 6 and 14 (two work-groups of 2 waves per CU) are the per-unit
// kernel's otherwise.  That one loads weights through registers, this one copies
// them to LDS 16 bytes at a time, so tensors off that bound stay there; and its
// units are 16 rows, not 64, so few tiles of few rows fill the CUs better.  The
// line is in units (64 rows of a tile of the table) per CU, per-unit kernel /
// this one (us) below and above it: K / 128 = 12, 1: 2 tiles of N = 2304 5.3 / 6.7,
// above 1.14 times as fast (geometric mean of 47 shapes); 6 and 14, 3: 4 of 896,
// K = 768 3.3 / 5.6, 8 of 640, K = 1792 5.0 / 6.9, above 1.14 and 1.19 times; 4, 8:
// 10 of 512 3.3 / 4.7, 51 of 1408 9.0 / 9.9, above 1.03 times.
inline bool w2_streams(int nkb, const void* w, long long units, int ncu) {
  if (w2_four_waves(nkb)) return true;
  const int least = nkb == 12 ? 1 : nkb == 6 || nkb == 14 ? 3 : nkb == 4 ? 8 : 0;
  return least != 0 && units >= (long long)least * ncu && (reinterpret_cast<uintptr_t>(w) & 15) == 0;
}

// Whether a unit takes two 16-row tiles of an expert (stream kernel, TB = 2), from
// the average of rows per expert and the units that one group per expert makes
// per CU.  Two tiles halve the weight bytes of an expert with 17 - 32 rows, but
// also the units: where those are few, CUs idle or a last round is nearly empty;
// and a unit of 2 K-steps per wave has no pipeline left to hide the second tile's
// activations (up to a fifth of its time with no second tile anywhere).  One tile -> two
// (us), even routing unless named:
//   w13, 7 K-steps per wave (K = 7168), 256 experts of N = 4096: 9.4 rows 1140 ->
//     1140, Zipf(1.1) 1413 -> 1238; 16 experts of 512 at 16 rows 17.6 -> 24.0, 64 of
//     512 at 9 rows 45.7 -> 52.6, 32 of 1280 at 15 rows 60.5 -> 52.1
//   w13, 2 (K = 2048): 256 experts of 512 at 7.4 rows 44.2 -> 49.9; 8 of 256 at 24
//     5.1 -> 7.4
//   w2, 4 (K = 2048), 256 experts of N = 7168: 15.6 rows 870 -> 652, 9.4 rows 634 ->
//     650; 128 of 768 at 10.5 35.7 -> 38.6
//   w2, 2 (K = 1024): 64 of 1536 at 12 rows 21.5 -> 25.6, 16 of 1024 at 23 8.4 ->
//     11.8
// The least rows below lose at most 4 % with an even routing, 14 % with a Zipf(1.1)
// one of few experts, and gain 35 % and 14 % in the mean (2000 shapes).
struct PairRule {
  int rows16, rows8, rows_few;  // least rows per expert from 16 units per CU, from 8, and from `few`
  int few;                      // units per CU below which no unit takes two tiles
};

inline bool pairs(const PairRule& r, long long num_pairs, int E, int units_n, int ncu) {
  const long long units = (long long)E * units_n;
  if (units < (long long)r.few * ncu) return false;
  return num_pairs >= (long long)(units >= 16LL * ncu ? r.rows16 : units >= 8LL * ncu ? r.rows8 : r.rows_few) * E;
}

inline bool w13_pairs(long long num_pairs, int E, int N, int nkb, int ncu) {
  const int ks = nkb / 8;  // K-steps per wave
  return pairs(ks <= 2 ? PairRule{12, 12, 12, 8} : ks <= 4 ? PairRule{10, 10, 14, 4} : PairRule{6, 8, 14, 4}, num_pairs,
               E, N / 32, ncu);
}

inline bool w2_pairs(long long num_pairs, int E, int N, int nkb, int ncu) {
  const int ks = w2_four_waves(nkb) || nkb == 12 ? nkb / 4 : nkb / 2;
  return pairs(ks <= 2 ? PairRule{14, 20, 20, 8} : ks <= 4 ? PairRule{12, 12, 14, 2} : PairRule{10, 12, 16, 2}, num_pairs,
               E, N / 64, ncu);
}

}  // namespace moe
}  // namespace ferret
