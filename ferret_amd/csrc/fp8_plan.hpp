// Dispatch rules of the FP8 block-scaled product past 16 tokens
// (ferret_fp8_gemm_tiled in fp8_tiled.hip): which kernel takes a shape, its K
// split and its workspace.  Plain C++17 without HIP, so that CPU tests compile
// the rules themselves.
#pragma once

#include <cstddef>

#include "fp8_mid.hpp"

namespace ferret {
namespace f8 {

constexpr int kRound = 256;  // work-groups a split grid may not exceed (one per CU)

// Split-K plan of the 128 x 128 tiles for small M (8 waves over K ranges): the
// largest power of two whose grid still fits the 256 CUs in one round (one
// 97.5-KB work-group per CU): a grid of 448 at 128 x 7168 x 2048 ran in two
// rounds, 26.5 us against 15.7 us with 224.  At 128 x 4096 x 7168 (256
// work-groups) this beat 64 x 128 and 256 x 128 tiles and two work-groups per
// CU (28 us vs 29-36 us).  Returns the number of splits (1 = no split-K).
inline int tile_splits(int M, int N, int K) {
  if (M > 256 || N % 128 != 0) return 1;
  const int tiles = (N / 128) * ((M + 127) / 128);
  const int nkb = K / 128;
  int s = 1;
  while (tiles * s * 2 <= kRound && s * 2 <= nkb / 2) s *= 2;
  return s;
}

// The small-tile kernel's plan (fp8_mid.hip) for the shapes it takes, else none:
// one round of work-groups, and K and N where its larger share of token loads
// costs less than the 128 x 128 tiles' splits.  us against those tiles:
//   K <= 3072: 4096 x 2048 at 24 / 100 / 256 tokens 7.8 / 12.0 / 13.4 against 8.9 /
//     15.4 / 20.6; 7168 x 3072 at 256 22.8 against 23.4.  In two rounds it loses
//     (12288 x 1024 at 256: 19.0 against 12.9).
//   Larger K, up to 128 tokens while N K <= 22 M: 4096 x 5376 at 100 16.5 against
//     18.9; 7168 x 4096 at 100 20.5 against 19.5, 4096 x 7168 19.3 against 19.0.
//   Past 128 tokens while N K <= 11.5 M: 2048 x 5376 at 256 18.4 against 20.1; 2048
//     x 7168 21.3 against 19.6.
//   Up to 32 tokens any K: 4096 x 7168 at 24 12.3 against 12.7.  In more than one
//     round it loses there too (34944 x 1024 at 23 19.1 against 11.3, 36608 x 5376
//     at 24 54.4 against 37.5, 10624 x 11904 at 20 38.4 against 38.1).
//   Not a single K block past 64 tokens, where its epilogue is the longer: 5248 x
//     128 at 172 5.2 against 4.4, 2048 x 128 at 76 4.2 against 3.9.
// Past 256 tokens there is no split, and 128 x 128 tiles that leave CUs idle take
// 0.95 us for each 128 of K whatever their number: one round of smaller tiles is
// the shorter.  4096 x 7168 at 320 / 512 tokens 45.6 / 47.5 against 53.8 / 54.9;
// 2048 x 4096 at 512 / 1000 21.3 / 29.5 against 32.3 / 33.4; 1536 x 7168 at 320 24.8
// against 55.1; geometric mean 1.48 over 70 shapes.  In two rounds they lose (7168
// x 2048 at 320: 28.6 against 18.4).
inline mid::Plan mid_plan(int M, int N, int K) {
  if (M > 256) return mid::unsplit_plan(M, N, K, kRound);
  const mid::Plan p = mid::plan(M, N, K, kRound);
  const long long groups = p.ok ? (long long)p.tok_tiles * (N / (16 * mid::kTiles[p.tile].rt)) * p.splits : 0;
  const long long nk = (long long)N * K;
  const bool small = M <= 32 || K <= 3072 || nk <= 11500000 || (M <= 128 && nk <= 22100000);
  return p.ok && groups <= kRound && small && (K > 128 || M <= 64) ? p : mid::Plan{};
}

// fp32 partials of S splits.
inline size_t partial_bytes(int S, int M, int N) { return S > 1 ? (size_t)S * M * N * sizeof(float) : 0; }

// What a call runs: the small-tile kernel by `mid` where that is ok, else the 128
// x 128 tiles with K split by `splits` (1: the unsplit tiles).
struct Route {
  mid::Plan mid;
  int splits = 1;
};

// Each kernel asks for its own partials only: a workspace that holds the 128 x
// 128 tiles' split but not the small tiles' (128 x 1408 at 17 tokens: 4 against 8
// splits) still gets that split.  e4m3: the FP8 MFMA, which the small-tile
// kernel does not have.
inline Route route(int M, int N, int K, bool e4m3, size_t ws_bytes) {
  Route r;
  if (!e4m3) r.mid = mid_plan(M, N, K);
  if (partial_bytes(r.mid.splits, M, N) > ws_bytes) r.mid = mid::Plan{};
  if (!r.mid.ok) {
    const int s = tile_splits(M, N, K);
    if (partial_bytes(s, M, N) <= ws_bytes) r.splits = s;
  }
  return r;
}

// Workspace that any of the kernels can use: which one runs also depends on the
// flags.
inline size_t workspace(int M, int N, int K) {
  const int tiles = tile_splits(M, N, K), small = mid_plan(M, N, K).splits;
  return partial_bytes(tiles > small ? tiles : small, M, N);
}

// Workspace of the UE8M0 entry: the scales decoded to fp32 (tokens, then weight
// blocks, each padded to 256 bytes), then the product's own.  It takes any that
// holds the 128 x 128 tiles' split, as the product does.
inline size_t align_up(size_t v) { return (v + 255) / 256 * 256; }
inline size_t ue8m0_scale_bytes(int M, int N, int K) {
  const size_t nk = (size_t)K / 128, nbk = ((size_t)N + 127) / 128;
  return align_up((size_t)M * nk * 4) + align_up(nbk * nk * 4);
}
inline size_t ue8m0_workspace(int M, int N, int K) {
  return ue8m0_scale_bytes(M, N, K) + (M > 16 ? workspace(M, N, K) : 0);
}
inline size_t ue8m0_least_workspace(int M, int N, int K) {
  return ue8m0_scale_bytes(M, N, K) + (M > 16 ? partial_bytes(tile_splits(M, N, K), M, N) : 0);
}

}  // namespace f8
}  // namespace ferret
