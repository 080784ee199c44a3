// Dispatch rules of the bf16 linear (ferret_linear_bf16 in skinny.hip): which
// kernel takes a shape, its K split and its workspace.  Plain C++17 without HIP,
// so that CPU tests compile the rules themselves.
#pragma once

#include <cstddef>
#include <cstdint>

#include "bf16_tiled.hpp"
#include "stream_plan.hpp"

namespace ferret {
namespace lin {

// K splits of the bf16 stream kernel for y = x.W^T: 1 when a work-group per CU
// is already evenly loaded (>= 90 % of the 256 CUs' share), else the split with
// the best balance whose K-steps per wave (of 8) the kernel instantiates.
// Measured reason: 384 row units (QKV) leave half the CUs with one unit and
// half with two; K = 12288 (Down) needs 12 K-steps per wave, more activation
// registers than a wave has.
inline int stream_splits(int M, int N, int K, int ncu) {
  const int nkb = K / 128;
  const long long units = (long long)((M + 15) / 16) * (N / 16);
  auto ks_ok = [](int ks) { return ks == 2 || ks == 4 || ks == 7 || ks == 8; };
  auto balance = [&](int s) {
    const long long items = units * s;
    const long long per = (items + ncu - 1) / ncu;
    return (double)items / (double)(per * ncu);
  };
  if (nkb % 8 == 0 && ks_ok(nkb / 8) && balance(1) >= 0.9) return 1;
  int best = 1;
  double best_b = -1.0;
  for (int s = 2; s <= 8; ++s) {
    if (nkb % (8 * s) != 0 || !ks_ok(nkb / (8 * s))) continue;
    const double b = balance(s);
    if (b > best_b + 1e-9) { best = s; best_b = b; }
  }
  return best;
}

// The LDS-tiled kernel's plan for the shapes it takes, else none.
//   * Past 16 tokens: it streams the weights once for all of them, the stream
//     and per-unit kernels once per 16 (4096 x 12288 at 17 tokens 20.5 against
//     36.2 us, 24576 x 4096 at 32 32.7 against 45.5, 6144 x 4096 at 32 14.1
//     against 14.7).
//   * Up to 16 tokens where the stream kernel does not take K (K / 128 not 2, 4,
//     7 or 8 per wave; 1536 x 9984: 11.2 against the per-unit kernel's 17.4 us
//     at one token, 12.1 against 23.4 at 16; 16000 x 1280 9.0 against 10.9 and
//     9.2 against 14.7).
//   * Not where the whole product is a few microseconds: a split's second launch
//     and the ring's fill cost 2-3 us more than the other kernels spend.  In
//     16-token tiles x N x K the line lies at 2^25 against the stream kernel (4
//     tiles of 2048 x 2048, 2^24: 9.7 against 7.0 us; 2 of 4096 x 4096, 2^25:
//     10.4 against 13.9) and at 10 * 2^20 against the per-unit one (2 tiles of
//     4096 x 640: 5.8 against 5.3; 4: 6.7 against 7.7).  Up to 3 tokens a
//     split of a K below 3584 asks for 12 * 2^20: 6352 x 1664 at one token 10.2
//     against 7.3, 4256 x 2688 11.0 against 9.5; and up to 16 the 128-token tile is
//     not split below K = 2048 (6464 x 1664 at 4 10.3 against 7.7).
inline bt::Plan tiled_plan(int M, int N, int K, int ncu) {
  const bool stream = stream_plan(false, 1, 8, N, K, 1, false, stream_splits(M, N, K, ncu), ncu).ok ||
                      (N / 16 >= 4 * ncu && stream_plan(false, 1, 4, N, K, 1, false, 1, ncu).ok);
  const long long work = (long long)((M + 15) / 16) * N * K;
  if ((stream && M <= 16) || work < (stream ? 32LL : 10LL) << 20) return bt::Plan{};
  const bt::Plan p = bt::plan(M, N, K, ncu);
  const bool few = (M <= 3 && K < 3584 && work < 12LL << 20) || (M <= 16 && K < 2048 && bt::kTiles[p.tile].tt == 8);
  return p.splits > 1 && few ? bt::Plan{} : p;
}

// The tiled kernel copies x and the weights global -> LDS 16 bytes at a time,
// reads the residual and stores y 8 bytes at a time, and keeps its partials in
// 16-byte pieces.  Tensors off these bounds (a view that starts inside a buffer)
// keep the kernels of 16 tokens, which load x through registers and store single
// elements.
inline bool tiled_aligned(const void* x, const void* w, const void* residual, const void* y, const void* ws) {
  const auto bits = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
  return ((bits(x) | bits(w) | bits(ws)) & 15) == 0 && ((bits(residual) | bits(y)) & 7) == 0;
}

// fp32 partials of S splits.
inline size_t partial_bytes(int S, int M, int N) { return S > 1 ? (size_t)S * M * N * sizeof(float) : 0; }

// Workspace for tensors on the tiled kernel's bounds, and for any: where its plan
// splits K less than the 16-token kernels (4432 x 16384 at 1036 tokens: 4 against 8),
// those need the larger one for their split (unaligned x, 1647 us; 2513 without).
inline size_t aligned_workspace(int M, int N, int K, int ncu) {
  const bt::Plan tiled = tiled_plan(M, N, K, ncu);
  return partial_bytes(tiled.ok ? tiled.splits : stream_splits(M, N, K, ncu), M, N);
}
inline size_t workspace(int M, int N, int K, int ncu) {
  const size_t tiled = aligned_workspace(M, N, K, ncu), units = partial_bytes(stream_splits(M, N, K, ncu), M, N);
  return tiled > units ? tiled : units;
}

// What a call runs: the LDS-tiled kernel by `tiled` where that is ok, else the
// 16-token kernels with K split by `splits`.
struct Route {
  bt::Plan tiled;
  int splits = 1;
};

// Each kernel asks for its own partials only: a workspace that a caller sized for
// the 16-token split (4096 x 12288 at 48 tokens: 3 splits, the tiled plan has 4)
// still holds that split, and tensors off the tiled kernel's bounds still take it.
inline Route route(int M, int N, int K, int ncu, const void* x, const void* w, const void* residual, const void* y,
                   const void* ws, size_t ws_bytes) {
  if (ws == nullptr) ws_bytes = 0;
  Route r;
  r.tiled = tiled_plan(M, N, K, ncu);
  const size_t need = partial_bytes(r.tiled.splits, M, N);
  if (need > ws_bytes || !tiled_aligned(x, w, residual, y, need == 0 ? nullptr : ws)) r.tiled.ok = false;
  if (!r.tiled.ok) {
    const int s = stream_splits(M, N, K, ncu);
    if (partial_bytes(s, M, N) <= ws_bytes) r.splits = s;
  }
  return r;
}

// Whether the allocation-free entry takes its partials from the library's one
// array, so that calls which overlap race: only where the 16-token kernels split
// K.  Any other call may overlap with all of them, and be captured into a graph
// before the array's address is known.
inline bool noalloc_shares_array(int M, int N, int K, int ncu) { return stream_splits(M, N, K, ncu) > 1; }

}  // namespace lin
}  // namespace ferret
