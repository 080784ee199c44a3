// Skinny (<= 16 token) weight-streaming GEMMs for gfx950: bf16 decode linear,
// small-M FP8 block-scaled GEMM, and the decode-sized MoE grouped GEMMs (FP8
// w13 and w2, INT4 W4A16 w13) with the fused SiLU(gate)*up epilogue.  Shapes
// whose K-steps split evenly into 2, 4, 7 or 8 per wave (w2 also 3) run the persistent
// LDS-staged stream kernel of stream_kernel.hpp (bf16 with K split over a
// workspace where the row units alone would leave CUs idle); the per-unit
// kernel below takes the rest.
//
// Design (swap-AB): the weight rows are the MFMA "A" side (16 rows per MFMA)
// and the <= 16 tokens of a unit are the MFMA "B" side, so a 16x16 MFMA tile
// wastes nothing at 16 tokens.  A work-group owns one unit = (token tile,
// RB blocks of 16 weight rows) and splits K across its waves: wave w streams
// K-steps [w*KS, (w+1)*KS) (one K-step = 128 K = one fp32 scale block), with a
// D-deep register prefetch of the weight and activation fragments.  Each lane
// reads 16-byte vectors; per load instruction a wave covers 16 rows x 64
// contiguous bytes.  The per-wave fp32 partials are summed through LDS and the
// epilogue (bf16 store, + residual, or SiLU(gate)*up) runs once per output.
//
// Reference counterparts: swapab_cg1_kernel / swapab_persistent_kernel
// (examples/qwen3-8b-decode-linear-bs16/v006_cg1_swapab_l2hints.cu:138-375,
// v019_swapab_cg2_l2hints.cu:138-391) and the split-K reduce (v019:395-417);
// grouped_fp8_gemm_bs (examples/fp8-group-gemm/v007_dsv3_decode_verified_105.cu:66-335);
// the INT4 w13 contract (tasks/kimi-moe-w13-int4-grouped-gemm.yaml:68-95,150-167).
#include "skinny_kernel.hpp"
#include "stream_kernel.hpp"
#include "linear_plan.hpp"
#include "int4_moe.hpp"
#include "moe_plan.hpp"

int ferret_bf16_tiled(int tile, const ferret::bt::Args& p, hipStream_t st);
int ferret_bf16_tiled_serial(int tile, ferret::bt::Args p, hipStream_t st);
int ferret_int4_moe(const ferret::SkinnyArgs& a, bool tiled, int span, int max_tiles, int ncu, hipStream_t st);

namespace ferret {

// Compute units of the current device (the persistent grid size), cached per
// device; concurrent first calls store the same value.
static int cu_count() {
  static std::atomic<int> cached[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) dev = 0;
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Stream-kernel launch (persistent grid, one work-group of NW waves per CU):
// returns 1 if the shape is not covered (the caller then uses the per-unit
// kernel), else the launch status.  KS = K-steps per wave = K / 128 / NW.
// `per_cu` work-groups share a CU (fewer waves each).
template <int F, int EPI, int RB, int D, int NW>
static int plan_and_launch(const SkinnyArgs& a_in, int dense_tiles, int max_tiles, hipStream_t st, int per_cu) {
  // The unit count, K-steps per wave and tile-table span come from the
  // host-only plan (stream_plan.hpp), which the CPU tests check over every
  // configuration instantiated here: a unit is RB 16-row blocks (SiLU: one
  // gate and one up block), counted from RB itself, not from the caller
  // (whose units_n sizes the per-unit fallback kernel).
  static_assert(EPI != kSilu || RB == 2, "SiLU units pair one gate and one up block");
  const bool grouped = a_in.tiles != nullptr;
  // bf16 dense split-K: each work item covers K / nsplit (see stream_gemm_kernel)
  const int nsplit = (F == kBF16 && !grouped && a_in.partial != nullptr) ? a_in.ksplit : 1;
  const int grid = cu_count() * per_cu;
  const StreamPlan plan = stream_plan(EPI == kSilu, RB, NW, a_in.N, a_in.K, grouped ? max_tiles : dense_tiles,
                                      grouped, nsplit, grid);
  if (!plan.ok) return 1;
  // INT4 unit scales are copied as 16-byte chunks of the scale rows.
  if (is_int4(F) && ((reinterpret_cast<uintptr_t>(a_in.w_scale) & 15) != 0 || a_in.K % 256 != 0)) return 1;
  SkinnyArgs a = a_in;
  a.units_n = plan.units_n;
  const int slots = grouped ? max_tiles : dense_tiles;
  // INT4 keeps at most one unit of scales ahead: ring depth <= KS.
  constexpr int D2 = (is_int4(F) && D > 2) ? 2 : D;
  constexpr int D4 = (is_int4(F) && D > 4) ? 4 : D;
  if constexpr (F == kFP8 && (EPI == kSilu || RB == 4)) {
    // The FP8 MoE products with several tiles per expert: two tiles per unit.
    if (a.pair_tiles && max_tiles <= kStreamPairTiles) {
      switch (plan.ks) {
        case 2: return launch_stream<F, EPI, RB, NW, 2, D, 2>(a, slots, grid, st);
        case 3: if constexpr (RB == 4) return launch_stream<F, EPI, RB, NW, 3, D, 2>(a, slots, grid, st); else break;
        case 4: if constexpr (NW != 2) return launch_stream<F, EPI, RB, NW, 4, D, 2>(a, slots, grid, st); else break;
        case 7: return launch_stream<F, EPI, RB, NW, 7, D, 2>(a, slots, grid, st);
      }
    }
  }
  switch (plan.ks) {
    case 2: return launch_stream<F, EPI, RB, NW, 2, D2>(a, slots, grid, st);
    case 3: if constexpr (RB == 4) return launch_stream<F, EPI, RB, NW, 3, D>(a, slots, grid, st); else return 1;
    case 4: if constexpr (NW != 2) return launch_stream<F, EPI, RB, NW, 4, D4>(a, slots, grid, st); else return 1;
    // More than 8 waves leave a wave 128 VGPRs (two work-groups' worth of waves
    // on some SIMDs), too few for 7 or 8 K-steps of activations: those shapes
    // take the 8-wave configuration (the caller's fallback).
    case 7: if constexpr (NW <= 8) return launch_stream<F, EPI, RB, NW, 7, D>(a, slots, grid, st); else return 1;
    case 8: if constexpr (NW <= 8 && NW != 2) return launch_stream<F, EPI, RB, NW, 8, D>(a, slots, grid, st); else return 1;
  }
  return 1;
}

template <int F, int EPI, int RB, int D, int NW = 8>
static int try_stream(const SkinnyArgs& a, int dense_tiles, int max_tiles, hipStream_t st) {
  return plan_and_launch<F, EPI, RB, D, NW>(a, dense_tiles, max_tiles, st, 1);
}

// Grouped: two work-groups of 2 waves per CU, each in at most half of its LDS,
// for the K / 128 that 4 waves leave (4, 6 and 14: 2, 3 and 7 K-steps per wave).
template <int F, int EPI, int RB, int D>
static int try_half_stream(const SkinnyArgs& a, int max_tiles, hipStream_t st) {
  static_assert(StreamCfg<F, RB, 2, 7, D, 2>::kLds <= 80 * 1024, "two work-groups share a CU's LDS");
  return plan_and_launch<F, EPI, RB, D, 2>(a, 0, max_tiles, st, 2);
}

// K-steps per wave: prefer a split giving 4..16 waves (balanced reduction
// against per-wave stream depth), else any split with <= 16 waves.
static int choose_ks(int nkb, const int* cand, int ncand) {
  for (int i = 0; i < ncand; ++i) {
    const int ks = cand[i];
    if (nkb % ks == 0 && nkb / ks >= 4 && nkb / ks <= 16) return ks;
  }
  for (int i = 0; i < ncand; ++i) {
    const int ks = cand[i];
    if (nkb % ks == 0 && nkb / ks <= 16) return ks;
  }
  return 0;
}

// K-steps per wave of the per-unit kernel, 0 past its range (K/128 > 128).
static int unit_steps(int nkb) {
  static const int cand[] = {4, 7, 8, 2, 1};
  const int ks = choose_ks(nkb, cand, 5);
  if (ks != 0) return ks;
  // No K-step count divides K/128 into <= 16 waves (K/128 = 19, 23, 38, ...):
  // the smallest of 2, 4, 7, 8 that fits 16 waves, the last wave ragged.
  for (const int kr : {2, 4, 7, 8})
    if ((nkb + kr - 1) / kr <= 16) return kr;
  return 0;
}

template <int F, int EPI, int RB>
static int launch_skinny(const SkinnyArgs& a, int ntile_slots, hipStream_t st) {
  const int nkb = a.K >> 7;
  const int ks = unit_steps(nkb);
  const int grid = ntile_slots * a.units_n;
  if (grid <= 0) return FERRET_OK;
  // Prefetch depth kept so a wave stays within 128 VGPRs (16 waves / CU).
  constexpr int DB = (F == kBF16) ? 2 : ((F == kFP8 && RB == 1) ? 4 : (F == kFP8 ? 3 : 2));
  // 7 or 8 K-steps per wave hold more activations: FP8 row pairs (SiLU) keep a
  // 2-deep prefetch and the ragged single-block form a 3-deep one, or they
  // spill past 128 VGPRs.
  constexpr int D78 = (F == kFP8 && RB >= 2) ? 2 : DB;
  constexpr int D78R = (F == kFP8 && RB == 1) ? 3 : D78;
  if (ks == 0) return FERRET_ERR_SHAPE;
  if (nkb % ks != 0) {
    const int nw = (nkb + ks - 1) / ks;
    switch (ks) {
      case 2: return launch_one<F, EPI, RB, 2, 1, true>(a, grid, nw, st);
      case 4: return launch_one<F, EPI, RB, 4, (DB < 3 ? DB : 3), true>(a, grid, nw, st);
      case 7: return launch_one<F, EPI, RB, 7, D78R, true>(a, grid, nw, st);
      case 8: return launch_one<F, EPI, RB, 8, D78R, true>(a, grid, nw, st);
    }
  }
  const int nwaves = nkb / ks;
  switch (ks) {
    case 1: return launch_one<F, EPI, RB, 1, 0>(a, grid, nwaves, st);
    case 2: return launch_one<F, EPI, RB, 2, 1>(a, grid, nwaves, st);
    case 4: return launch_one<F, EPI, RB, 4, (DB < 3 ? DB : 3)>(a, grid, nwaves, st);
    case 7: return launch_one<F, EPI, RB, 7, D78>(a, grid, nwaves, st);
    case 8: return launch_one<F, EPI, RB, 8, D78>(a, grid, nwaves, st);
  }
  return FERRET_ERR_SHAPE;
}

// y[m, n] = bf16(sum_{s < S} partial[s, m, n] (+ residual[m, n])) for the N
// outputs of row m = blockIdx.y (row strides: partial N, y and residual ldo),
// splits in order; SN > 0: S == SN, all split loads issued before the first add.
template <int SN>
__global__ __launch_bounds__(256) void linear_splitk_reduce_kernel(const float* __restrict__ partial, int S, int N,
                                                                   int ldo, const uint16_t* __restrict__ res,
                                                                   uint16_t* __restrict__ y) {
  const int n4 = N / 4;
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  f32x4 v = sum_splits<SN>(reinterpret_cast<const f32x4*>(partial), S, (size_t)gridDim.y * n4,
                           (size_t)blockIdx.y * n4 + i);
  const size_t o = (size_t)blockIdx.y * ldo + (size_t)i * 4;
  if (res) {
    const u32x2 r = *reinterpret_cast<const u32x2*>(res + o);
    v[0] += __uint_as_float(r[0] << 16);
    v[1] += __uint_as_float(r[0] & 0xffff0000u);
    v[2] += __uint_as_float(r[1] << 16);
    v[3] += __uint_as_float(r[1] & 0xffff0000u);
  }
  *reinterpret_cast<u32x2*>(y + o) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

static int launch_splitk_reduce(const float* partial, int S, int M, int N, int ldo, const uint16_t* residual,
                                uint16_t* out, hipStream_t st) {
  auto* reduce = S == 2 ? linear_splitk_reduce_kernel<2> : S == 3 ? linear_splitk_reduce_kernel<3>
               : S == 4 ? linear_splitk_reduce_kernel<4> : linear_splitk_reduce_kernel<0>;
  hipLaunchKernelGGL(reduce, dim3((N / 4 + 255) / 256, M), dim3(256), 0, st, partial, S, N, ldo, residual, out);
  return (int)hipGetLastError();
}

// Arguments of the LDS-tiled product over weight rows [n0, n0 + n) by `plan`.
static bt::Args bf16_tiled_args(const bt::Plan& plan, const SkinnyArgs& a, int n0, int n) {
  bt::Args p{};
  p.w = a.w + (size_t)n0 * a.K * 2;
  p.x = a.x;
  p.residual = a.residual ? a.residual + n0 : nullptr;
  p.out = a.out + n0;
  p.M = a.M;
  p.N = n;
  p.K = a.K;
  p.ldo = a.N;
  p.splits = plan.splits;
  p.tok_tiles = plan.tok_tiles;
  return p;
}

// The LDS-tiled product over weight rows [n0, n0 + n) by `plan`, partials in ws.
static int launch_bf16_tiled(const bt::Plan& plan, const SkinnyArgs& a, int n0, int n, void* ws, hipStream_t st) {
  const bt::Tile& t = bt::kTiles[plan.tile];
  bt::Args p = bf16_tiled_args(plan, a, n0, n);
  p.partial = static_cast<float*>(ws);
  p.rt0 = n0 / (16 * t.rt);
  // Weights that only one work-group reads: past the caches (24576 x 4096 at 64
  // tokens 37.3 -> 34.0 us, 4096 x 12288 at 32 22.0 -> 20.3); beside the tokens
  // of a wide split it was slower (4096 x 4096 at 64 tokens 12.0 -> 12.8).
  p.nt = plan.tok_tiles == 1 && (plan.splits == 1 || t.tt <= 2);
  const int rc = ferret_bf16_tiled(plan.tile, p, st);
  if (rc != 0 || plan.splits == 1) return rc;
  return launch_splitk_reduce(p.partial, p.splits, p.M, p.N, p.ldo, p.residual, p.out, st);
}

// The same result from one launch with no partials.
static int launch_bf16_tiled_serial(const bt::Plan& plan, const SkinnyArgs& a, hipStream_t st) {
  return ferret_bf16_tiled_serial(plan.tile, bf16_tiled_args(plan, a, 0, a.N), st);
}

}  // namespace ferret

using namespace ferret;

size_t ferret_linear_bf16_workspace(int M, int N, int K) { return lin::workspace(M, N, K, cu_count()); }

size_t ferret_linear_bf16_aligned_workspace(int M, int N, int K) {
  return lin::aligned_workspace(M, N, K, cu_count());
}

extern "C" int ferret_linear_bf16(const void* x, const void* w, const void* residual, void* y, int M,
                                  int N, int K, void* ws, size_t ws_bytes, void* stream) {
  FERRET_REQUIRE(x && w && y, FERRET_ERR_NULL);
  FERRET_REQUIRE(M >= 1 && N >= 16 && K >= 128, FERRET_ERR_SHAPE);
  FERRET_REQUIRE(N % 16 == 0 && K % 128 == 0 && K / 128 <= 128, FERRET_ERR_SHAPE);
  const hipStream_t st = (hipStream_t)stream;
  SkinnyArgs a{};
  a.w = static_cast<const uint8_t*>(w);
  a.x = static_cast<const uint8_t*>(x);
  a.residual = static_cast<const uint16_t*>(residual);
  a.out = static_cast<uint16_t*>(y);
  a.M = M;
  a.N = N;
  a.K = K;
  a.units_n = N / 16;
  const lin::Route route = lin::route(M, N, K, cu_count(), x, w, residual, y, ws, ws_bytes);
  if (route.tiled.ok) return launch_bf16_tiled(route.tiled, a, 0, N, ws, st);
  const int splits = route.splits;
  if (splits > 1) {
    a.partial = static_cast<float*>(ws);
    a.ksplit = splits;
    const int rc = try_stream<kBF16, kStore, 1, 3, 8>(a, (M + 15) / 16, 0, st);
    if (rc != 1) {
      if (rc != 0) return rc;
      return launch_splitk_reduce(a.partial, splits, M, N, N, a.residual, a.out, st);
    }
    a.partial = nullptr;
    a.ksplit = 0;
  }
  // Unsplit: with >= 4 row units per CU, 4 waves of 8 K-steps per unit stream
  // faster than 8 waves of 4 (the work-group's units start sooner and reduce
  // over half the waves): GateUp 39.6 -> 36.7 us, LMHead 202 -> 195 us; with one
  // unit per CU (O) 8 waves keep more bytes in flight.
  const long long units = (long long)((M + 15) / 16) * (N / 16);
  int rc = 1;
  if (units >= 4LL * cu_count()) rc = try_stream<kBF16, kStore, 1, 4, 4>(a, (M + 15) / 16, 0, st);
  if (rc == 1) rc = try_stream<kBF16, kStore, 1, 3, 8>(a, (M + 15) / 16, 0, st);
  if (rc != 1) return rc;
  return launch_skinny<kBF16, kStore, 1>(a, (M + 15) / 16, st);
}

// ---- allocation-free decode linear (no counterpart in the reference).
// Callers that cannot allocate (code under HIP graph capture, serving loops)
// get the split-K partials of ferret_linear_bf16 from this file-scope device
// array instead of a workspace argument.  Each GPU holds its own copy until
// the process ends; its address is looked up once per device
// (hipGetSymbolAddress, with that device current) and only that address is
// handed to kernels.  Calls that overlap on one GPU share the array and race;
// every split writes all of its partials before the reduce reads them, so
// nothing needs clearing between calls.  Only shapes that the 16-token kernels
// split use it (lin::noalloc_shares_array); the tiled kernel's splits of all
// others run in its serial form.
constexpr size_t kNoAllocScratchBytes = 4u << 20;
static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];
static std::atomic<void*> g_scratch_ptr[64];

// Device address of `scratch` on the current device (cached per device), or
// the hipGetSymbolAddress error.
static hipError_t scratch_address(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (p == nullptr) {
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    if (p == nullptr) return hipErrorInvalidSymbol;
    g_scratch_ptr[dev].store(p, std::memory_order_release);
  }
  *out = p;
  return hipSuccess;
}

// Also looks the array's address up on the current device (errors are left
// for the entry point to report), so that a caller can do it before capturing
// ferret_linear_bf16_noalloc into a graph.
extern "C" size_t ferret_linear_bf16_noalloc_max_bytes(void) {
  void* p = nullptr;
  (void)scratch_address(&p);
  return kNoAllocScratchBytes;
}

extern "C" int ferret_linear_bf16_noalloc(const void* x, const void* w, const void* residual, void* y, int M,
                                          int N, int K, void* stream) {
  FERRET_REQUIRE(x && w && y, FERRET_ERR_NULL);
  FERRET_REQUIRE(M >= 1 && N >= 16 && K >= 128, FERRET_ERR_SHAPE);
  FERRET_REQUIRE(N % 16 == 0 && K % 128 == 0 && K / 128 <= 128, FERRET_ERR_SHAPE);
  const int splits = lin::stream_splits(M, N, K, cu_count());
  FERRET_REQUIRE(splits <= 1 || (size_t)splits * M * N * sizeof(float) <= kNoAllocScratchBytes, FERRET_ERR_WORKSPACE);
  const bt::Plan tiled = lin::tiled_plan(M, N, K, cu_count());
  const size_t need = lin::partial_bytes(tiled.splits, M, N);
  SkinnyArgs a{};
  a.w = static_cast<const uint8_t*>(w);
  a.x = static_cast<const uint8_t*>(x);
  a.residual = static_cast<const uint16_t*>(residual);
  a.out = static_cast<uint16_t*>(y);
  a.M = M;
  a.N = N;
  a.K = K;
  const bool aligned = lin::tiled_aligned(x, w, residual, y, nullptr);
  if (!lin::noalloc_shares_array(M, N, K, cu_count())) {
    if (tiled.ok && tiled.splits > 1 && aligned) return launch_bf16_tiled_serial(tiled, a, (hipStream_t)stream);
    return ferret_linear_bf16(x, w, residual, y, M, N, K, nullptr, 0, stream);
  }
  void* ws = nullptr;
  FERRET_HIP_CHECK(scratch_address(&ws));
  if (!tiled.ok || need <= kNoAllocScratchBytes || !aligned)
    return ferret_linear_bf16(x, w, residual, y, M, N, K, ws, kNoAllocScratchBytes, stream);
  // Partials larger than the array: the same plan over runs of whole row tiles
  // whose partials fit (each output's sums are those of one launch).
  const int tile_rows = 16 * bt::kTiles[tiled.tile].rt;
  const int rows = (int)(kNoAllocScratchBytes / ((size_t)tiled.splits * M * sizeof(float))) / tile_rows * tile_rows;
  for (int n0 = 0; n0 < N; n0 += rows) {
    const int rc = launch_bf16_tiled(tiled, a, n0, std::min(rows, N - n0), ws, (hipStream_t)stream);
    if (rc != 0) return rc;
  }
  return FERRET_OK;
}

extern "C" void launch_gemv(void* input, void* weight, void* residual, void* output, int N, int K,
                            void* stream) {
  (void)ferret_linear_bf16(input, weight, residual, output, 1, N, K, nullptr, 0, stream);
}

// Small-M FP8 block-scaled GEMM (M <= 16 per token tile); called by the dense
// FP8 entry point for skinny shapes.
int ferret_fp8_gemm_skinny(const void* a_, const float* sa, const void* b, const float* sb, void* c,
                           int M, int N, int K, hipStream_t st) {
  SkinnyArgs a{};
  a.w = static_cast<const uint8_t*>(b);
  a.w_scale = sb;
  a.x = static_cast<const uint8_t*>(a_);
  a.x_scale = sa;
  a.out = static_cast<uint16_t*>(c);
  a.M = M;
  a.N = N;
  a.K = K;
  a.units_n = N / 16;  // units of the per-unit fallback (RB = 1)
  // Short K (<= 2 K-steps per wave, e.g. K = 2048): two row blocks per unit
  // halve the per-unit reductions (o_proj, K = 2048: 8.2 -> 7.5 us); at K = 7168
  // one block with a deeper ring is faster (12.2 vs 13.5 us).
  // With at most one 16-row unit per CU (M = 16, N = 4096, K = 7168: 256 units)
  // the whole unit is requested up front, so more waves per unit, each with
  // fewer K-steps, shorten the first-byte-to-last-byte time: 14 waves x 4
  // K-steps (ring depth 4) run 9.0 us against 10.0 us for 8 x 7.
  const long long units16 = (long long)((M + 15) / 16) * (N / 16);
  int rc = 1;
  if ((K >> 7) <= 16) {
    rc = try_stream<kFP8, kStore, 2, 3, 8>(a, (M + 15) / 16, 0, st);
  } else {
    if ((K >> 7) % 14 == 0 && units16 <= cu_count()) rc = try_stream<kFP8, kStore, 1, 4, 14>(a, (M + 15) / 16, 0, st);
    if (rc == 1) rc = try_stream<kFP8, kStore, 1, 6, 8>(a, (M + 15) / 16, 0, st);
  }
  if (rc != 1) return rc;
  return launch_skinny<kFP8, kStore, 1>(a, (M + 15) / 16, st);
}

// Decode-sized FP8 MoE w13 (tile_m = 16).
int ferret_moe_w13_fp8_skinny(const void* x, const float* sx, const void* w, const float* sw,
                              const int32_t* sorted_pair, const int32_t* tiles, const int32_t* ntiles,
                              int max_tiles, long long num_pairs, int topk, int E, int N, int K, void* out,
                              hipStream_t st) {
  SkinnyArgs a{};
  a.w = static_cast<const uint8_t*>(w);
  a.w_scale = sw;
  a.x = static_cast<const uint8_t*>(x);
  a.x_scale = sx;
  a.out = static_cast<uint16_t*>(out);
  a.sorted_pair = sorted_pair;
  a.tiles = tiles;
  a.ntiles = ntiles;
  a.topk = topk;
  a.N = N;
  a.K = K;
  a.units_n = N / 32;
  a.pair_tiles = moe::w13_pairs(num_pairs, E, N, K >> 7, cu_count());
  if (max_tiles <= 0) return FERRET_OK;
  const int rc = try_stream<kFP8, kSilu, 2, 3, 8>(a, 0, max_tiles, st);
  if (rc != 1) return rc;
  return launch_skinny<kFP8, kSilu, 2>(a, max_tiles, st);
}

// Decode-sized FP8 MoE w2 / down projection (tile_m = 16): the A row and the
// output row of a sorted row are both its routed pair (topk = 1 indexing).
int ferret_moe_w2_fp8_skinny(const void* h, const float* sh, const void* w, const float* sw,
                             const int32_t* sorted_pair, const int32_t* tiles, const int32_t* ntiles,
                             int max_tiles, long long num_pairs, int E, int N, int K, void* out, hipStream_t st) {
  SkinnyArgs a{};
  a.w = static_cast<const uint8_t*>(w);
  a.w_scale = sw;
  a.x = static_cast<const uint8_t*>(h);
  a.x_scale = sh;
  a.out = static_cast<uint16_t*>(out);
  a.sorted_pair = sorted_pair;
  a.tiles = tiles;
  a.ntiles = ntiles;
  a.topk = 1;
  a.N = N;
  a.K = K;
  if (max_tiles <= 0) return FERRET_OK;
// K = 2048 gives 8 waves only 2 K-steps per 16-row unit, so wider units with
// fewer waves pay (fewer cross-wave reductions per weight byte): two blocks
// per unit took 32 experts x 1 row 79 -> 71 us and 256 experts 605 -> 592 us;
// four blocks on 4 waves of 4 K-steps take 256 experts 593 -> 555 us and
// 32 experts x 16 rows 82 -> 79 us.  The per-unit kernel, which ran K / 128 of
// 12 and 6 before, reached 4.2 TB/s of weights: 256 experts x 4 rows, N = 7168,
// K = 1536 659 -> 425 us (6.5 TB/s); with 15 rows 1079 -> 552, K = 768 634 -> 350.
  a.units_n = N / 16;  // units of the per-unit fallback (RB = 1); try_stream derives its own
  a.pair_tiles = moe::w2_pairs(num_pairs, E, N, K >> 7, cu_count());
  if (moe::w2_streams(K >> 7, w, (long long)max_tiles * (N / 64), cu_count())) {
    int rc = try_stream<kFP8, kStore, 4, 3, 4>(a, 0, max_tiles, st);
    if (rc == 1) rc = try_half_stream<kFP8, kStore, 4, 3>(a, max_tiles, st);
    if (rc != 1) return rc;
  }
  return launch_skinny<kFP8, kStore, 1>(a, max_tiles, st);
}

namespace ferret {

// The W4A16 w13 decode over either weight layout (F = kINT4: the checkpoint's
// [E, N, K/8] words; kINT4T: the same words in 16-row x 128-K tiles).
template <int F>
static int moe_w13_w4a16(const void* x, const int32_t* wq, const void* ws, const int32_t* sorted_pair,
                         const int32_t* tiles, const int32_t* ntiles, int max_tiles, int tile_m, int T, int topk,
                         int E, int N, int K, void* out, hipStream_t st) {
  FERRET_REQUIRE(x && wq && ws && sorted_pair && tiles && ntiles && out, FERRET_ERR_NULL);
  FERRET_REQUIRE(T >= 1 && topk >= 1 && E >= 1 && max_tiles >= 0, FERRET_ERR_SHAPE);
  FERRET_REQUIRE(tile_m == 16 && N % 32 == 0 && N >= 32 && K % 128 == 0 && K >= 128, FERRET_ERR_SHAPE);
  SkinnyArgs a{};
  a.w = reinterpret_cast<const uint8_t*>(wq);
  a.w_scale = ws;
  a.x = static_cast<const uint8_t*>(x);
  a.out = static_cast<uint16_t*>(out);
  a.sorted_pair = sorted_pair;
  a.tiles = tiles;
  a.ntiles = ntiles;
  a.topk = topk;
  a.N = N;
  a.K = K;
  a.units_n = N / 32;
  if (max_tiles <= 0) return FERRET_OK;
  // The two-tile kernel loads x and the weights as 16-byte chunks, the scales
  // as words, and stores 8 bytes.  It sums K in the spans of the other kernels'
  // waves (the stream kernel's eight, or the per-unit kernel's), in their order.
  const auto bits = [](const void* p) { return reinterpret_cast<uintptr_t>(p); };
  const int nkb = K >> 7, eighth = nkb % 8 == 0 ? nkb / 8 : 0;
  const bool stream = (eighth == 2 || eighth == 4 || eighth == 7 || eighth == 8) && (bits(ws) & 15) == 0;
  const int span = stream ? eighth : unit_steps(nkb);
  if (span != 0 && ((bits(x) | bits(wq)) & 15) == 0 && (bits(ws) & 3) == 0 && (bits(out) & 7) == 0 &&
      i4::takes((long long)T * topk, E, N, nkb, max_tiles, cu_count(), stream, F == kINT4T))
    return ferret_int4_moe(a, F == kINT4T, span, max_tiles, cu_count(), st);
  const int rc = try_stream<F, kSilu, 2, 5, 8>(a, 0, max_tiles, st);
  if (rc != 1) return rc;
  return launch_skinny<F, kSilu, 2>(a, max_tiles, st);
}

// One thread per 16-byte chunk of the tiled output:
// out[e][n/16][k/128][n%16][64 B] = the K-step k/128 slice (64 B) of row n.
__global__ __launch_bounds__(256) void int4_tile_kernel(const uint8_t* __restrict__ w, uint8_t* __restrict__ t,
                                                        long long nchunks, int nkb) {
  const long long row_bytes = (long long)nkb * 64;
  for (long long o = (long long)blockIdx.x * 256 + threadIdx.x; o < nchunks; o += (long long)gridDim.x * 256) {
    const int c = (int)(o & 3);
    const int row = (int)((o >> 2) & 15);
    const long long tile = o >> 6;  // (e * N/16 + block) * nkb + k-step
    const int ks = (int)(tile % nkb);
    const long long eb = tile / nkb;  // e * N/16 + block: rows 16 * eb .. of the [E * N] row list
    const u32x4 v = ld_u32x4_stream(w + (eb * 16 + row) * row_bytes + ks * 64 + c * 16);
    *reinterpret_cast<u32x4*>(t + o * 16) = v;
  }
}

}  // namespace ferret

using namespace ferret;

extern "C" int ferret_moe_w13_w4a16(const void* x, const int32_t* wq, const void* ws,
                                    const int32_t* sorted_pair, const int32_t* tiles,
                                    const int32_t* ntiles, int max_tiles, int tile_m, int T, int topk,
                                    int E, int N, int K, void* out, void* stream) {
  return moe_w13_w4a16<kINT4>(x, wq, ws, sorted_pair, tiles, ntiles, max_tiles, tile_m, T, topk, E, N, K, out,
                              (hipStream_t)stream);
}

extern "C" int ferret_moe_w13_w4a16_tiled(const void* x, const void* wq_tiled, const void* ws,
                                          const int32_t* sorted_pair, const int32_t* tiles,
                                          const int32_t* ntiles, int max_tiles, int tile_m, int T, int topk,
                                          int E, int N, int K, void* out, void* stream) {
  return moe_w13_w4a16<kINT4T>(x, static_cast<const int32_t*>(wq_tiled), ws, sorted_pair, tiles, ntiles,
                               max_tiles, tile_m, T, topk, E, N, K, out, (hipStream_t)stream);
}

extern "C" int ferret_int4_tile_weights(const int32_t* wq, void* wq_tiled, int E, int N, int K, void* stream) {
  FERRET_REQUIRE(wq && wq_tiled, FERRET_ERR_NULL);
  FERRET_REQUIRE(E >= 1 && N >= 16 && N % 16 == 0 && K >= 128 && K % 128 == 0, FERRET_ERR_SHAPE);
  const long long bytes = (long long)E * N * (K / 2);
  const uint8_t* src = reinterpret_cast<const uint8_t*>(wq);
  uint8_t* dst = static_cast<uint8_t*>(wq_tiled);
  FERRET_REQUIRE(dst + bytes <= src || src + bytes <= dst, FERRET_ERR_SHAPE);  // out of place only
  const long long nchunks = bytes / 16;
  const unsigned grid = (unsigned)std::min<long long>((nchunks + 255) / 256, 65536);
  hipLaunchKernelGGL(int4_tile_kernel, dim3(grid), dim3(256), 0, (hipStream_t)stream, src, dst, nchunks, K / 128);
  return (int)hipGetLastError();
}
