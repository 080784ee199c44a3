// LDS-tiled bf16 product for gfx950, y[M,N] = x[M,K] . w[N,K]^T (+ residual),
// past the 16 tokens that a unit of the stream kernel holds.
//
// HBM-bound on the weights up to about 100 tokens.  A work-group of 8 waves
// takes RT x 16 weight rows by all tokens (TT x 16) over one K split; both
// operands go global -> LDS in stages of 128 K (256 bytes of each row, whole
// lines) through a ring of NS stages, one barrier per stage.  Weights are read
// once per work-group, the tokens once per row tile (from L2), so RT is the
// larger of two sizes wherever the row tiles still fill the CUs.  The waves
// split the K of a stage as well as the tile (WK), which keeps the fragment
// reads near one LDS read per MFMA at small tiles; the parts meet in LDS once.
//
// Every work-group starts at another K-step (row tile index modulo its steps)
// and wraps around: in lockstep, all of them read the same columns of rows a
// power of two apart, which sit on few of the memory channels (24576 x 4096 at
// 64 tokens: 46.6 -> 37.3 us, 34.0 with the weights non-temporal).
//
// Serial form (kSerial): a work-group of 16 weight rows runs all K splits of a
// plan, G at a time, and sums them itself, in the order and from the K rotation
// of the plan's own tiles: their results bit for bit with no partials in memory.
// For the allocation-free entry where the 16-token kernels need no split, so that
// calls there share no memory.  Over 1509 such shapes of 1 .. 128 tokens 1.44
// times as fast as those kernels (geometric mean; 32 of them more than 4 % slower,
// by up to 33 %), the split form about 1.7 times.
//
// Measured, start to now (the 16-token stream kernel once per 16 tokens):
// 4096 x 12288 + residual at 48 tokens 53.4 -> 23 us, 24576 x 4096 at 64 tokens
// 77.0 -> 34.2 us, at 128 tokens 141.6 -> 51.6 us.
#include "common.hpp"
#include "bf16_tiled.hpp"

namespace ferret {
namespace bt {

// Waves: WR along the rows, WT along the tokens, WK along the K of a stage; G such
// groups, each with a ring of its own, on K splits of their own (serial form).
template <int RT, int TT, int KS, int NS, int WR, int WT, int WK, int G = 1>
struct Cfg {
  static constexpr int kRows = 16 * RT, kToks = 16 * TT;
  static constexpr int kRowB = KS * 2;                         // bytes of a stage row
  static constexpr int kStage = (RT + TT) * 16 * kRowB;
  static constexpr int kInstr = kStage / 1024;                 // 1-KB loads of a stage: weights, then tokens
  static constexpr int kWInstr = RT * 16 * kRowB / 1024;
  static constexpr int kIRows = 1024 / kRowB;                  // rows of a load
  static constexpr int kWaves = WR * WT * WK, kThreads = 64 * kWaves * G;
  static constexpr int kLd = (kInstr + kWaves - 1) / kWaves;   // loads per wave (past kInstr: the last one again)
  static constexpr int kRB = RT / WR, kTB = TT / WT, kKB = KS / 32 / WK;  // row and token blocks, MFMAs deep, per wave
  static constexpr int kPitch = kRows + 4;                     // floats of a token row of the epilogue
  static constexpr int kRing = NS * kStage;                    // of a group of waves
  static constexpr int kEpi = G * WK * kToks * kPitch * 4;
  static constexpr int kLds = G * kRing > kEpi ? G * kRing : kEpi;
  static constexpr int kQuads = kRows / 4;                     // groups of four outputs of a token
  static constexpr int kOuts = (kToks * kQuads + kThreads - 1) / kThreads;  // of a thread
  static_assert(kThreads <= 1024 && RT % WR == 0 && TT % WT == 0 && (KS / 32) % WK == 0, "waves");
  static_assert(kStage % 1024 == 0 && kLds <= 160 * 1024, "LDS budget");
  static_assert(NS >= 2 && (NS - 2) * kLd < 63, "vmcnt range");
};

// Slot of 16-byte chunk c of stage row `row`: the 16 rows of a fragment read
// fall on distinct banks.
template <int KS>
__device__ __forceinline__ int swz(int row, int c) {
  return KS == 128 ? c ^ (((row & 7) << 1) | ((row >> 3) & 1)) : c ^ ((row & 7) ^ ((row >> 3) & 1));
}

// Wait until at most min(n, N) stages of L loads are in flight.
template <int L, int N>
__device__ __forceinline__ void wait_younger(int n) {
  if constexpr (N == 0) {
    wait_vmcnt<0>();
  } else {
    if (n >= N) wait_vmcnt<N * L>();
    else wait_younger<L, N - 1>(n);
  }
}

template <int RT, int TT, int KS, int NS, int WR, int WT, int WK, bool kSerial = false, int G = 1>
__global__ __launch_bounds__(64 * WR * WT * WK * G) void bf16_tiled_kernel(Args p) {
  using C = Cfg<RT, TT, KS, NS, WR, WT, WK, G>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wg_wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wg_wave % C::kWaves, group = wg_wave / C::kWaves;
  uint8_t* ring = lds + group * C::kRing;
  const int r = lane & 15, g = lane >> 4;
  const int wr = wave % WR, wt = (wave / WR) % WT, wk = wave / (WR * WT);

  // Splits vary fastest: with 2, 4 or 8 of them an XCD (work-groups are dealt
  // to the 8 round-robin) reads one K-range of the tokens only.
  const int first_split = kSerial ? 0 : blockIdx.x % p.splits, last_split = kSerial ? p.splits - 1 : first_split;
  const int tile = kSerial ? blockIdx.x : blockIdx.x / p.splits;
  const int tt = tile % p.tok_tiles, rt = tile / p.tok_tiles;
  const int nkb = p.K / KS;
  const int row0 = rt * C::kRows, tok0 = tt * C::kToks;
  const int place = kSerial ? row0 / p.rot_rows : p.rt0 + rt;  // in the K rotation
  f32x4 total[kSerial ? C::kOuts : 1];

  for (int split0 = first_split; split0 <= last_split; split0 += G) {
    const int split = G == 1 ? split0 : min(split0 + group, p.splits);  // p.splits: none left for this group
    const int k0 = (int)((long long)split * nkb / p.splits), k1 = (int)((long long)(split + 1) * nkb / p.splits);
    const int nsteps = split < p.splits ? k1 - k0 : 0;
    const int wg_steps = G == 1 ? nsteps : (nkb + p.splits - 1) / p.splits;  // of the longest group: they share barriers
    const int rot = nsteps > 0 ? (int)((unsigned)place % (unsigned)nsteps) : 0;

    const uint8_t* src[C::kLd];
    int dst[C::kLd];
#pragma unroll
    for (int i = 0; i < C::kLd; ++i) {
      const int j = min(wave * C::kLd + i, C::kInstr - 1);
      constexpr int LR = 64 / C::kIRows;         // lanes of a row
      const int lr = C::kIRows * j + lane / LR;  // stage row
      const int c = swz<KS>(lr & 15, lane % LR);
      const bool is_w = j < C::kWInstr;
      // rows past N or M repeat the last one (never stored)
      const size_t row = is_w ? min(row0 + lr, p.N - 1) : min(tok0 + lr - C::kRows, p.M - 1);
      src[i] = (is_w ? p.w : p.x) + (row * p.K + (size_t)k0 * KS) * 2 + c * 16;
      dst[i] = j * 1024;
    }
    auto issue = [&](int step) {
      uint8_t* st = ring + (step % NS) * C::kStage;
      const int ks = step + rot < nsteps ? step + rot : step + rot - nsteps;
#pragma unroll
      for (int i = 0; i < C::kLd; ++i) {
        if (p.nt && wave * C::kLd + i < C::kWInstr) g2l_16_nt(src[i] + (size_t)ks * C::kRowB, st + dst[i]);
        else g2l_16(src[i] + (size_t)ks * C::kRowB, st + dst[i]);
      }
    };

    f32x4 acc[C::kRB][C::kTB];
#pragma unroll
    for (int a = 0; a < C::kRB; ++a)
#pragma unroll
      for (int b = 0; b < C::kTB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int s = 0; s < NS - 1; ++s)
      if (s < nsteps) issue(s);
    for (int step = 0; step < wg_steps; ++step) {
      // This stage has landed for every wave, and the slot of the stage before
      // (the one refilled below) has been read by every wave.
      wait_younger<C::kLd, NS - 2>(nsteps - 1 - step);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
      if (step + NS - 1 < nsteps) issue(step + NS - 1);
      __builtin_amdgcn_sched_barrier(0);
      if (G > 1 && step >= nsteps) continue;
      const uint8_t* st = ring + (step % NS) * C::kStage;
#pragma unroll
      for (int k = 0; k < C::kKB; ++k) {
        const int c = swz<KS>(r, 4 * (wk * C::kKB + k) + g) << 4;
        u32x4 wf[C::kRB], xf[C::kTB];
#pragma unroll
        for (int a = 0; a < C::kRB; ++a)
          wf[a] = *reinterpret_cast<const u32x4*>(st + ((wr * C::kRB + a) * 16 + r) * C::kRowB + c);
#pragma unroll
        for (int b = 0; b < C::kTB; ++b)
          xf[b] = *reinterpret_cast<const u32x4*>(st + (C::kRows + (wt * C::kTB + b) * 16 + r) * C::kRowB + c);
#pragma unroll
        for (int a = 0; a < C::kRB; ++a)
#pragma unroll
          for (int b = 0; b < C::kTB; ++b) acc[a][b] = mfma_bf16_16x16x32(wf[a], xf[b], acc[a][b]);
      }
    }

    // Epilogue through the idle ring: [K part][token][row], then four outputs of
    // a token per thread, the parts in order.
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    float* red = reinterpret_cast<float*>(lds);
#pragma unroll
    for (int a = 0; a < C::kRB; ++a)
#pragma unroll
      for (int b = 0; b < C::kTB; ++b)
        *reinterpret_cast<f32x4*>(red + ((group * WK + wk) * C::kToks + (wt * C::kTB + b) * 16 + r) * C::kPitch +
                                  (wr * C::kRB + a) * 16 + 4 * g) = acc[a][b];
    __syncthreads();
    constexpr int Q = C::kQuads;
#pragma unroll(kSerial ? C::kOuts : 1)
    for (int o = 0; o < C::kOuts; ++o) {
      const int i = threadIdx.x + o * C::kThreads;
      const int t = i / Q, q = i % Q, n = row0 + 4 * q;
      if (i >= C::kToks * Q || tok0 + t >= p.M || n >= p.N) continue;
      f32x4 v;
#pragma unroll
      for (int h = 0; h < G; ++h) {
        if (G > 1 && split0 + h >= p.splits) break;
        const float* part = red + (h * WK * C::kToks + t) * C::kPitch + 4 * q;
        v = *reinterpret_cast<const f32x4*>(part);
#pragma unroll
        for (int k = 1; k < WK; ++k) v += *reinterpret_cast<const f32x4*>(part + k * C::kToks * C::kPitch);
        if constexpr (kSerial) total[o] = split0 + h == 0 ? v : total[o] + v;
      }
      if constexpr (kSerial) {
        if (split0 + G <= last_split) continue;
        v = total[o];
      }
      if (!kSerial && p.splits > 1) {  // summed (+ residual) by the reduce kernel
        *reinterpret_cast<f32x4*>(p.partial + ((size_t)split * p.M + tok0 + t) * p.N + n) = v;
      } else {
        const size_t at = (size_t)(tok0 + t) * p.ldo + n;
        if (p.residual) {
          const u32x2 s = *reinterpret_cast<const u32x2*>(p.residual + at);
          v[0] += __uint_as_float(s[0] << 16);
          v[1] += __uint_as_float(s[0] & 0xffff0000u);
          v[2] += __uint_as_float(s[1] << 16);
          v[3] += __uint_as_float(s[1] & 0xffff0000u);
        }
        *reinterpret_cast<u32x2*>(p.out + at) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      }
    }
    // The sums are read before the next split's stages overwrite them.
    if constexpr (kSerial) __syncthreads();
  }
}

// Tile I of kTiles, its waves split by WR, WT, WK.
template <int I, int WR, int WT, int WK>
static int launch(const Args& p, hipStream_t st) {
  constexpr Tile t = kTiles[I];
  using C = Cfg<t.rt, t.tt, t.ks, t.ns, WR, WT, WK>;
  constexpr auto kernel = bf16_tiled_kernel<t.rt, t.tt, t.ks, t.ns, WR, WT, WK>;
  FERRET_HIP_CHECK((set_lds_limit_once<bf16_tiled_kernel<t.rt, t.tt, t.ks, t.ns, WR, WT, WK>>(C::kLds)));
  const int row_tiles = (p.N + C::kRows - 1) / C::kRows;
  hipLaunchKernelGGL(kernel, dim3(row_tiles * p.tok_tiles * p.splits), dim3(C::kThreads), C::kLds, st, p);
  return (int)hipGetLastError();
}

// The serial form of a plan's tile by TT x 16 tokens: its waves' WK, G splits at a time.
template <int TT, int KS, int NS, int WT, int WK, int G>
static int launch_serial(Args p, hipStream_t st) {
  using C = Cfg<1, TT, KS, NS, 1, WT, WK, G>;
  constexpr auto kernel = bf16_tiled_kernel<1, TT, KS, NS, 1, WT, WK, true, G>;
  FERRET_HIP_CHECK((set_lds_limit_once<bf16_tiled_kernel<1, TT, KS, NS, 1, WT, WK, true, G>>(C::kLds)));
  p.tok_tiles = (p.M + C::kToks - 1) / C::kToks;
  p.nt = p.tok_tiles == 1;
  hipLaunchKernelGGL(kernel, dim3(p.N / 16 * p.tok_tiles), dim3(C::kThreads), C::kLds, st, p);
  return (int)hipGetLastError();
}

}  // namespace bt
}  // namespace ferret

int ferret_bf16_tiled(int tile, const ferret::bt::Args& p, hipStream_t st) {
  using namespace ferret::bt;
  static_assert(kNumTiles == 12, "one case per tile");
  switch (tile) {
    case 0: return launch<0, 2, 1, 4>(p, st);
    case 1: return launch<1, 2, 1, 4>(p, st);
    case 2: return launch<2, 2, 1, 4>(p, st);
    case 3: return launch<3, 2, 1, 4>(p, st);
    case 4: return launch<4, 2, 1, 4>(p, st);
    case 5: return launch<5, 2, 1, 4>(p, st);
    case 6: return launch<6, 2, 2, 2>(p, st);
    case 7: return launch<7, 2, 2, 2>(p, st);
    case 8: return launch<8, 2, 2, 2>(p, st);
    case 9: return launch<9, 2, 2, 2>(p, st);
    case 10: return launch<10, 2, 4, 1>(p, st);
    case 11: return launch<11, 2, 4, 1>(p, st);
  }
  return FERRET_ERR_SHAPE;
}

int ferret_bf16_tiled_serial(int tile, ferret::bt::Args p, hipStream_t st) {
  using namespace ferret::bt;
  static_assert(kNumTiles == 12, "one case per tile");
  p.rot_rows = 16 * kTiles[tile].rt;
  // Few rows leave CUs idle where a work-group takes all tokens: below 2560 of
  // them it takes 16 (geometric means against the 16-token kernels: 1.28 - 1.75
  // there against 0.55 - 1.2; from 2560 rows on 1.0 - 1.7 against 1.3 - 3).  As
  // many splits at a time as the plan has, or a quarter to all of the waves idle:
  // 10304 x 3072 at 2 tokens (3 splits) 26.3 us with 8 at a time, 13.8 with 4; 7664
  // x 1536 at 9 (2 splits) 8.9 with 4, 6.4 with 2.  Plans of 64 K a stage pick their
  // 128-token tile for few tokens too: up to 32 it takes 16 (6368 x 7168 at 25 53.1
  // us with 128).
  if (p.M <= 16 && tile < 6)
    return p.splits <= 2 ? launch_serial<1, 128, 4, 1, 4, 2>(p, st) : launch_serial<1, 128, 4, 1, 4, 4>(p, st);
  if (p.M <= 16 || p.N < 2560 || (tile == 11 && p.M <= 32)) {
    if (tile < 6) return launch_serial<1, 128, 2, 1, 4, 4>(p, st);
    if (tile < 10) return launch_serial<1, 128, 2, 1, 2, 4>(p, st);
    if (tile < 11) return launch_serial<1, 128, 2, 1, 1, 4>(p, st);
    return p.splits <= 4 ? launch_serial<1, 64, 4, 1, 1, 4>(p, st) : launch_serial<1, 64, 2, 1, 1, 8>(p, st);
  }
  switch (tile) {
    case 0: case 1: return FERRET_ERR_SHAPE;  // 16 tokens: above
    case 2: case 3: return launch_serial<2, 128, 6, 1, 4, 1>(p, st);
    case 4: case 5: return launch_serial<3, 128, 5, 1, 4, 1>(p, st);
    case 6: case 7: return launch_serial<4, 128, 4, 2, 2, 1>(p, st);
    case 8: case 9: return launch_serial<6, 128, 4, 2, 2, 1>(p, st);
    case 10: return launch_serial<8, 128, 4, 4, 1, 1>(p, st);
    case 11: return launch_serial<8, 64, 4, 4, 1, 1>(p, st);
  }
  return FERRET_ERR_SHAPE;
}
