// FP8 (OCP e4m3) block-scaled product for gfx950 between the decode kernels
// (16 tokens) and the large tiles: c[M,N] = sum_kb (a_kb . b_kb^T) sa sb for
// 16 < M <= 256 and the K where it beats the split-K tiles of fp8_tiled.hip, and
// past 256 tokens where its work-groups fit one round.
//
// These shapes are a few microseconds of loads between fixed costs: a launch,
// the first stage, the epilogue and, where K is split, 13 MB of fp32 partials
// (8 splits of 100 x 4096) and a second launch.  Small tiles (32 or 64 weight
// rows by all tokens) fill the CUs with no split or half the splits of 128 x
// 128 tiles.  Both operands go global -> LDS in stages of 256 K (two scale
// blocks, 256 bytes of each row) through a short ring: more than two or three
// stages in flight were slower.  Of the 8 waves WK = 2 halves each take one
// scale block of every stage, so a wave widens its fragments (exactly, to bf16),
// chains four MFMAs per 16 x 16 block and folds them with sa * sb; the halves
// meet in LDS once.
//
// Measured against the split-K tiles (us): 7168 x 2048 at 24 / 64 / 100 / 256
// tokens 9.9 / 10.3 / 12.7 / 17.3 against 10.6 / 13.6 / 17.0 / 22.2; 4096 x 512
// 4.8 / 4.7 / 5.6 / 6.4 against 6.9 / 7.8 / 8.9 / 12.1; 4096 x 4096 at 100
// tokens 15.8 against 18.5.  The K loop is not bound by the widening (without
// it 0.3 - 0.6 us less) nor by the MFMAs but by the loads' round trip.
#include "common.hpp"
#include "fp8_mid.hpp"

namespace ferret {
namespace mid {

// 8 waves: WR along the rows, WT along the tokens, 2 along the scale blocks.
template <int RT, int TT, int NS, int WR, int WT>
struct Cfg {
  static constexpr int kRows = 16 * RT, kToks = 16 * TT;
  static constexpr int kOps = (RT + TT) * 16 * 256;            // operand bytes of a stage
  static constexpr int kSInstr = 2 * kToks / 64;               // 64-lane loads of the tokens' scales (block 0, block 1)
  static constexpr int kStage = kOps + 1024;                   // + the scales (at most 256 of them)
  static constexpr int kInstr = kOps / 1024;                   // 1-KB operand loads: weights, then tokens
  static constexpr int kWInstr = RT * 4;
  static constexpr int kLd = (kInstr + 7) / 8;                 // operand loads per wave (past kInstr: the last again)
  static constexpr int kL = kLd + 1;                           // + one scale load (past kSInstr: the last again)
  static constexpr int kRB = RT / WR, kTB = TT / WT;           // row and token blocks per wave
  static constexpr int kPitch = kRows + 4;                     // floats of a token row of the epilogue
  static constexpr int kEpi = 2 * kToks * kPitch * 4;
  static constexpr int kLds = NS * kStage > kEpi ? NS * kStage : kEpi;
  static_assert(WR * WT == 4 && RT % WR == 0 && TT % WT == 0, "8 waves");
  static_assert(128 % kRows == 0 && kSInstr >= 1 && kSInstr <= 4, "one weight-scale row; scales fit their KB");
  static_assert(kLds <= 160 * 1024 && NS >= 2 && (NS - 2) * kL < 63, "LDS and vmcnt range");
};

// Slot of 16-byte chunk c of stage row `row`: the 16 rows of a fragment read
// fall on distinct banks.
__device__ __forceinline__ int swz(int row, int c) { return c ^ (((row & 7) << 1) | ((row >> 3) & 1)); }

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

template <int RT, int TT, int NS, int WR, int WT>
__global__ __launch_bounds__(512) void fp8_mid_kernel(Args p) {
  using C = Cfg<RT, TT, NS, WR, WT>;
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int wr = wave % WR, wt = (wave / WR) % WT, wk = wave / 4;

  // Splits vary fastest (2, 4 or 8): an XCD reads one K-range of the tokens.
  const int split = blockIdx.x % p.splits;
  const int tile = blockIdx.x / p.splits;
  const int tt = tile % p.tok_tiles, rt = tile / p.tok_tiles;
  const int nkb = p.K >> 7;
  const int k0 = (int)((long long)split * nkb / p.splits), k1 = (int)((long long)(split + 1) * nkb / p.splits);
  const int nblk = k1 - k0;           // scale blocks of this split
  const int nsteps = (nblk + 1) / 2;  // an odd count leaves the last stage one block
  const int row0 = rt * C::kRows, tok0 = tt * C::kToks;

  const uint8_t* src[C::kLd];
  int dst[C::kLd];
  bool second[C::kLd];  // this lane's chunk lies in the stage's second block
#pragma unroll
  for (int i = 0; i < C::kLd; ++i) {
    const int j = min(wave * C::kLd + i, C::kInstr - 1);
    const int lr = 4 * j + (lane >> 4);  // stage row: weight rows, then token rows
    const int c = swz(lr & 15, lane & 15);
    const bool is_w = j < C::kWInstr;
    const size_t row = is_w ? row0 + lr : min(tok0 + lr - C::kRows, p.M - 1);  // tokens past M repeat the last
    src[i] = (is_w ? p.b : p.a) + row * p.K + (size_t)k0 * 128 + c * 16;
    dst[i] = j * 1024;
    second[i] = c >= 8;
  }
  const int sw = min(wave, C::kSInstr - 1);
  const int se = sw * 64 + lane;  // scale entry: [block][token]
  const float* ssrc = p.sa + (size_t)min(tok0 + se % C::kToks, p.M - 1) * nkb + k0;
  const int sblk = se / C::kToks;
  auto issue = [&](int step) {
    uint8_t* st = lds + (step % NS) * C::kStage;
    const bool half = 2 * step + 1 >= nblk;  // no second block: its bytes repeat the first's
#pragma unroll
    for (int i = 0; i < C::kLd; ++i) {
      const uint8_t* s = src[i] + (size_t)step * 256 - (half && second[i] ? 128 : 0);
      if (wave * C::kLd + i < C::kWInstr) g2l_16_nt(s, st + dst[i]);
      else g2l_16(s, st + dst[i]);
    }
    g2l_4(ssrc + 2 * step + (half ? 0 : sblk), st + C::kOps + sw * 256);
  };

  // The tile's weight scales: lane l holds blocks l and 64 + l of the split.
  const float* sbp = p.sb + (size_t)(row0 >> 7) * nkb + k0;
  const float sb_lo = lane < nblk ? sbp[lane] : 0.f;
  const float sb_hi = 64 + lane < nblk ? sbp[64 + lane] : 0.f;

  f32x4 acc[C::kRB][C::kTB];
#pragma unroll
  for (int a = 0; a < C::kRB; ++a)
#pragma unroll
    for (int b = 0; b < C::kTB; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
  for (int s = 0; s < NS - 1; ++s)
    if (s < nsteps) issue(s);
  for (int step = 0; step < nsteps; ++step) {
    // This stage has landed for every wave, and the slot of the stage before
    // (the one refilled below) has been read by every wave.
    wait_younger<C::kL, NS - 2>(nsteps - 1 - step);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (step + NS - 1 < nsteps) issue(step + NS - 1);
    __builtin_amdgcn_sched_barrier(0);
    const int kb = 2 * step + wk;
    if (kb >= nblk) continue;  // the second half of an odd last stage
    const uint8_t* st = lds + (step % NS) * C::kStage;
    const float* ss = reinterpret_cast<const float*>(st + C::kOps) + wk * C::kToks;
    const float sbv = __builtin_bit_cast(float, __builtin_amdgcn_readlane(
        __builtin_bit_cast(int, kb < 64 ? sb_lo : sb_hi), kb & 63));
    // Lane (r, g): K 32g .. +32 of the block, 8 per MFMA.
    const int c0 = swz(r, 8 * wk + 2 * g) << 4, c1 = swz(r, 8 * wk + 2 * g + 1) << 4;
    auto frag = [&](int row, bf16x8 (&f)[4]) {
      const u32x4 lo = *reinterpret_cast<const u32x4*>(st + row * 256 + c0);
      const u32x4 hi = *reinterpret_cast<const u32x4*>(st + row * 256 + c1);
      f[0] = e4m3x8_to_bf16x8(lo[0], lo[1]);
      f[1] = e4m3x8_to_bf16x8(lo[2], lo[3]);
      f[2] = e4m3x8_to_bf16x8(hi[0], hi[1]);
      f[3] = e4m3x8_to_bf16x8(hi[2], hi[3]);
    };
    bf16x8 xf[C::kTB][4];
    float sc[C::kTB];
#pragma unroll
    for (int b = 0; b < C::kTB; ++b) {
      const int t = (wt * C::kTB + b) * 16 + r;
      frag(C::kRows + t, xf[b]);
      sc[b] = ss[t] * sbv;
    }
#pragma unroll
    for (int a = 0; a < C::kRB; ++a) {
      bf16x8 wf[4];
      frag((wr * C::kRB + a) * 16 + r, wf);
#pragma unroll
      for (int b = 0; b < C::kTB; ++b) {
        f32x4 part = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 4; ++j) part = mfma_bf16(wf[j], xf[b][j], part);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[a][b][i] = fmaf(part[i], sc[b], acc[a][b][i]);
      }
    }
  }

  // Epilogue through the idle ring: [half][token][row], then four outputs of a
  // token per thread.
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int a = 0; a < C::kRB; ++a)
#pragma unroll
    for (int b = 0; b < C::kTB; ++b)
      *reinterpret_cast<f32x4*>(red + (wk * C::kToks + (wt * C::kTB + b) * 16 + r) * C::kPitch +
                                (wr * C::kRB + a) * 16 + 4 * g) = acc[a][b];
  __syncthreads();
  constexpr int Q = C::kRows / 4;
  for (int i = threadIdx.x; i < C::kToks * Q; i += 512) {
    const int t = i / Q, q = i % Q;
    if (tok0 + t >= p.M) continue;
    const f32x4 v = *reinterpret_cast<const f32x4*>(red + t * C::kPitch + 4 * q) +
                    *reinterpret_cast<const f32x4*>(red + (C::kToks + t) * C::kPitch + 4 * q);
    const size_t o = (size_t)(tok0 + t) * p.N + row0 + 4 * q;
    if (p.splits > 1) *reinterpret_cast<f32x4*>(p.partial + (size_t)split * p.M * p.N + o) = v;
    else *reinterpret_cast<u32x2*>(p.out + o) = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
  }
}

template <int I, int WR, int WT>
static int launch(const Args& p, hipStream_t st) {
  constexpr Tile t = kTiles[I];
  using C = Cfg<t.rt, t.tt, t.ns, WR, WT>;
  FERRET_HIP_CHECK((set_lds_limit_once<fp8_mid_kernel<t.rt, t.tt, t.ns, WR, WT>>(C::kLds)));
  hipLaunchKernelGGL((fp8_mid_kernel<t.rt, t.tt, t.ns, WR, WT>), dim3(p.N / C::kRows * p.tok_tiles * p.splits),
                     dim3(512), C::kLds, st, p);
  return (int)hipGetLastError();
}

}  // namespace mid
}  // namespace ferret

int ferret_fp8_mid(int tile, const ferret::mid::Args& p, hipStream_t st) {
  using namespace ferret::mid;
  static_assert(kNumTiles == 5, "one case per tile");
  switch (tile) {
    case 0: return launch<0, 4, 1>(p, st);
    case 1: return launch<1, 2, 2>(p, st);
    case 2: return launch<2, 2, 2>(p, st);
    case 3: return launch<3, 2, 2>(p, st);
    case 4: return launch<4, 2, 2>(p, st);
  }
  return FERRET_ERR_SHAPE;
}
