// INT4 W4A16 MoE gate-up (w13) product with fused SiLU(gate) * up for gfx950
// past one 16-row tile per expert, and for the K that the stream kernel leaves.
//
// The stream kernel takes one tile per unit, so an expert with 17 rows reads
// and widens its weights twice; next to the bytes of the weights it is the
// widening (int4 -> bf16 x scale, 17 VALU operations per 8 weights) that bounds
// these products.  Here an item is up to 32 tokens of an expert by 128 gate and
// 128 up rows over all of K: each widened fragment feeds both tiles' MFMAs, the
// tokens of a stage are shared by the work-group through LDS, and there is no
// cross-wave sum.  4 waves of 2 x 16 gate and up rows each: 8 waves of one block
// read the tokens from LDS twice as often (N = 4096, K = 7168, 512 tokens of 384
// experts 1527 -> 1419 us).  Three stages of 128 K, so that two work-groups share
// a CU and one widens while the other waits at its barrier.
//
// One-tile kernels -> this kernel (us), tiled weights, 8 experts a token:
//   384 experts, N = 512, K = 7168:  672 / 1152 / 3840 tokens 201 / 321 / 845 -> 187 / 231 / 601
//   384 experts, N = 4096, K = 7168: 768 / 1152 / 3840 tokens 1754 / 2442 / 6659 -> 1491 / 1672 / 4709
//   64 experts, N = 2048, K = 5120:  64 / 192 tokens 134 / 277 -> 84 / 131
// int4_moe.hpp has the rule.
#include "int4_moe.hpp"
#include "stream_kernel.hpp"

namespace ferret {
namespace i4 {

template <int F>
__global__ __launch_bounds__(kWaves * 64) void int4_moe_kernel(SkinnyArgs a, int span, int tile_slots) {
  extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int N = a.N, K = a.K, nkb = K >> 7;
  const int nb_cnt = N / kItemRows;  // row tiles of an expert

  // The groups of the table: a bit per table row that starts one, and per 64
  // rows the groups before them.
  const int table_rows = min(max(__builtin_amdgcn_readfirstlane(a.ntiles[0]), 0), tile_slots);
  uint64_t* start_bits = reinterpret_cast<uint64_t*>(lds + kBitsOff);
  int* before = reinterpret_cast<int*>(lds + kBeforeOff);
  int* count = reinterpret_cast<int*>(lds + kCountOff);
  if (wave == 0) {
    const int n = walk_groups<kTB>(a.tiles, table_rows, lane, [&](int base, uint64_t firsts, int n_before) {
      if (lane == 0) {
        start_bits[base >> 6] = firsts;
        before[base >> 6] = n_before;
      }
    });
    if (lane >= (table_rows + 63) / 64) before[lane] = 0x7fffffff;  // no group
    if (lane == 0) *count = n;
  }
  __syncthreads();
  const int my_before = before[lane];  // of table rows 64 * lane ..
  const int items = __builtin_amdgcn_readfirstlane(*count) * nb_cnt;

  for (int item = blockIdx.x; item < items; item += gridDim.x) {
    const int grp = item / nb_cnt, nb = item % nb_cnt;
    // The last 64 rows with at most grp groups before them hold the group: its
    // row is their (grp - before)-th set bit.
    const int word = 63 - __clzll((long long)__ballot(my_before <= grp));
    const uint64_t bits = start_bits[word];
    const int nth = grp - __builtin_amdgcn_readlane(my_before, word);
    const bool mine = (bits >> lane & 1) && __popcll(bits & ((1ull << lane) - 1)) == nth;
    const int t0 = word * 64 + __ffsll((long long)__ballot(mine)) - 1;
    const bool two = t0 + 1 < table_rows && !(start_bits[(t0 + 1) >> 6] >> ((t0 + 1) & 63) & 1);
    const int e = __builtin_amdgcn_readfirstlane(a.tiles[3 * t0]);
    int row0[kTB], nrows[kTB], pair[kTB];
#pragma unroll
    for (int b = 0; b < kTB; ++b) {
      const int t = b == 0 || two ? t0 + b : t0;
      row0[b] = __builtin_amdgcn_readfirstlane(a.tiles[3 * t + 1]);
      nrows[b] = b == 0 || two ? __builtin_amdgcn_readfirstlane(a.tiles[3 * t + 2]) : 0;
      pair[b] = a.sorted_pair[row0[b] + max(0, min(r, nrows[b] - 1))];  // of token column r
    }

    // ---- sources of this wave's loads of a stage
    const int gate = nb * (kItemRows / 2) + wave * BW * 16, up = N / 2 + gate;
    const uint8_t* wsrc[2 * BW];
    const uint8_t* ssrc[BW];
    const uint8_t* xsrc[kXLoads];
#pragma unroll
    for (int h = 0; h < 2 * BW; ++h) {
      const int row = (h & 1 ? up : gate) + (h >> 1) * 16;
      const int lr = lane >> 2, c = sw_int4(lr, lane & 3);
      if constexpr (F == kINT4T)
        wsrc[h] = a.w + ((size_t)e * (N >> 4) + (row >> 4)) * (size_t)nkb * 1024 + lr * 64 + c * 16;
      else
        wsrc[h] = a.w + ((size_t)e * N + row + lr) * (size_t)(K / 2) + c * 16;
    }
#pragma unroll
    for (int i = 0; i < BW; ++i) {  // 32 lanes' words: gate rows, then up rows, two groups of 32 K a word
      const size_t srow = (size_t)e * N + (lane < 32 ? gate : up) + i * 16 + (lane >> 1 & 15);
      ssrc[i] = static_cast<const uint8_t*>(a.w_scale) + srow * (size_t)(K >> 4) + (lane & 1) * 4;
    }
#pragma unroll
    for (int i = 0; i < kXLoads; ++i) {
      const int xr = 4 * (wave * kXLoads + i) + (lane >> 4);  // token row of the stage
      const int xb = xr >> 4, xt = max(0, min(xr & 15, nrows[xb] - 1));
      const int xtok = a.sorted_pair[row0[xb] + xt] / a.topk;
      xsrc[i] = a.x + (size_t)xtok * K * 2 + sw_bf16(xr & 15, lane & 15) * 16;
    }
    constexpr size_t wstep = F == kINT4T ? 1024 : 64;
    auto issue = [&](int step) {
      uint8_t* st = lds + (step % kNS) * kStage;
      uint8_t* wv = st + wave * kWaveBytes;
#pragma unroll
      for (int h = 0; h < 2 * BW; ++h) {
        // A K-step of a checkpoint row is half a cache line: the other half is kept.
        if constexpr (F == kINT4T) g2l_16_nt(wsrc[h] + (size_t)step * wstep, wv + h * 1024);
        else g2l_16(wsrc[h] + (size_t)step * wstep, wv + h * 1024);
      }
#pragma unroll
      for (int i = 0; i < BW; ++i) g2l_4(ssrc[i] + (size_t)step * 8, wv + kScaleOff + i * 256);
#pragma unroll
      for (int i = 0; i < kXLoads; ++i)
        g2l_16(xsrc[i] + (size_t)step * 256, st + kXOff + (wave * kXLoads + i) * 1024);
    };

    // K runs in spans, each summed from zero and then added in turn, as the waves
    // of the one-tile kernels do: the results are theirs bit for bit (one chain
    // over all of K differed from the rounded exact sum three times as often).
    f32x4 acc[2 * BW][kTB], sum[2 * BW][kTB];
#pragma unroll
    for (int h = 0; h < 2 * BW; ++h)
#pragma unroll
      for (int b = 0; b < kTB; ++b) acc[h][b] = sum[h][b] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int s = 0; s < kNS - 1; ++s)
      if (s < nkb) issue(s);
    // One loop for groups of two tiles and one for single tiles: with the second
    // tile's MFMAs under a condition instead, 512 tokens lost 4 %.
    auto run = [&](auto tbc) {
      constexpr int TB = decltype(tbc)::value;
      int left = span;
      for (int step = 0; step < nkb; ++step) {
        if (nkb - 1 - step >= kNS - 2) wait_vmcnt<(kNS - 2) * kOps>();
        else wait_vmcnt<0>();
        // Past the barrier every wave's loads of this stage are in, and every
        // wave is past its reads of the stage that issue() overwrites.
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        if (step + kNS - 1 < nkb) issue(step + kNS - 1);
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t* st = lds + (step % kNS) * kStage;
        const uint8_t* wv = st + wave * kWaveBytes;
        u32x4 wq[2 * BW];
        float sc[2 * BW];
#pragma unroll
        for (int h = 0; h < 2 * BW; ++h) {
          wq[h] = *reinterpret_cast<const u32x4*>(wv + h * 1024 + r * 64 + (sw_int4(r, g) << 4));
          sc[h] = bf16_bits_to_f32(*reinterpret_cast<const uint16_t*>(wv + kScaleOff + (h >> 1) * 256 +
                                                                      ((h & 1) * 16 + r) * 8 + g * 2));
        }
        u32x4 xf[TB][4];
#pragma unroll
        for (int b = 0; b < TB; ++b)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            xf[b][j] = *reinterpret_cast<const u32x4*>(st + kXOff + (b * 16 + r) * 256 + (sw_bf16(r, 4 * g + j) << 4));
#pragma unroll
        for (int h = 0; h < 2 * BW; ++h) {
          const Int4Scale s = int4_scale(sc[h]);
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const u32x4 w = dequant_int4x8(wq[h][j], s);
#pragma unroll
            for (int b = 0; b < TB; ++b) acc[h][b] = mfma_bf16_16x16x32(w, xf[b][j], acc[h][b]);
          }
        }
        if (--left == 0 || step + 1 == nkb) {
          left = span;
#pragma unroll
          for (int h = 0; h < 2 * BW; ++h)
#pragma unroll
            for (int b = 0; b < TB; ++b) {
              sum[h][b] += acc[h][b];
              acc[h][b] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        }
      }
    };
    if (two) run(IntC<2>{});
    else run(IntC<1>{});
    // Every wave is past its last reads before the next item's loads overwrite
    // the ring.
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int b = 0; b < kTB; ++b) {
      if (r < nrows[b]) {
#pragma unroll
        for (int i = 0; i < BW; ++i) {
          const f32x4 gt = sum[2 * i][b], u = sum[2 * i + 1][b];
          const u32x2 v = {pack_bf16x2(silu_mul(gt[0], u[0]), silu_mul(gt[1], u[1])),
                           pack_bf16x2(silu_mul(gt[2], u[2]), silu_mul(gt[3], u[3]))};
          *reinterpret_cast<u32x2*>(a.out + (size_t)pair[b] * (N / 2) + gate + i * 16 + 4 * g) = v;
        }
      }
    }
  }
}

template <int F>
static int launch(const SkinnyArgs& a, int span, int max_tiles, int ncu, hipStream_t st) {
  FERRET_HIP_CHECK((set_lds_limit_once<int4_moe_kernel<F>>(kLds)));
  hipLaunchKernelGGL((int4_moe_kernel<F>), dim3(2 * ncu), dim3(kWaves * 64), kLds, st, a, span,
                     max_tiles);
  return (int)hipGetLastError();
}

}  // namespace i4
}  // namespace ferret

// span: K-steps summed from zero before they are added to the whole.
int ferret_int4_moe(const ferret::SkinnyArgs& a, bool tiled, int span, int max_tiles, int ncu, hipStream_t st) {
  using namespace ferret;
  return tiled ? i4::launch<kINT4T>(a, span, max_tiles, ncu, st) : i4::launch<kINT4>(a, span, max_tiles, ncu, st);
}
