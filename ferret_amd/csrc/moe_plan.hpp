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
// kernel's otherwise; that one loads weights through registers, this one copies
// them to LDS 16 bytes at a time, so tensors off that bound stay there.
inline bool w2_streams(int nkb, const void* w) {
  if (w2_four_waves(nkb)) return true;
  return (nkb == 12 || nkb == 4 || nkb == 6 || nkb == 14) && (reinterpret_cast<uintptr_t>(w) & 15) == 0;
}

}  // namespace moe
}  // namespace ferret
