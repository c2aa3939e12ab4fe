// Kernel arguments are written by the host just before a launch, and read where
// they are first needed they miss the scalar cache one line after the other.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace pfft {

// Touches every 64-byte line of the first BYTES of a kernel's arguments at once.
// Measured on the line pass: the first global load of a pass left 1.8 us after
// the wavefront started, half the time of a pass on a small array (0.9 us with
// this and reciprocals for the tile's divisions).  In the specialised kernels: pairs
// of Float64 r2c plans 64^3 29.0 -> 26.6 us, 16 x 32 x 64 by single passes 29.2 -> 27.0,
// 256^3 304 -> 296.
template <int BYTES>
__device__ __forceinline__ void touch_args() {
  static_assert(BYTES <= 24 * 64, "one word of each 64 bytes");
  const auto* k = (const __attribute__((address_space(4))) uint32_t*)
      __builtin_amdgcn_kernarg_segment_ptr();
  auto word = [&](int line) { return k[line * 64 < BYTES ? line * 16 : 0]; };
  // (one wait for all, and no use: a sum of the words cost the line pass 0.6 to 1.8 %)
  asm volatile("" ::"s"(word(0)), "s"(word(1)), "s"(word(2)), "s"(word(3)), "s"(word(4)),
               "s"(word(5)), "s"(word(6)), "s"(word(7)), "s"(word(8)), "s"(word(9)),
               "s"(word(10)), "s"(word(11)), "s"(word(12)), "s"(word(13)), "s"(word(14)),
               "s"(word(15)), "s"(word(16)), "s"(word(17)), "s"(word(18)), "s"(word(19)),
               "s"(word(20)), "s"(word(21)), "s"(word(22)), "s"(word(23)));
}

}  // namespace pfft
