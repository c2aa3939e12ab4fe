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
// of Float64 r2c plans 64^3 29.0 -> 27.7 us, 16 x 32 x 64 by single passes 29.2 -> 27.0,
// 256^3 304 -> 299.
template <int BYTES>
__device__ __forceinline__ void touch_args() {
  const auto* k = (const __attribute__((address_space(4))) uint32_t*)
      __builtin_amdgcn_kernarg_segment_ptr();
  uint32_t x = 0;
#pragma unroll
  for (int i = 0; i < BYTES / 4; i += 16) x ^= k[i];
  asm volatile("" ::"s"(x));
}

}  // namespace pfft
