// GPU kernel of the line pass (line_pass.hpp).  The file is compiled once per
// precision (PFFT_LINE_REAL, PFFT_LINE_NAME) and class (PFFT_LINE_CLASS): each
// object holds one kernel with the butterflies of every radix.
#include <hip/hip_runtime.h>

#include <string>

#include "line_pass.hpp"
#include "plan.hpp"

#define PFFT_CAT3_(a, b, c) a##b##c
#define PFFT_CAT3(a, b, c) PFFT_CAT3_(a, b, c)

namespace pfft {

// A copy of x the compiler knows nothing about: index arithmetic made from
// it stays inside its radix's case.  Shared over the cases, the hoisted
// addresses of all 15 radices raised the c2c kernels from 81 to 165 (float)
// and from 142 to 227 (double) VGPRs.
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

template <typename R, int CLS>
__global__ __launch_bounds__(kLineMaxThreads) void k_line(PassArgs a, LineArgs b) {
  extern __shared__ __align__(16) char lds[];
  cpx<R>* W = (cpx<R>*)lds;
  const uint32_t tid = threadIdx.x;
  constexpr bool direct = line_direct(CLS);
  const LineOp<R> op(a);
  for (int64_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    TileCtx c;
    tile_init(a, tile, c);
    OpLine<R> o = {R(0), R(1)};
    if constexpr (CLS == LC_C2C_OP) {
      int64_t m0;
      if (op.op) o = op_tile<R>(a, tile, &m0);
    }
    cpx<R> v[kLinePoints];
    // stage s leaves its butterflies in LDS, or (fin, direct) in memory
    const bool one = b.S == 1;
#define PFFT_F(RAD)                                                          \
  line_first<R, CLS, RAD>(a, b, c, op, o, opaque(tid), v);                     \
  if (direct && one) line_store<R, CLS, RAD>(a, b, c, op, o, opaque(tid), v);  \
  else line_put<R, RAD>(a, b, c, 0, one, opaque(tid), v, W)
    PFFT_LINE_RADIX(b.st[0].rad, PFFT_F)
#undef PFFT_F
    for (int s = 1; s < b.S; ++s) {
      const bool fin = s == b.S - 1;
      __syncthreads();
#define PFFT_F(RAD)                                                          \
  line_get<R, RAD>(b, c, s, direct && fin && b.jf_out, opaque(tid), v, W);   \
  if (direct && fin) {                                                       \
    line_store<R, CLS, RAD>(a, b, c, op, o, opaque(tid), v);                 \
  } else {                                                                   \
    __syncthreads();                                                         \
    line_put<R, RAD>(a, b, c, s, fin, opaque(tid), v, W);                    \
  }
      PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
    }
    if constexpr (!direct) {
      __syncthreads();
      line_post<R, CLS>(a, b, c, tid, lds);
    }
    __syncthreads();
  }
}

int PFFT_CAT3(line_prepare_, PFFT_LINE_NAME, PFFT_LINE_CLASS)(const PassPlan& pp) {
  if (pp.lds_bytes <= 64 * 1024) return PFFT_OK;
  const hipError_t e =
      hipFuncSetAttribute((const void*)k_line<PFFT_LINE_REAL, PFFT_LINE_CLASS>,
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)pp.lds_bytes);
  if (e != hipSuccess)
    return fail(PFFT_ERR_DEVICE, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
  return PFFT_OK;
}

void PFFT_CAT3(line_launch_, PFFT_LINE_NAME, PFFT_LINE_CLASS)(const PassPlan& pp,
                                                              const PassArgs& a,
                                                              const LineArgs& b, hipStream_t st) {
  hipLaunchKernelGGL((k_line<PFFT_LINE_REAL, PFFT_LINE_CLASS>), dim3((unsigned)pp.grid),
                     dim3(b.threads), (size_t)pp.lds_bytes, st, a, b);
}

}  // namespace pfft
