// GPU kernels of the plane pass (plane_pass.hpp), compiled once per precision
// (PFFT_PLANE_REAL, PFFT_PLANE_NAME).
#include <hip/hip_runtime.h>

#include <string>

#include "plan.hpp"
#include "plane_pass.hpp"
#include "touch_args.hpp"

#define PFFT_CAT_(a, b) a##b
#define PFFT_CAT(a, b) PFFT_CAT_(a, b)

namespace pfft {

__device__ __forceinline__ uint32_t opaque(uint32_t x) {   // (as in line_kernel.hip)
  asm volatile("" : "+v"(x));
  return x;
}

template <typename R, int CLS, bool FWD>
__global__ __launch_bounds__(plane_max_threads(sizeof(R) == 4)) void k_plane(PassArgs a,
                                                                           PlaneArgs p) {
  touch_args<sizeof(PassArgs) + sizeof(PlaneArgs)>();
  extern __shared__ __align__(16) char lds[];
  cpx<R>* W = (cpx<R>*)lds;
  const uint32_t tid = threadIdx.x;
  const PlaneDim& d0 = FWD ? p.x : p.y;
  const PlaneDim& d1 = FWD ? p.y : p.x;
  for (int64_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    TileCtx c;
    plane_tile(a, p, (uint32_t)tile, c);
    cpx<R> v[kLinePoints];
#define PFFT_F(RAD)                                            \
  plane_load<R, CLS, FWD, RAD>(a, p, c, opaque(tid), v);       \
  plane_put<R, !FWD, RAD>(p, d0, 0, opaque(tid), v, W)
    PFFT_LINE_RADIX(d0.st[0].rad, PFFT_F)
#undef PFFT_F
    for (int s = 1; s < d0.S; ++s) {
      __syncthreads();
#define PFFT_F(RAD)                                            \
  plane_get<R, !FWD, RAD>(p, d0, s, opaque(tid), v, W);        \
  __syncthreads();                                             \
  plane_put<R, !FWD, RAD>(p, d0, s, opaque(tid), v, W)
      PFFT_LINE_RADIX(d0.st[s].rad, PFFT_F)
#undef PFFT_F
    }
    __syncthreads();
    if constexpr (plane_has_middle(CLS)) {
      plane_middle<R, CLS>(a, p, tid, W);
      __syncthreads();
    }
    for (int s = 0; s < d1.S; ++s) {
      const bool fin = s == d1.S - 1;
#define PFFT_F(RAD)                                            \
  plane_get<R, FWD, RAD>(p, d1, s, opaque(tid), v, W);         \
  __syncthreads();                                             \
  if (fin) plane_store<R, CLS, FWD, RAD>(a, p, c, opaque(tid), v); \
  else plane_put<R, FWD, RAD>(p, d1, s, opaque(tid), v, W)
      PFFT_LINE_RADIX(d1.st[s].rad, PFFT_F)
#undef PFFT_F
      if (!fin) __syncthreads();
    }
  }
}

namespace {
struct PlaneKernel {
  const void* fn;
  void (*launch)(dim3, dim3, size_t, hipStream_t, const PassArgs&, const PlaneArgs&);
};
template <typename R, int CLS, bool FWD>
PlaneKernel plane_kernel() {
  return {(const void*)k_plane<R, CLS, FWD>,
          [](dim3 g, dim3 t, size_t lds, hipStream_t s, const PassArgs& a, const PlaneArgs& p) {
            hipLaunchKernelGGL((k_plane<R, CLS, FWD>), g, t, lds, s, a, p);
          }};
}
template <typename R>
PlaneKernel kernel_of(const PlaneArgs& p) {
  switch (p.cls) {
    case LC_R2C: return plane_kernel<R, LC_R2C, true>();
    case LC_R2C_ODD: return plane_kernel<R, LC_R2C_ODD, true>();
    case LC_C2R: return plane_kernel<R, LC_C2R, false>();
    case LC_C2R_ODD: return plane_kernel<R, LC_C2R_ODD, false>();
    default:
      return p.fwd ? plane_kernel<R, LC_C2C, true>() : plane_kernel<R, LC_C2C, false>();
  }
}
}  // namespace

int PFFT_CAT(plane_prepare_, PFFT_PLANE_NAME)(const PassPlan& pp) {
  if (pp.lds_bytes <= 64 * 1024) return PFFT_OK;
  const hipError_t e =
      hipFuncSetAttribute(kernel_of<PFFT_PLANE_REAL>(pp.plane).fn,
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)pp.lds_bytes);
  if (e != hipSuccess)
    return fail(PFFT_ERR_DEVICE, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
  return PFFT_OK;
}

void PFFT_CAT(plane_launch_, PFFT_PLANE_NAME)(const PassPlan& pp, const PassArgs& a,
                                              const PlaneArgs& p, hipStream_t st) {
  kernel_of<PFFT_PLANE_REAL>(p).launch(dim3((unsigned)pp.grid), dim3(p.threads),
                                       (size_t)pp.lds_bytes, st, a, p);
}

}  // namespace pfft
