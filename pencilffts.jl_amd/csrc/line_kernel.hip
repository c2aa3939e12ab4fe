// GPU kernels of the line pass.  The file is compiled once per precision
// (PFFT_LINE_REAL, PFFT_LINE_NAME), form (PFFT_LINE_FORM: line_pass.hpp,
// line_bluestein.hpp or line_prime.hpp) and class (PFFT_LINE_CLASS): each
// object holds one kernel with the butterflies of every radix.
#include <hip/hip_runtime.h>

#include <string>

#include "line_prime.hpp"
#include "plan.hpp"
#include "touch_args.hpp"

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

#if PFFT_LINE_FORM == 1
// (float: held to 128 VGPRs, 4 waves per SIMD; it asks for 130)
template <typename R, int CLS>
__global__ __launch_bounds__(line_max_threads(CLS, LF_BLUESTEIN, sizeof(R) == 4),
                             sizeof(R) == 4 ? 4 : 2) void k_line_bs(PassArgs a, LineArgs b) {
  touch_args<sizeof(PassArgs) + sizeof(LineArgs)>();
  extern __shared__ __align__(16) char lds[];
  cpx<R>* W = (cpx<R>*)lds;
  const uint32_t tid = threadIdx.x;
  const LineOp<R> op(a);
  for (int64_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    TileCtx c;
    line_tile(a, b, (uint32_t)tile, c);
    OpLine<R> o = {R(0), R(1)};
    if constexpr (CLS == LC_C2C_OP) {
      if (op.op) o = op.tile(a, b, (uint32_t)tile);
    }
#define PFFT_F(RAD) bs_first<R, CLS, RAD>(a, b, c, op, o, opaque(tid), W)
    PFFT_LINE_RADIX_POW2(b.st[0].rad, PFFT_F)
#undef PFFT_F
    __syncthreads();
    // forward stages 1 .. S-2, the middle one, backward S-2 .. 1
    for (int i = 1; i < 2 * b.S - 2; ++i) {
      const int s = i < b.S ? i : 2 * b.S - 2 - i;
      const int dir = i < b.S - 1 ? 0 : i == b.S - 1 ? 1 : 2;
#define PFFT_F(RAD) bs_stage<R, RAD>(a, b, c, s, dir, opaque(tid), W)
      PFFT_LINE_RADIX_POW2(b.st[s].rad, PFFT_F)
#undef PFFT_F
      __syncthreads();
    }
#define PFFT_F(RAD) bs_last<R, CLS, RAD>(a, b, c, op, o, opaque(tid), W)
    PFFT_LINE_RADIX_POW2(b.st[0].rad, PFFT_F)
#undef PFFT_F
    if constexpr (!line_direct(CLS)) {
      __syncthreads();
      line_post<R, CLS>(a, b, c, tid, lds);
    }
    __syncthreads();
  }
}
#define PFFT_LINE_KERNEL k_line_bs<PFFT_LINE_REAL, PFFT_LINE_CLASS>
#elif PFFT_LINE_FORM == 2
template <typename R, int CLS>
__global__ __launch_bounds__(kLineMaxThreads) void k_line_prime(PassArgs a, LineArgs b) {
  touch_args<sizeof(PassArgs) + sizeof(LineArgs)>();
  extern __shared__ __align__(16) char lds[];
  cpx<R>* W = (cpx<R>*)lds;
  const uint32_t tid = threadIdx.x;
  const LineOp<R> op(a);
  for (int64_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    TileCtx c;
    line_tile(a, b, (uint32_t)tile, c);
    OpLine<R> o = {R(0), R(1)};
    if constexpr (CLS == LC_C2C_OP) {
      if (op.op) o = op.tile(a, b, (uint32_t)tile);
    }
    prime_load<R, CLS>(a, b, c, op, o, tid, W);
    __syncthreads();
    for (int s = 0; s < b.S; ++s) {
      const bool fin = s == b.S - 1;
      if (b.st[s].rad > 16) {
        PrimeRegs<R> v;
        prime_get<R>(b, c, s, tid, v, W);
        __syncthreads();
        prime_put<R>(a, b, c, s, fin, tid, v, W);
      } else {
        cpx<R> v[kLinePoints];
#define PFFT_F(RAD)                                       \
  line_get<R, kLinePoints, RAD>(b, c, s, false, opaque(tid), v, W);    \
  __syncthreads();                                        \
  line_put<R, kLinePoints, RAD>(a, b, c, s, false, fin, opaque(tid), v, W)
        PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
      }
      __syncthreads();
    }
    if constexpr (line_direct(CLS)) prime_save<R, CLS>(a, b, c, op, o, tid, W);
    else line_post<R, CLS>(a, b, c, tid, lds);
    __syncthreads();
  }
}
#define PFFT_LINE_KERNEL k_line_prime<PFFT_LINE_REAL, PFFT_LINE_CLASS>
#else
template <typename R, int CLS, int PTS>
__global__ __launch_bounds__(kLineMaxThreads) void k_line(PassArgs a, LineArgs b) {
  touch_args<sizeof(PassArgs) + sizeof(LineArgs)>();
  extern __shared__ __align__(16) char lds[];
  cpx<R>* W = (cpx<R>*)lds;
  const uint32_t tid = threadIdx.x;
  constexpr bool direct = line_direct(CLS);
  const LineOp<R> op(a);
  for (int64_t tile = blockIdx.x; tile < a.ntiles; tile += gridDim.x) {
    TileCtx c;
    line_tile(a, b, (uint32_t)tile, c);
    OpLine<R> o = {R(0), R(1)};
    if constexpr (CLS == LC_C2C_OP) {
      if (op.op) o = op.tile(a, b, (uint32_t)tile);
    }
    cpx<R> v[kLinePoints];
    // stage s leaves its butterflies in LDS, or (fin, direct) in memory
    const bool one = b.S == 1;
#define PFFT_F(RAD)                                                          \
  line_first<R, CLS, PTS, RAD>(a, b, c, op, o, opaque(tid), v);                     \
  if (direct && one) line_store<R, CLS, PTS, RAD>(a, b, c, op, o, opaque(tid), v);  \
  else line_put<R, PTS, RAD>(a, b, c, 0, b.jf_in, one, opaque(tid), v, W)
    PFFT_LINE_RADIX(b.st[0].rad, PFFT_F)
#undef PFFT_F
    for (int s = 1; s < b.S; ++s) {
      const bool fin = s == b.S - 1;
      __syncthreads();
#define PFFT_F(RAD)                                                          \
  line_get<R, PTS, RAD>(b, c, s, direct && fin && b.jf_out, opaque(tid), v, W);   \
  if (direct && fin) {                                                       \
    line_store<R, CLS, PTS, RAD>(a, b, c, op, o, opaque(tid), v);                 \
  } else {                                                                   \
    __syncthreads();                                                         \
    line_put<R, PTS, RAD>(a, b, c, s, false, fin, opaque(tid), v, W);                    \
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

#define PFFT_LINE_KERNEL \
  k_line<PFFT_LINE_REAL, PFFT_LINE_CLASS, PFFT_LINE_FORM == LF_SMALL ? 1 : kLinePoints>
#endif

int PFFT_CAT3(line_prepare_, PFFT_LINE_NAME, PFFT_LINE_CLASS)(const PassPlan& pp) {
  if (pp.lds_bytes <= 64 * 1024) return PFFT_OK;
  const hipError_t e =
      hipFuncSetAttribute((const void*)PFFT_LINE_KERNEL,
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)pp.lds_bytes);
  if (e != hipSuccess)
    return fail(PFFT_ERR_DEVICE, std::string("hipFuncSetAttribute: ") + hipGetErrorString(e));
  return PFFT_OK;
}

void PFFT_CAT3(line_launch_, PFFT_LINE_NAME, PFFT_LINE_CLASS)(const PassPlan& pp,
                                                              const PassArgs& a,
                                                              const LineArgs& b, hipStream_t st) {
  hipLaunchKernelGGL((PFFT_LINE_KERNEL),
                     dim3((unsigned)pp.grid), dim3(b.threads), (size_t)pp.lds_bytes, st, a, b);
}

}  // namespace pfft
