// Host emulator of the generic pass, for the CPU test-suite only.
//
// Runs the exact phase functions of generic_pass.hpp that the GPU kernel runs
// (same pass descriptors, same twiddle tables rounded to the plan precision),
// with the workgroup's threads executed one after another between barriers.
// It is built into its own library (libpencilffts_emu.so) that only tests
// load; the product library has no host execution path.
#include <string.h>

#include <string>
#include <vector>

#include "../../include/pfft.h"
#include "generic_pass.hpp"
#include "line_prime.hpp"
#include "plane_pass.hpp"
#include "plan.hpp"

using namespace pfft;

struct pfft_emu_plan {
  Plan p;
  int32_t tile_order = 0, tile_rev = 0;   // tile traversal (tile_split)
};

template <typename R>
static void emu_pass(const PassPlan& pp, const PassArgs& a) {
  std::vector<char> lds((size_t)pp.lds_bytes);  // exact size: overruns show under ASan
  const int nthr = pp.threads;
  for (int64_t tile = 0; tile < a.ntiles; ++tile) {
    TileCtx c;
    tile_init(a, tile, c);
    for (int t = 0; t < nthr; ++t) phase_load<R>(a, c, t, nthr, lds.data());
    for (int t = 0; t < nthr; ++t) phase_pre<R>(a, c, t, nthr, lds.data());
    for (int s = 0; s < a.nstages; ++s)
      for (int t = 0; t < nthr; ++t) phase_stage<R>(a, c, s, t, nthr, lds.data());
    for (int t = 0; t < nthr; ++t) phase_post<R>(a, c, t, nthr, lds.data());
  }
}

// The line pass: every thread's registers live across the barriers.
template <typename R, int CLS, int PTS>
static void emu_line(const PassPlan& pp, const PassArgs& a, const LineArgs& b) {
  const int nthr = (int)b.threads;
  std::vector<char> store((size_t)pp.lds_bytes + 16);
  char* lds = store.data() + (16 - (size_t)store.data() % 16) % 16;
  cpx<R>* W = (cpx<R>*)lds;
  std::vector<cpx<R>> regs((size_t)nthr * kLinePoints);
  const bool direct = line_direct(CLS);
  const LineOp<R> op(a);
  for (int64_t tile = 0; tile < a.ntiles; ++tile) {
    TileCtx c;
    line_tile(a, b, (uint32_t)tile, c);
    const OpLine<R> o = a.op ? op.tile(a, b, (uint32_t)tile) : OpLine<R>{R(0), R(1)};
    for (int s = 0; s < b.S; ++s) {
      const bool fin = s == b.S - 1;
      for (int t = 0; t < nthr; ++t) {
        cpx<R>* v = &regs[(size_t)t * kLinePoints];
        if (s == 0) {
#define PFFT_F(RAD) line_first<R, CLS, PTS, RAD>(a, b, c, op, o, t, v)
          PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
        } else {
#define PFFT_F(RAD) line_get<R, PTS, RAD>(b, c, s, fin && direct && b.jf_out, t, v, W)
          PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
        }
      }
      for (int t = 0; t < nthr; ++t) {
        cpx<R>* v = &regs[(size_t)t * kLinePoints];
        if (fin && direct) {
#define PFFT_F(RAD) line_store<R, CLS, PTS, RAD>(a, b, c, op, o, t, v)
          PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
        } else {
#define PFFT_F(RAD) line_put<R, PTS, RAD>(a, b, c, s, s == 0 && b.jf_in, fin, t, v, W)
          PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
        }
      }
    }
    if (!direct)
      for (int t = 0; t < nthr; ++t) line_post<R, CLS>(a, b, c, t, lds);
  }
}

template <typename R, int CLS>
static void emu_line_bs(const PassPlan& pp, const PassArgs& a, const LineArgs& b) {
  const int nthr = (int)b.threads;
  std::vector<char> store((size_t)pp.lds_bytes + 16);
  char* lds = store.data() + (16 - (size_t)store.data() % 16) % 16;
  cpx<R>* W = (cpx<R>*)lds;
  const LineOp<R> op(a);
  for (int64_t tile = 0; tile < a.ntiles; ++tile) {
    TileCtx c;
    line_tile(a, b, (uint32_t)tile, c);
    const OpLine<R> o = a.op ? op.tile(a, b, (uint32_t)tile) : OpLine<R>{R(0), R(1)};
    for (int t = 0; t < nthr; ++t) {
#define PFFT_F(RAD) bs_first<R, CLS, RAD>(a, b, c, op, o, t, W)
      PFFT_LINE_RADIX_POW2(b.st[0].rad, PFFT_F)
#undef PFFT_F
    }
    for (int i = 1; i < 2 * b.S - 2; ++i) {
      const int s = i < b.S ? i : 2 * b.S - 2 - i;
      const int dir = i < b.S - 1 ? 0 : i == b.S - 1 ? 1 : 2;
      for (int t = 0; t < nthr; ++t) {
#define PFFT_F(RAD) bs_stage<R, RAD>(a, b, c, s, dir, t, W)
        PFFT_LINE_RADIX_POW2(b.st[s].rad, PFFT_F)
#undef PFFT_F
      }
    }
    for (int t = 0; t < nthr; ++t) {
#define PFFT_F(RAD) bs_last<R, CLS, RAD>(a, b, c, op, o, t, W)
      PFFT_LINE_RADIX_POW2(b.st[0].rad, PFFT_F)
#undef PFFT_F
    }
    if (!line_direct(CLS))
      for (int t = 0; t < nthr; ++t) line_post<R, CLS>(a, b, c, t, lds);
  }
}

template <typename R, int CLS>
static void emu_line_prime(const PassPlan& pp, const PassArgs& a, const LineArgs& b) {
  const int nthr = (int)b.threads;
  std::vector<char> store((size_t)pp.lds_bytes + 16);
  char* lds = store.data() + (16 - (size_t)store.data() % 16) % 16;
  cpx<R>* W = (cpx<R>*)lds;
  std::vector<cpx<R>> regs((size_t)nthr * kLinePoints);
  std::vector<PrimeRegs<R>> pregs((size_t)nthr);
  const LineOp<R> op(a);
  for (int64_t tile = 0; tile < a.ntiles; ++tile) {
    TileCtx c;
    line_tile(a, b, (uint32_t)tile, c);
    const OpLine<R> o = a.op ? op.tile(a, b, (uint32_t)tile) : OpLine<R>{R(0), R(1)};
    for (int t = 0; t < nthr; ++t) prime_load<R, CLS>(a, b, c, op, o, t, W);
    for (int s = 0; s < b.S; ++s) {
      const bool fin = s == b.S - 1;
      if (b.st[s].rad > 16) {
        for (int t = 0; t < nthr; ++t) prime_get<R>(b, c, s, t, pregs[t], W);
        for (int t = 0; t < nthr; ++t) prime_put<R>(a, b, c, s, fin, t, pregs[t], W);
        continue;
      }
      for (int t = 0; t < nthr; ++t) {
        cpx<R>* v = &regs[(size_t)t * kLinePoints];
#define PFFT_F(RAD) line_get<R, kLinePoints, RAD>(b, c, s, false, t, v, W)
        PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
      }
      for (int t = 0; t < nthr; ++t) {
        cpx<R>* v = &regs[(size_t)t * kLinePoints];
#define PFFT_F(RAD) line_put<R, kLinePoints, RAD>(a, b, c, s, false, fin, t, v, W)
        PFFT_LINE_RADIX(b.st[s].rad, PFFT_F)
#undef PFFT_F
      }
    }
    for (int t = 0; t < nthr; ++t) {
      if constexpr (line_direct(CLS)) prime_save<R, CLS>(a, b, c, op, o, t, W);
      else line_post<R, CLS>(a, b, c, t, lds);
    }
  }
}

template <typename R, int CLS>
static void emu_form(const PassPlan& pp, const PassArgs& a, const LineArgs& b) {
  if (b.form == LF_BLUESTEIN) emu_line_bs<R, CLS>(pp, a, b);
  else if (b.form == LF_PRIME) emu_line_prime<R, CLS>(pp, a, b);
  else if constexpr (CLS != LC_R2R) {
    if (b.form == LF_SMALL) emu_line<R, CLS, 1>(pp, a, b);
    else emu_line<R, CLS, kLinePoints>(pp, a, b);
  }
}

template <typename R, int CLS, bool FWD>
static void emu_plane(const PassPlan& pp, const PassArgs& a, const PlaneArgs& p) {
  const int nthr = (int)p.threads;
  std::vector<char> store((size_t)pp.lds_bytes + 16);
  char* lds = store.data() + (16 - (size_t)store.data() % 16) % 16;
  cpx<R>* W = (cpx<R>*)lds;
  std::vector<cpx<R>> regs((size_t)nthr * kLinePoints);
  auto v = [&](int t) { return &regs[(size_t)t * kLinePoints]; };
  const PlaneDim& d0 = FWD ? p.x : p.y;
  const PlaneDim& d1 = FWD ? p.y : p.x;
  for (int64_t tile = 0; tile < a.ntiles; ++tile) {
    TileCtx c;
    plane_tile(a, p, (uint32_t)tile, c);
    for (int s = 0; s < d0.S; ++s) {
      for (int t = 0; t < nthr; ++t) {
        if (s == 0) {
#define PFFT_F(RAD) plane_load<R, CLS, FWD, RAD>(a, p, c, t, v(t))
          PFFT_LINE_RADIX(d0.st[s].rad, PFFT_F)
#undef PFFT_F
        } else {
#define PFFT_F(RAD) plane_get<R, !FWD, RAD>(p, d0, s, t, v(t), W)
          PFFT_LINE_RADIX(d0.st[s].rad, PFFT_F)
#undef PFFT_F
        }
      }
      for (int t = 0; t < nthr; ++t) {
#define PFFT_F(RAD) plane_put<R, !FWD, RAD>(p, d0, s, t, v(t), W)
        PFFT_LINE_RADIX(d0.st[s].rad, PFFT_F)
#undef PFFT_F
      }
    }
    if (plane_has_middle(CLS))
      for (int t = 0; t < nthr; ++t) plane_middle<R, CLS>(a, p, t, W);
    for (int s = 0; s < d1.S; ++s) {
      for (int t = 0; t < nthr; ++t) {
#define PFFT_F(RAD) plane_get<R, FWD, RAD>(p, d1, s, t, v(t), W)
        PFFT_LINE_RADIX(d1.st[s].rad, PFFT_F)
#undef PFFT_F
      }
      for (int t = 0; t < nthr; ++t) {
        if (s == d1.S - 1) {
#define PFFT_F(RAD) plane_store<R, CLS, FWD, RAD>(a, p, c, t, v(t))
          PFFT_LINE_RADIX(d1.st[s].rad, PFFT_F)
#undef PFFT_F
        } else {
#define PFFT_F(RAD) plane_put<R, FWD, RAD>(p, d1, s, t, v(t), W)
          PFFT_LINE_RADIX(d1.st[s].rad, PFFT_F)
#undef PFFT_F
        }
      }
    }
  }
}

template <typename R>
static void emu_any(const Plan& p, const PassPlan& pp, const PassArgs& a) {
  if (pp.plane.on) {
    PlaneArgs q = pp.plane;
    q.tw = table_at(p, pp.line_tw_id, true);
    switch (q.cls) {
      case LC_R2C: emu_plane<R, LC_R2C, true>(pp, a, q); break;
      case LC_R2C_ODD: emu_plane<R, LC_R2C_ODD, true>(pp, a, q); break;
      case LC_C2R: emu_plane<R, LC_C2R, false>(pp, a, q); break;
      case LC_C2R_ODD: emu_plane<R, LC_C2R_ODD, false>(pp, a, q); break;
      default:
        if (q.fwd) emu_plane<R, LC_C2C, true>(pp, a, q);
        else emu_plane<R, LC_C2C, false>(pp, a, q);
    }
    return;
  }
  if (!pp.line.S) {
    emu_pass<R>(pp, a);
    return;
  }
  LineArgs b = pp.line;
  b.tw = table_at(p, pp.line_tw_id, true);
  switch (b.cls == LC_C2C && (a.op || a.fs_M) ? (int)LC_C2C_OP : b.cls) {
    case LC_C2C: emu_form<R, LC_C2C>(pp, a, b); break;
    case LC_R2C: emu_form<R, LC_R2C>(pp, a, b); break;
    case LC_C2R: emu_form<R, LC_C2R>(pp, a, b); break;
    case LC_R2C_ODD: emu_form<R, LC_R2C_ODD>(pp, a, b); break;
    case LC_C2R_ODD: emu_form<R, LC_C2R_ODD>(pp, a, b); break;
    case LC_R2R: emu_form<R, LC_R2R>(pp, a, b); break;
    default: emu_form<R, LC_C2C_OP>(pp, a, b); break;
  }
}

extern "C" {

__attribute__((visibility("default"))) int pfft_emu_plan_create(
    pfft_emu_plan** out, int32_t ndims, const int64_t* dims, const int32_t* kinds,
    int32_t real_type, int32_t permute, int32_t n_extra, const int64_t* extra, uint32_t flags) {
  *out = nullptr;
  pfft_emu_plan* h = new pfft_emu_plan();
  // bit 31 lets plans fuse their first two dims (the emulator's plans are
  // otherwise chains of single passes)
  const uint32_t fl = flags >> 31 ? flags & 0x7fffffffu : flags | PFFT_FLAG_GENERIC_ONLY;
  int r = plan_build(h->p, ndims, dims, kinds, real_type, permute, n_extra, extra, fl);
  if (r) {
    delete h;
    return r;
  }
  *out = h;
  return PFFT_OK;
}

__attribute__((visibility("default"))) int pfft_emu_plan_destroy(pfft_emu_plan* h) {
  delete h;
  return PFFT_OK;
}

__attribute__((visibility("default"))) const char* pfft_emu_last_error(void) {
  return last_error();
}

__attribute__((visibility("default"))) int pfft_emu_nbytes(const pfft_emu_plan* h,
                                                          size_t* in_b, size_t* out_b) {
  *in_b = h->p.in_bytes;
  *out_b = h->p.out_bytes;
  return PFFT_OK;
}

// Host buffers in the same layouts as pfft_execute's device buffers; op as
// in pfft_execute_op (null: none).
__attribute__((visibility("default"))) int pfft_emu_execute_op(pfft_emu_plan* h, int32_t dir,
                                                              const pfft_spectral_op* op,
                                                              const void* in, void* out) {
  Plan& p = h->p;
  int op_pass = -1, op_side = 0;
  if (op && op->op) {
    const int r0 = op_setup(p, dir, *op, &op_pass, &op_side);
    if (r0) return r0;
  }
  if (dir < PFFT_FORWARD || dir > PFFT_ADJOINT_BACKWARD)
    return fail(PFFT_ERR_ARGUMENT, "unknown direction");
  if ((dir == PFFT_ADJOINT_FORWARD || dir == PFFT_ADJOINT_BACKWARD) && !p.adjoint_ok)
    return fail(PFFT_ERR_UNSUPPORTED, "no adjoint for R2R plans");
  const bool fwd_shape = dir == PFFT_FORWARD || dir == PFFT_ADJOINT_BACKWARD;
  if (p.inplace && in != out)
    return fail(PFFT_ERR_ARGUMENT, "input and output arrays for in-place plan must be the same");
  // the two work buffers as separate exact-size allocations
  std::vector<char> work0(p.work0_bytes), work1(p.work_bytes - p.work0_bytes);
  const std::vector<PassPlan>& passes = fwd_shape ? p.fwd : p.bwd;
  void* bufs[3] = {nullptr, work0.data(), work1.data()};
  const int np = (int)passes.size();
  for (int i = 0; i < np; ++i) {
    const PassPlan& pp = passes[i];
    PassArgs a = pp.args;
    a.in = pp.src == 0 ? in : bufs[pp.src];
    a.out = pp.dst == 0 ? out : bufs[pp.dst];
    bind_tables(p, pp, a, true);
    if (dir == PFFT_BACKWARD_SCALED && i == np - 1) {
      a.do_scale = 1;
      a.scale = 1.0 / p.scale;
    }
    a.adjoint = (dir == PFFT_ADJOINT_FORWARD || dir == PFFT_ADJOINT_BACKWARD) ? 1 : 0;
    a.tile_order = h->tile_order;
    a.tile_rev = h->tile_rev;
    if (i == op_pass) op_fill(p, dir, *op, op_side, a);
    if (p.real_type == PFFT_F32) emu_any<float>(p, pp, a);
    else emu_any<double>(p, pp, a);
  }
  return PFFT_OK;
}

// Tile traversal of every pass (the specialised kernels' tuned tile order and
// direction), to check on the host that each order covers every line once.
__attribute__((visibility("default"))) int pfft_emu_set_traversal(pfft_emu_plan* h,
                                                                 int32_t order, int32_t rev) {
  h->tile_order = order ? 1 : 0;
  h->tile_rev = rev ? 1 : 0;
  return PFFT_OK;
}

// Convolution length of the Bluestein form of each forward pass (0: direct
// stages); returns the number of passes.
__attribute__((visibility("default"))) int pfft_emu_bluestein(pfft_emu_plan* h, int64_t* out,
                                                             int32_t n) {
  const int np = (int)h->p.fwd.size();
  for (int i = 0; i < np && i < n; ++i) out[i] = h->p.fwd[i].args.bs_M;
  return np;
}

__attribute__((visibility("default"))) int pfft_emu_execute(pfft_emu_plan* h, int32_t dir,
                                                           const void* in, void* out) {
  return pfft_emu_execute_op(h, dir, nullptr, in, out);
}

}  // extern "C"
