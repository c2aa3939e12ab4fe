// Plane pass: the first two dims of a 3D transform in one launch.
//
// One workgroup holds one x-y plane in LDS: x lines (complex FFT, r2c or c2r,
// even or odd) and y lines (complex FFT), both of 13-smooth length.  Forward it
// loads the plane straight into the x lines' first butterflies, splits the r2c
// in LDS, and stores from the y lines' last butterflies; backward the other way
// round.  Planes are contiguous in memory on both sides, so the order between
// this pass and the one along z is the natural one and no transposition is
// needed.
//
// It is for arrays whose time is that of the launches (4 to 5 us each on the
// device, 3.5 us of the host's): one launch of three and one trip through memory
// less.  What bounds it: latency, of the launch, of one load of the plane and of two
// barriers a stage, with as many CUs at work as there are planes.  Measured, pairs
// of Float64 r2c plans called one by one (single passes -> plane pass): 16 x 32 x 64 27.0 -> 21.7 us, 28 x 28 x 12
// 29.2 -> 22.2, 105 planes of 112 x 65 59.3 -> 50.6 (the rule, with both sides: plane_fits
// in plan.cpp).
//
// A row of the plane is a line's points with the odd pitch and the padding of the
// line pass, so that neighbouring threads take neighbouring points of a row, along x
// lines and across y lines, on neighbouring banks.
//
// Phases as functions of (thread id, the thread's registers, LDS), shared with the
// host emulator of the CPU test-suite.
#pragma once

#include "line_pass.hpp"

namespace pfft {

// workgroup (double: 512, so that 16 points a thread stay in registers)
constexpr int plane_max_threads(bool f32) { return f32 ? 1024 : 512; }

// LDS slot of point k of line w: x lines are rows, y lines (COL) columns
template <bool COL>
PFFT_HD uint32_t plane_at(const PlaneArgs& p, uint32_t w, uint32_t k) {
  return COL ? k * p.pitch + wp(w, p.sh) : w * p.pitch + wp(k, p.sh);
}

// Butterfly e of a stage: line w, index j.  Neighbouring threads run along the
// row, and across the columns: x is contiguous in memory and in LDS.
template <bool COL>
PFFT_HD bool plane_slot(const PlaneDim& d, const LineStage& st, uint32_t e, uint32_t* w,
                        uint32_t* j) {
  bool act;
  if (COL) {
    *j = line_div(e, d.m_lines);
    *w = e - *j * d.lines;
    act = *j < st.nb;
  } else {
    *w = line_div(e, st.m_nb);
    *j = e - *w * st.nb;
    act = *w < d.lines;
  }
  if (!act) *w = *j = 0;
  return act;
}

// the i-th butterflies of the workgroup are all past the plane
PFFT_HD bool plane_idle(const PlaneArgs& p, const PlaneDim& d, const LineStage& st, int i) {
  return i > 0 && i * p.threads >= d.lines * st.nb;
}

PFFT_HD void plane_tile(const PassArgs& a, const PlaneArgs& p, uint32_t tile, TileCtx& c) {
  int64_t ib = 0, ob = 0;
  uint32_t rest = tile;
  for (int d = 0; d < a.D; ++d) {
    const uint32_t q = d + 1 < a.D ? line_div64(rest, p.m_dim[d]) : 0;
    const int64_t m = rest - q * (uint32_t)a.ldim[d];
    rest = q;
    ib += m * a.lsin[d];
    ob += m * a.lsout[d];
  }
  c.in_base = ib;
  c.out_base = ob;
}

// ---- memory -> first butterflies of the first dim ------------------------------------
template <typename R, int CLS, bool FWD, int RAD>
PFFT_HD void plane_load(const PassArgs& a, const PlaneArgs& p, const TileCtx& c, uint32_t tid,
                        cpx<R>* v) {
  constexpr int BPT = line_bpt(RAD);
  constexpr bool real = FWD && (CLS == LC_R2C || CLS == LC_R2C_ODD);
  constexpr int pair = FWD && CLS == LC_R2C ? 2 : 1;
  const PlaneDim& d = FWD ? p.x : p.y;
  const LineStage& st = d.st[0];
  constexpr uint32_t esz = real ? sizeof(R) : sizeof(cpx<R>);
  const uint32_t sk = (uint32_t)(FWD ? p.sx_in : p.sy_in), ls = (uint32_t)(FWD ? p.sy_in : p.sx_in);
  const char* base = (const char*)a.in + c.in_base * (int64_t)esz;
  const uint64_t step = opaque_s((uint64_t)st.nb * sk * esz * pair);
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    if (plane_idle(p, d, st, i)) break;
    uint32_t w, j;
    plane_slot<!FWD>(d, st, tid + i * p.threads, &w, &j);
    const uint32_t off = (w * ls + j * sk * pair) * esz;
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      // (x is contiguous: an r2c's real pairs are one load)
      if constexpr (real && pair == 1) v[i * RAD + r] = mk(*(const R*)(base + r * step + off), R(0));
      else v[i * RAD + r] = *(const cpx<R>*)(base + r * step + off);
    }
  }
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    if (plane_idle(p, d, st, i)) break;
    if (d.bwd) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) v[i * RAD + r] = conj(v[i * RAD + r]);
    }
    dft<R, RAD>(v + i * RAD);
  }
}

// ---- LDS -> registers, twiddles, butterflies of stage s --------------------------------
template <typename R, bool COL, int RAD>
PFFT_HD void plane_get(const PlaneArgs& p, const PlaneDim& d, int s, uint32_t tid, cpx<R>* v,
                       const cpx<R>* W) {
  constexpr int BPT = line_bpt(RAD);
  const LineStage& st = d.st[s];
  const cpx<R>* tw = (const cpx<R>*)p.tw + st.tw;
  const bool cj = s == 0 && d.bwd;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    if (plane_idle(p, d, st, i)) break;
    uint32_t w, j;
    plane_slot<COL>(d, st, tid + i * p.threads, &w, &j);
    const uint32_t jj = j - line_div(j, st.m_ns) * st.ns;
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      const cpx<R> z = lds_get(&W[plane_at<COL>(p, w, j + r * st.nb)]);
      v[i * RAD + r] = cj ? conj(z) : z;
    }
    if (s > 0) {
#pragma unroll
      for (int r = 1; r < RAD; ++r) v[i * RAD + r] = v[i * RAD + r] * tw[(r - 1) * st.ns + jj];
    }
    dft<R, RAD>(v + i * RAD);
  }
}

// ---- registers -> LDS after stage s ---------------------------------------------------
template <typename R, bool COL, int RAD>
PFFT_HD void plane_put(const PlaneArgs& p, const PlaneDim& d, int s, uint32_t tid, const cpx<R>* v,
                       cpx<R>* W) {
  constexpr int BPT = line_bpt(RAD);
  const LineStage& st = d.st[s];
  const bool cj = s == d.S - 1 && d.bwd;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    if (plane_idle(p, d, st, i)) break;
    uint32_t w, j;
    if (!plane_slot<COL>(d, st, tid + i * p.threads, &w, &j)) continue;
    const uint32_t jq = line_div(j, st.m_ns), jj = j - jq * st.ns;
    const uint32_t k = jq * st.ns * RAD + jj;
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      const cpx<R> z = v[i * RAD + r];
      lds_put(&W[plane_at<COL>(p, w, k + r * st.ns)], cj ? conj(z) : z);
    }
  }
}

// ---- last butterflies of the second dim -> memory -------------------------------------
template <typename R, int CLS, bool FWD, int RAD>
PFFT_HD void plane_store(const PassArgs& a, const PlaneArgs& p, const TileCtx& c, uint32_t tid,
                         const cpx<R>* v) {
  constexpr int BPT = line_bpt(RAD);
  constexpr bool real = !FWD && (CLS == LC_C2R || CLS == LC_C2R_ODD);
  constexpr int pair = !FWD && CLS == LC_C2R ? 2 : 1;
  const PlaneDim& d = FWD ? p.y : p.x;
  const LineStage& st = d.st[d.S - 1];
  constexpr uint32_t esz = real ? sizeof(R) : sizeof(cpx<R>);
  const uint32_t sk = (uint32_t)(FWD ? p.sy_out : p.sx_out);
  const uint32_t ls = (uint32_t)(FWD ? p.sx_out : p.sy_out);
  char* base = (char*)a.out + c.out_base * (int64_t)esz;
  const uint64_t step = opaque_s((uint64_t)st.nb * sk * esz * pair);
  const R sc = a.do_scale ? (R)a.scale : R(1);
  const R sci = d.bwd ? -sc : sc;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    if (plane_idle(p, d, st, i)) break;
    uint32_t w, j;
    if (!plane_slot<FWD>(d, st, tid + i * p.threads, &w, &j)) continue;
    const uint32_t off = (w * ls + j * sk * pair) * esz;
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      const cpx<R> z = mk(v[i * RAD + r].re * sc, v[i * RAD + r].im * sci);
      if constexpr (real && pair == 1) *(R*)(base + r * step + off) = z.re;
      else *(cpx<R>*)(base + r * step + off) = z;
    }
  }
}

// ---- between the dims: r2c split (odd: the adjoint's weights), c2r merge or extension,
// in place in LDS ----------------------------------------------------------------------
// One work item takes the points k and M - k (n - k) of a row.
template <typename R, int CLS>
PFFT_HD void plane_middle(const PassArgs& a, const PlaneArgs& p, uint32_t tid, cpx<R>* W) {
  const uint32_t M = (uint32_t)a.M, H = M / 2 + 1;
  const cpx<R>* aux = (const cpx<R>*)a.aux;
  const R half = a.adjoint ? R(0.5) : R(1);   // X_k / w_k of the c2r's adjoint
  for (uint32_t e = tid; e < p.x.lines * H; e += p.threads) {
    const uint32_t y = line_div(e, p.m_pairs), k = e - y * H;
    cpx<R>* L = W + y * p.pitch;
    cpx<R>* u = &L[wp(k, p.sh)];
    if constexpr (CLS == LC_R2C) {
      // X_k = E + w_n^k O of Z_k and Z_{M-k}, and X_{M-k} of the same two
      const cpx<R> z = lds_get(u), q = lds_get(&L[wp(k == 0 ? 0 : M - k, p.sh)]);
      auto bin = [&](cpx<R> s, cpx<R> sc, uint32_t kk) {
        const cpx<R> E = scl(s + sc, R(0.5)), O = scl(mul_mi(s - sc), R(0.5));
        const cpx<R> x = E + aux[kk] * O;
        return a.adjoint ? scl(x, R(herm_weight(kk, a.n))) : x;
      };
      lds_put(u, bin(z, conj(q), k));
      if (2 * k != M) lds_put(&L[wp(M - k, p.sh)], bin(q, conj(z), M - k));
    } else if constexpr (CLS == LC_C2R) {
      // Z_k = (X_k + conj X_{M-k}) + i (X_k - conj X_{M-k}) w_n^-k, and Z_{M-k}
      cpx<R>* t = &L[wp(M - k, p.sh)];
      cpx<R> A = lds_get(u), B = lds_get(t);
      if (k == 0) { A.im = R(0); B.im = R(0); }   // Im of DC and Nyquist ignored
      else { A = scl(A, half); B = scl(B, half); }
      auto point = [&](cpx<R> s, cpx<R> q, uint32_t kk) {
        return (s + q) + mul_pi((s - q) * conj(aux[kk]));
      };
      lds_put(u, point(A, conj(B), k));
      if (k != 0 && 2 * k != M) lds_put(t, point(B, conj(A), M - k));
    } else if constexpr (CLS == LC_R2C_ODD) {
      if (a.adjoint && k) lds_put(u, scl(lds_get(u), R(2)));   // w_k X_k
    } else if constexpr (CLS == LC_C2R_ODD) {
      cpx<R> A = lds_get(u);
      if (k == 0) {
        A.im = R(0);   // Im of DC ignored
        lds_put(u, A);
      } else {
        A = scl(A, half);
        lds_put(u, A);
        lds_put(&L[wp(M - k, p.sh)], conj(A));
      }
    }
  }
}
constexpr bool plane_has_middle(int cls) { return cls != LC_C2C; }

}  // namespace pfft
