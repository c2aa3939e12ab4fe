// Line pass for FFT lengths with prime factors of 17 to 61, and for the R2R kinds
// of all lengths without larger ones.
//
// The tile is loaded into LDS, every radix is one trip through it, and the
// outputs are stored from it.  A prime p takes its stage in the symmetric form
//   y_0 = v_0 + sum_r A_r,  y_q, y_{p-q} = P_q -+ i Q_q  (r, q = 1 .. (p-1)/2),
//   P_q = v_0 + sum_r A_r cos(2 pi q r / p),  Q_q = sum_r B_r sin(2 pi q r / p),
//   A_r = v_r + v_{p-r},  B_r = v_r - v_{p-r}:
// a thread keeps P and Q of up to kPrimePairs values of q of one butterfly and
// runs over its p points in LDS once, p - 1 real multiply-adds an output.  The
// q of a wavefront are the same for all its lanes, so the cosines and sines
// come by scalar loads.
//
// What bounds it: arithmetic (60 multiply-adds a point at p = 61) beside the
// LDS trips.  The generic phases computed one output per work item, p complex
// products and p LDS reads each.  The Bluestein form (2 to 2.1 times the points, two
// FFTs) measured slower and less exact at these factors: 306 x 170 x 190
// complex floats 1254 us a pair against 1106 us in the generic phases, its
// largest error 2.2e-6 against 1.2e-6.
// The R2R kinds take this form for its load loop: their gathers, expanded for
// every point of every radix's first butterfly, made kernels that took ten
// minutes to compile, for one trip through LDS less.
#pragma once

#include "line_bluestein.hpp"

namespace pfft {

PFFT_HD uint32_t wave_uniform(uint32_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
  return __builtin_amdgcn_readfirstlane(x);
#else
  return x;
#endif
}

template <typename R>
struct PrimeRegs {
  cpx<R> P[kPrimePairs], Q[kPrimePairs], y0;
};

// Element e of the tile: line w, point k (neighbouring threads along the line,
// jf, or across the lines).
PFFT_HD void line_element(const PassArgs& a, const LineArgs& b, bool jf, uint32_t e, uint32_t* w,
                          uint32_t* k) {
  if (jf) {
    *w = line_div(e, b.m_line);
    *k = e - *w * (uint32_t)a.M;
  } else {
    *w = e & (b.Tw - 1);
    *k = e >> b.twlog;
  }
}

// global memory -> LDS, eight points in flight
template <typename R, int CLS>
PFFT_HD void prime_load(const PassArgs& a, const LineArgs& b, const TileCtx& c,
                        const LineOp<R>& op, const OpLine<R>& otile, uint32_t tid, cpx<R>* W) {
  const uint32_t count = (b.jf_in ? (uint32_t)c.Tw : b.Tw) * (uint32_t)a.M;
  constexpr int U = CLS == LC_R2R ? 4 : 8;
  for (uint32_t e0 = tid; e0 < count; e0 += U * b.threads) {
    cpx<R> z[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
      uint32_t w, k;
      line_element(a, b, b.jf_in != 0, e0 + i * b.threads, &w, &k);
      const bool in = e0 + i * b.threads < count && w < (uint32_t)c.Tw;
      z[i] = line_in<R, CLS>(a, c, op, otile, in ? w : 0, in ? k : 0);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
      uint32_t w, k;
      line_element(a, b, b.jf_in != 0, e0 + i * b.threads, &w, &k);
      if (e0 + i * b.threads < count && w < (uint32_t)c.Tw)
        lds_put(&W[w * b.pitch + wp(k, b.sh)], a.bwd ? conj(z[i]) : z[i]);
    }
  }
}

// LDS -> global memory (kinds without post-processing)
template <typename R, int CLS>
PFFT_HD void prime_save(const PassArgs& a, const LineArgs& b, const TileCtx& c,
                        const LineOp<R>& op, const OpLine<R>& otile, uint32_t tid,
                        const cpx<R>* W) {
  const uint32_t count = (b.jf_out ? (uint32_t)c.Tw : b.Tw) * (uint32_t)a.M;
  for (uint32_t e = tid; e < count; e += b.threads) {
    uint32_t w, k;
    line_element(a, b, b.jf_out != 0, e, &w, &k);
    if (w >= (uint32_t)c.Tw) continue;
    line_out<R, CLS>(a, c, op, otile, w, k, lds_get(&W[w * b.pitch + wp(k, b.sh)]));
  }
}

// The thread's share of a prime stage: chunk (which q, the same for a
// wavefront), line w and butterfly j; false past the tile.
PFFT_HD bool prime_slot(const LineArgs& b, const LineStage& st, const TileCtx& c, uint32_t tid,
                        uint32_t* chunk, uint32_t* w, uint32_t* j) {
  const uint32_t slots = (b.Tw * st.nb + 63) & ~63u;
  uint32_t ch = 0, e = tid;
  while (e >= slots) { e -= slots; ++ch; }
  *chunk = wave_uniform(ch);
  *w = e & (b.Tw - 1);
  *j = e >> b.twlog;
  const bool act = *chunk * kPrimePairs < (st.rad - 1) / 2 && *w < (uint32_t)c.Tw && *j < st.nb;
  if (!act) *w = *j = 0;
  return act;
}

template <typename R>
PFFT_HD void prime_get(const LineArgs& b, const TileCtx& c, int s, uint32_t tid, PrimeRegs<R>& v,
                       const cpx<R>* W) {
  const LineStage& st = b.st[s];
  const uint32_t p = st.rad, H = (p - 1) / 2;
  uint32_t chunk, w, j;
  prime_slot(b, st, c, tid, &chunk, &w, &j);
  const cpx<R>* root = (const cpx<R>*)b.tw + st.tw;   // w_p^m = cos - i sin
  const cpx<R>* tw = root + p + (j - line_div(j, st.m_ns) * st.ns);
  const cpx<R>* L = W + w * b.pitch;
  const cpx<R> v0 = lds_get(&L[wp(j, b.sh)]);
  v.y0 = v0;
  uint32_t q[kPrimePairs], m[kPrimePairs];
#pragma unroll
  for (int i = 0; i < kPrimePairs; ++i) {
    v.P[i] = v0;
    v.Q[i] = mk(R(0), R(0));
    q[i] = chunk * kPrimePairs + 1 + i;
    if (q[i] > H) q[i] = 0;   // no such output: not stored
    m[i] = 0;
  }
  for (uint32_t r = 1; r <= H; ++r) {
    cpx<R> x = lds_get(&L[wp(j + r * st.nb, b.sh)]);
    cpx<R> z = lds_get(&L[wp(j + (p - r) * st.nb, b.sh)]);
    if (s > 0) {
      x = x * tw[(r - 1) * st.ns];
      z = z * tw[(p - r - 1) * st.ns];
    }
    const cpx<R> A = x + z, B = x - z;
    v.y0 = v.y0 + A;
#pragma unroll
    for (int i = 0; i < kPrimePairs; ++i) {
      m[i] += q[i];
      if (m[i] >= p) m[i] -= p;
      const cpx<R> f = root[m[i]];
      v.P[i] = v.P[i] + scl(A, f.re);
      v.Q[i] = v.Q[i] + scl(B, -f.im);
    }
  }
}

template <typename R>
PFFT_HD void prime_put(const PassArgs& a, const LineArgs& b, const TileCtx& c, int s, bool fin,
                       uint32_t tid, const PrimeRegs<R>& v, cpx<R>* W) {
  const LineStage& st = b.st[s];
  const uint32_t p = st.rad, H = (p - 1) / 2;
  uint32_t chunk, w, j;
  if (!prime_slot(b, st, c, tid, &chunk, &w, &j)) return;
  const bool cj = fin && a.bwd;
  const uint32_t jq = line_div(j, st.m_ns);
  const uint32_t k = jq * st.ns * p + (j - jq * st.ns);
  cpx<R>* L = W + w * b.pitch;
  if (chunk == 0) lds_put(&L[wp(k, b.sh)], cj ? conj(v.y0) : v.y0);
#pragma unroll
  for (int i = 0; i < kPrimePairs; ++i) {
    const uint32_t q = chunk * kPrimePairs + 1 + i;
    if (q > H) continue;
    const cpx<R> lo = v.P[i] + mul_mi(v.Q[i]), hi = v.P[i] - mul_mi(v.Q[i]);
    lds_put(&L[wp(k + q * st.ns, b.sh)], cj ? conj(lo) : lo);
    lds_put(&L[wp(k + (p - q) * st.ns, b.sh)], cj ? conj(hi) : hi);
  }
}

}  // namespace pfft
