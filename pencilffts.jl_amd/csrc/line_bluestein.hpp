// Line pass in the Bluestein (chirp-z) form, for FFT lengths M with a prime
// factor above 61: X_k = c_k sum_j (x_j c_j) conj(c_{k-j}), c_j =
// exp(-i pi j^2 / M), the sum a convolution of Mb >= 2M - 1 points:
//   first   point j of the line (as in the direct form) times c_j, zero from M
//           up; first butterflies of the forward FFT, decimation in frequency
//   fwd     the next stages: bins end in digit-reversed positions
//   mid     the last forward stage, times the transform of b_m = conj(c_|m|)
//           (stored in those positions, 1 / Mb included), and the first
//           stage of the backward FFT, all in registers
//   bwd     decimation in time, the stages in reverse: natural order again
//   last    its last stage, times c_k; stored from the registers, or put into
//           LDS for the kinds with post-processing
// Every stage writes the LDS slots it has read, so one barrier a stage is
// enough, and the S stages of the two FFTs make 2 (S - 1) trips through LDS.
// The backward FFT runs on conjugates (conj(FFT(conj x))), conjugated back once
// at the end; a backward transform conjugates on the way in and out.
//
// What bounds it: arithmetic and the latency between barriers, on two to four
// times the line's points (1031-point lines of 1031 x 128 x 128 complex floats,
// 4096-point convolutions: 530 us a pass; 221 us of it is the issue of the
// butterflies).  In the generic phases, in radices of at most 8 with a barrier after
// each of 2 S + 5 phases, the same pass took 731 us.
#pragma once

#include <type_traits>

#include "line_pass.hpp"

namespace pfft {

// ---- single points of the kinds --------------------------------------------------
// Point k < M of work line w, as line_first reads it.
template <typename R, int CLS>
PFFT_HD cpx<R> line_in(const PassArgs& a, const TileCtx& c, const LineOp<R>& op,
                       const OpLine<R>& otile, uint32_t w, uint32_t k) {
  using E = std::conditional_t<CLS == LC_R2C || CLS == LC_R2C_ODD, R, cpx<R>>;
  const int64_t sk = a.sk_in;
  const E* in = (const E*)a.in + c.in_base + (int64_t)w * a.lsin[0];
  if constexpr (CLS == LC_R2R) {
    return line_point<R>(a, c, w, k);
  } else if constexpr (CLS == LC_R2C) {
    const R* x = in + 2 * (int64_t)k * sk;
    return sk == 1 ? *(const cpx<R>*)x : mk(x[0], x[sk]);
  } else if constexpr (CLS == LC_R2C_ODD) {
    return mk(in[k * sk], R(0));
  } else if constexpr (CLS == LC_C2R) {
    cpx<R> p = in[k * sk], q = conj(in[(a.M - k) * sk]);
    if (k == 0) { p.im = R(0); q.im = R(0); }   // Im of DC and Nyquist ignored
    else if (a.adjoint) { p = scl(p, R(0.5)); q = scl(q, R(0.5)); }   // X_k / w_k
    return (p + q) + mul_pi((p - q) * conj(((const cpx<R>*)a.aux)[k]));
  } else if constexpr (CLS == LC_C2R_ODD) {
    const uint32_t n = (uint32_t)a.n;
    const bool up = 2 * k > n;
    cpx<R> z = in[(up ? n - k : k) * sk];
    if (k == 0) z.im = R(0);   // Im of DC ignored
    else if (a.adjoint) z = scl(z, R(0.5));   // X_k / w_k
    return up ? conj(z) : z;
  } else {
    cpx<R> z[1] = {in[k * sk]};
    if constexpr (CLS == LC_C2C_OP) {
      if (op.op && op.side == 1) op.template apply<1>(op.line(otile, c.m0 + w), k, 0, z);
    }
    return z[0];
  }
}

// Output point k < M of work line w from the transform's value (scaling applied
// here), as line_store writes it.
template <typename R, int CLS>
PFFT_HD void line_out(const PassArgs& a, const TileCtx& c, const LineOp<R>& op,
                      const OpLine<R>& otile, uint32_t w, uint32_t k, cpx<R> v) {
  using E = std::conditional_t<CLS == LC_C2R || CLS == LC_C2R_ODD, R, cpx<R>>;
  const int64_t sk = a.sk_out;
  E* out = (E*)a.out + c.out_base + (int64_t)w * a.lsout[0];
  cpx<R> z[1] = {scl(v, a.do_scale ? (R)a.scale : R(1))};
  if constexpr (CLS == LC_C2R) {
    R* x = out + 2 * (int64_t)k * sk;
    if (sk == 1) {
      *(cpx<R>*)x = z[0];
    } else {
      x[0] = z[0].re;
      x[sk] = z[0].im;
    }
  } else if constexpr (CLS == LC_C2R_ODD) {
    out[k * sk] = z[0].re;
  } else if constexpr (CLS == LC_R2C_ODD) {
    if (2 * k < (uint32_t)a.n) out[k * sk] = a.adjoint && k ? scl(z[0], R(2)) : z[0];
  } else {
    cpx<R>* p = out + k * sk;
    if constexpr (CLS == LC_C2C_OP) {
      if (a.fs_M) {
        const cpx<R> f = ((const cpx<R>*)a.fs_tw)[(c.m0 + w) * k];
        z[0] = z[0] * (a.bwd ? conj(f) : f);
      }
      if (op.op && op.side == 2) {
        op.template apply<1>(op.line(otile, c.m0 + w), k, 0, z);
        if (op.acc) z[0] = z[0] + *p;
      }
    }
    *p = z[0];
  }
}

// ---- stages ------------------------------------------------------------------------
// Stage s over blocks of Bs = Mb / (r_0 ... r_{s-1}) points: butterfly j =
// blk ns + jj (ns = Bs / rad, nb = Mb / rad of them) takes positions blk Bs +
// jj + q ns; output q (forward) or input q (backward) carries w_Bs^(q jj), at
// (q - 1) ns + jj of the stage's table.
PFFT_HD uint32_t bs_base(const LineStage& st, uint32_t j, uint32_t* jj) {
  const uint32_t blk = line_div(j, st.m_ns);
  *jj = j - blk * st.ns;
  return blk * st.ns * st.rad + *jj;
}

template <typename R, int CLS, int RAD>
PFFT_HD void bs_first(const PassArgs& a, const LineArgs& b, const TileCtx& c, const LineOp<R>& op,
                      const OpLine<R>& otile, uint32_t tid, cpx<R>* W) {
  constexpr int BPT = line_bpt(RAD);
  const LineStage& st = b.st[0];
  const uint32_t M = (uint32_t)a.M;
  const cpx<R>* ch = (const cpx<R>*)a.bs_chirp;
  const cpx<R>* tw = (const cpx<R>*)b.tw + st.tw;
  cpx<R> v[BPT * RAD];
  uint32_t w[BPT], j[BPT];
  bool act[BPT];
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    act[i] = line_slot(b, st, c, tid + i * b.threads, b.jf_in != 0, &w[i], &j[i]);
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      cpx<R> x = mk(R(0), R(0));
      if (r * st.nb < M) {   // the same for every thread: nothing but padding above
        const uint32_t k = j[i] + r * st.nb;
        const uint32_t kk = k < M ? k : 0;
        const cpx<R> z = line_in<R, CLS>(a, c, op, otile, w[i], kk);
        const cpx<R> y = (a.bwd ? conj(z) : z) * ch[kk];
        if (k < M) x = y;
      }
      v[i * RAD + r] = x;
    }
  }
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    dft<R, RAD>(v + i * RAD);
    if (!act[i]) continue;
    cpx<R>* L = W + w[i] * b.pitch;
    lds_put(&L[wp(j[i], b.sh)], v[i * RAD]);
#pragma unroll
    for (int q = 1; q < RAD; ++q)
      lds_put(&L[wp(j[i] + q * st.ns, b.sh)], v[i * RAD + q] * tw[(q - 1) * st.ns + j[i]]);
  }
}

// dir 0: a forward stage, 1: the last forward stage, the product and the first
// backward one, 2: a backward stage
template <typename R, int RAD>
PFFT_HD void bs_stage(const PassArgs& a, const LineArgs& b, const TileCtx& c, int s, int dir,
                      uint32_t tid, cpx<R>* W) {
  constexpr int BPT = line_bpt(RAD);
  const LineStage& st = b.st[s];
  const cpx<R>* tw = (const cpx<R>*)b.tw + st.tw;
  const cpx<R>* bh = (const cpx<R>*)a.bs_bhat;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    uint32_t w, j, jj;
    const bool act = line_slot(b, st, c, tid + i * b.threads, false, &w, &j);
    const uint32_t p0 = bs_base(st, j, &jj);
    cpx<R>* L = W + w * b.pitch;
    cpx<R> v[RAD];
#pragma unroll
    for (int q = 0; q < RAD; ++q) v[q] = lds_get(&L[wp(p0 + q * st.ns, b.sh)]);
    if (dir == 2) {
#pragma unroll
      for (int q = 1; q < RAD; ++q) v[q] = v[q] * tw[(q - 1) * st.ns + jj];
    }
    dft<R, RAD>(v);
    if (dir == 1) {
#pragma unroll
      for (int q = 0; q < RAD; ++q) v[q] = conj(v[q] * bh[p0 + q * st.ns]);
      dft<R, RAD>(v);
    } else if (dir == 0) {
#pragma unroll
      for (int q = 1; q < RAD; ++q) v[q] = v[q] * tw[(q - 1) * st.ns + jj];
    }
    if (!act) continue;
#pragma unroll
    for (int q = 0; q < RAD; ++q) lds_put(&L[wp(p0 + q * st.ns, b.sh)], v[q]);
  }
}

template <typename R, int CLS, int RAD>
PFFT_HD void bs_last(const PassArgs& a, const LineArgs& b, const TileCtx& c, const LineOp<R>& op,
                     const OpLine<R>& otile, uint32_t tid, cpx<R>* W) {
  constexpr int BPT = line_bpt(RAD);
  constexpr bool direct = line_direct(CLS);
  const LineStage& st = b.st[0];
  const uint32_t M = (uint32_t)a.M;
  const cpx<R>* ch = (const cpx<R>*)a.bs_chirp;
  const cpx<R>* tw = (const cpx<R>*)b.tw + st.tw;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    uint32_t w, j;
    const bool act = line_slot(b, st, c, tid + i * b.threads, direct && b.jf_out, &w, &j);
    cpx<R>* L = W + w * b.pitch;
    cpx<R> v[RAD];
#pragma unroll
    for (int q = 0; q < RAD; ++q) v[q] = lds_get(&L[wp(j + q * st.ns, b.sh)]);
#pragma unroll
    for (int q = 1; q < RAD; ++q) v[q] = v[q] * tw[(q - 1) * st.ns + j];
    dft<R, RAD>(v);
    if (!act) continue;
#pragma unroll
    for (int q = 0; q < RAD; ++q) {
      if (q * st.nb >= M) continue;
      const uint32_t k = j + q * st.nb;
      if (k >= M) continue;
      const cpx<R> z = conj(v[q]) * ch[k];
      const cpx<R> y = a.bwd ? conj(z) : z;
      if constexpr (direct) line_out<R, CLS>(a, c, op, otile, w, k, y);
      else lds_put(&L[wp(k, b.sh)], y);
    }
  }
}

}  // namespace pfft
