// Line pass: lines of any length whose FFT length factors into radices of 2
// to 16, complex FFTs, r2c and c2r in any layout, float or double.  (The R2R
// kinds and lengths with larger primes: line_prime.hpp, line_bluestein.hpp.)
//
// One workgroup transforms a tile of lines.  Every thread holds 16 points of
// the tile in registers (one radix-9..16 butterfly, two of radix 6..8, ...):
//   first   global memory -> registers (with the c2r's merge), first
//           butterflies, registers -> LDS
//   middle  LDS -> registers, twiddles, butterflies, back to the same LDS lines
//   last    LDS -> registers, twiddles, butterflies, stored from the registers
//           (the even r2c puts the transform into LDS and splits it from there)
// A stage moves points within the line, so a barrier lies between its reads
// and its writes: one LDS copy of the tile, S - 1 trips through it for S
// radices, S <= 3 up to 4096 points.
//
// The fused transposes need no tile of their own.  On a transposed side
// neighbouring threads take neighbouring lines (the same butterfly of each), so
// every load or store instruction covers runs of T consecutive elements;
// on a contiguous side they take neighbouring butterflies of one line.  No
// access needs more than its element's alignment, and a last tile with fewer
// lines masks the others: odd and ragged extents take the same path.
//
// What bounds it: HBM traffic on the two-stage lengths (180-point lines of
// 240 x 200 x 180 complex doubles, 276 MB, in 48-53 us), latency between the
// barriers with two workgroups on a CU on the three-stage ones (448-point lines
// of 448 x 352 x 208 complex floats, 525 MB, in 123-128 us).  The generic
// phases, with one trip through LDS and one barrier per radix of at most 8
// and two more for loading and storing, took 119-167 and 303-343 us.  16
// points a thread keep S low; 8 (radices to 8) cost one more trip.
//
// The phases are functions of (thread id, the thread's registers, LDS base),
// shared by the GPU kernel and the host emulator of the CPU test-suite.
#pragma once

#include "common.hpp"
#include "dft.hpp"
#include "generic_pass.hpp"

namespace pfft {

// butterflies of one radix a thread holds: as many as fit pts points
constexpr int line_bpt(int rad, int pts = kLinePoints) { return pts / rad > 1 ? pts / rad : 1; }

// A copy of the uniform value x the compiler knows nothing about: the products
// of a step with every r of every radix stay in their case instead of filling
// the launch's first instructions (and spilling there).
PFFT_HD uint64_t opaque_s(uint64_t x) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(x));
#endif
  return x;
}

// x / d for the divisors of the index maps (m = ceil(2^32 / d), 0 for d = 1;
// exact while x d < 2^32)
PFFT_HD uint32_t line_div(uint32_t x, uint32_t m) {
  return m ? (uint32_t)(((uint64_t)x * m) >> 32) : x;
}

template <typename R>
PFFT_HD cpx<R> lds_get(const cpx<R>* p) {
  typedef R v2 __attribute__((ext_vector_type(2)));
  const v2 x = *(const v2*)p;
  return mk(x.x, x.y);
}
template <typename R>
PFFT_HD void lds_put(cpx<R>* p, cpx<R> z) {
  typedef R v2 __attribute__((ext_vector_type(2)));
  *(v2*)p = v2{z.re, z.im};
}

// x / d for tile indexes (below 2^31): m = ceil(2^64 / d), 0 for d = 1
PFFT_HD uint32_t line_div64(uint32_t x, uint64_t m) {
  if (!m) return x;
#if defined(__HIP_DEVICE_COMPILE__)
  return (uint32_t)__umul64hi((uint64_t)x, m);
#else
  return (uint32_t)(((unsigned __int128)x * m) >> 64);
#endif
}

// tile_init by reciprocals (tiles always in ascending order, line dim 0 first)
PFFT_HD void line_tile(const PassArgs& a, const LineArgs& b, uint32_t tile, TileCtx& c) {
  uint32_t rest = line_div64(tile, b.m_blocks);
  const uint32_t b0 = tile - rest * b.blocks;
  const int64_t m0 = (int64_t)b0 * a.T;
  int64_t ib = m0 * a.lsin[0], ob = m0 * a.lsout[0];
  for (int d = 1; d < a.D; ++d) {
    const uint32_t q = d + 1 < a.D ? line_div64(rest, b.m_dim[d]) : 0;
    const int64_t m = rest - q * (uint32_t)a.ldim[d];
    rest = q;
    ib += m * a.lsin[d];
    ob += m * a.lsout[d];
  }
  c.in_base = ib;
  c.out_base = ob;
  const int64_t left = a.ldim[0] - m0;
  c.Tact = (int32_t)(left < a.T ? left : a.T);
  c.tile = tile;
  c.m0 = m0;
  const int32_t nreal = a.r2r_cplx ? 2 * c.Tact : c.Tact;
  c.Tw = a.pair_real ? (nreal + 1) / 2 : nreal;
}

// Thread tid's i-th butterfly of a stage: line w and index j; jf: the
// neighbouring threads take neighbouring butterflies of one line, else the
// same butterfly of neighbouring lines.  False past the tile (w = j = 0 then,
// so that loads stay in bounds and need no branch).
PFFT_HD bool line_slot(const LineArgs& b, const LineStage& st, const TileCtx& c, uint32_t e,
                       bool jf, uint32_t* w, uint32_t* j) {
  if (jf) {
    *w = line_div(e, st.m_nb);
    *j = e - *w * st.nb;
  } else {
    *w = e & (b.Tw - 1);
    *j = e >> b.twlog;
  }
  const bool act = *w < (uint32_t)c.Tw && *j < st.nb;
  if (!act) *w = *j = 0;
  return act;
}

// ---- input points of the kinds that gather ------------------------------------
// Real line q of the tile (parts of complex data, or real lines), point j.
template <typename R>
PFFT_HD R line_real(const PassArgs& a, const TileCtx& c, uint32_t q, int64_t j) {
  const R* in = (const R*)a.in;
  if (a.r2r_cplx)
    return in[2 * (c.in_base + (int64_t)(q >> 1) * a.lsin[0] + j * a.sk_in) + (q & 1)];
  return in[c.in_base + (int64_t)q * a.lsin[0] + j * a.sk_in];
}
// Point j of real lines 2w and 2w + 1 as one complex number (zero for a last
// line without a partner).
template <typename R>
PFFT_HD cpx<R> line_pair(const PassArgs& a, const TileCtx& c, uint32_t w, int64_t j) {
  if (a.r2r_cplx)
    return ((const cpx<R>*)a.in)[c.in_base + (int64_t)w * a.lsin[0] + j * a.sk_in];
  const bool hi = 2 * w + 1 < (uint32_t)c.Tact;
  return mk(line_real<R>(a, c, 2 * w, j), hi ? line_real<R>(a, c, 2 * w + 1, j) : R(0));
}

// Point j of work line w: the input side of the R2R kinds, as phase_pre of the
// generic pass has it.
template <typename R>
PFFT_HD cpx<R> line_point(const PassArgs& a, const TileCtx& c, uint32_t w, uint32_t j) {
  const cpx<R>* aux = (const cpx<R>*)a.aux;
  const int64_t n = a.n, M = a.M;
  const cpx<R> zero = mk(R(0), R(0));
  switch (a.kind) {
    case L_DHT:
      return line_pair<R>(a, c, w, j);
    case L_DCT1:
      return line_pair<R>(a, c, w, (int64_t)j < n ? j : M - j);
    case L_DST1: {
      const int64_t jj = j;
      if (jj == 0 || jj == n + 1) return zero;
      if (jj <= n) return line_pair<R>(a, c, w, jj - 1);
      const cpx<R> z = line_pair<R>(a, c, w, M - jj - 1);
      return mk(-z.re, -z.im);
    }
    case L_DCT2:
    case L_DST2: {
      const int64_t h = (n + 1) / 2;
      const bool up = (int64_t)j < h;
      const cpx<R> z = line_pair<R>(a, c, w, up ? 2 * (int64_t)j : 2 * n - 2 * (int64_t)j - 1);
      return !up && a.kind == L_DST2 ? mk(-z.re, -z.im) : z;
    }
    case L_DCT3:
    case L_DST3: {
      const bool dst = a.kind == L_DST3;
      const cpx<R> x = line_pair<R>(a, c, w, dst ? n - 1 - (int64_t)j : (int64_t)j);
      const cpx<R> y =
          j == 0 ? zero : line_pair<R>(a, c, w, dst ? (int64_t)j - 1 : n - (int64_t)j);
      const cpx<R> wj = conj(aux[j]);
      return wj * mk(x.re, -y.re) + mul_pi(wj * mk(x.im, -y.im));
    }
    case L_DCT4:
      return (int64_t)j < n ? scl(aux[j], line_real<R>(a, c, w, j)) : zero;
    case L_DST4:
      return (int64_t)j < n ? scl(aux[j], line_real<R>(a, c, w, n - 1 - j)) : zero;
    case L_DCT4H:
    case L_DST4H: {
      if (j & 1) return zero;
      const R xa = line_real<R>(a, c, w, j), xb = line_real<R>(a, c, w, n - 1 - j);
      return aux[j >> 1] * (a.kind == L_DCT4H ? mk(xa, xb) : mk(xb, xa));
    }
    default:
      return zero;
  }
}

// ---- spectral operator -------------------------------------------------------------
// What a launch needs of the operator, read once: the pass's own dim and line
// dim 0 as scalars.  (Read where it is used, under the operator's branches, the
// descriptor's indexed fields put the whole descriptor into scratch memory:
// 752 bytes a lane, and the 180-point pass of 240 x 200 x 180 complex doubles
// took 188 us against 60 us without an operator.)
template <typename R>
struct LineOp {
  int32_t op, dim, side, acc, own;   // own: the derivative is along the pass's dim
  int32_t n, mode, d0, n0, mode0;    // d0: logical dim of line dim 0 (-1: an extra dim)
  R lim, lim0, al, alc;              // 2/3 limits; alpha, and its sign for i k
  PFFT_HD explicit LineOp(const PassArgs& a) {
    op = a.op;
    dim = a.op_dim;
    side = a.op_side;
    acc = a.op_acc;
    own = a.op_dim == a.pdim;
    d0 = a.llog[0];
    const int32_t d = d0 < 0 ? 0 : d0;
    n = (int32_t)a.kn[a.pdim];
    mode = a.kmode[a.pdim];
    n0 = (int32_t)a.kn[d];
    mode0 = a.kmode[d];
    lim = R(2.0 / 3.0) * R(a.kmax[a.pdim]);
    lim0 = R(2.0 / 3.0) * R(a.kmax[d]);
    al = (R)a.op_alpha;
    alc = a.op_conj ? -al : al;
  }
  PFFT_HD static R wave(int c, int n, int mode) {
    return mode == 1 ? R(c) : R(c < (n + 1) / 2 ? c : c - n);
  }
  // the tile's part o with line dim 0 at index m
  PFFT_HD OpLine<R> line(OpLine<R> o, int64_t m) const {
    if (d0 < 0) return o;
    const R k = wave((int)m, n0, mode0);
    if (op == 1) o.a = d0 == dim ? k : o.a;
    else if (op == 4) o.b = fabs(k) > lim0 ? R(0) : o.b;
    else o.a += k * k;
    return o;
  }
  // the part of a tile: its line dims 1 .. D - 1 (as op_tile)
  PFFT_HD OpLine<R> tile(const PassArgs& a, const LineArgs& b, uint32_t t) const {
    OpLine<R> o = {R(0), R(1)};
    uint32_t rest = line_div64(t, b.m_blocks);
    for (int d = 1; d < a.D; ++d) {
      const uint32_t q = d + 1 < a.D ? line_div64(rest, b.m_dim[d]) : 0;
      op_add<R>(a, d, (int)(rest - q * (uint32_t)a.ldim[d]), o);
      rest = q;
    }
    return o;
  }
  // points j + r nb of one line times alpha m(k)
  template <int RAD>
  PFFT_HD void apply(const OpLine<R>& o, uint32_t j, uint32_t nb, cpx<R>* x) const {
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      const R kp = wave((int)(j + r * nb), n, mode);
      cpx<R> f;
      if (op == 1) {
        f = mk(R(0), (own ? kp : o.a) * alc);
      } else if (op == 4) {
        f = mk((o.b != R(0) && fabs(kp) <= lim ? R(1) : R(0)) * al, R(0));
      } else {
        const R s2 = o.a + kp * kp;
        f = mk((op == 2 ? -s2 : s2 > R(0) ? R(-1) / s2 : R(0)) * al, R(0));
      }
      x[r] = x[r] * f;
    }
  }
};

// ---- first stage: global memory -> butterflies ----------------------------------
// op, otile: the operator and its part shared by the tile (LC_C2C_OP)
template <typename R, int CLS, int PTS, int RAD>
PFFT_HD void line_first(const PassArgs& a, const LineArgs& b, const TileCtx& c,
                        const LineOp<R>& op, const OpLine<R>& otile, uint32_t tid, cpx<R>* v) {
  constexpr int BPT = line_bpt(RAD, PTS);
  const LineStage& st = b.st[0];
  const uint32_t ls = (uint32_t)a.lsin[0], sk = (uint32_t)a.sk_in;
  const bool jf = b.jf_in != 0;
  const bool cj = a.bwd != 0;   // backward FFTs run as conj(FFT(conj x))
  // A uniform base per point and one 32-bit lane offset (the plan keeps it
  // below 2^31 bytes).
  constexpr uint32_t esz = sizeof(R) * (CLS == LC_R2C || CLS == LC_R2C_ODD ? 1 : 2);
  const char* base = (const char*)a.in + c.in_base * (int64_t)esz;
  const uint64_t step = opaque_s((uint64_t)st.nb * a.sk_in * esz * (CLS == LC_R2C ? 2 : 1));
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    uint32_t w, j;
    line_slot(b, st, c, tid + i * b.threads, jf, &w, &j);
    cpx<R>* x = v + i * RAD;
    const uint32_t off = (w * ls + j * sk * (CLS == LC_R2C ? 2 : 1)) * esz;
    if constexpr (CLS == LC_C2C || CLS == LC_C2C_OP) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) x[r] = *(const cpx<R>*)(base + r * step + off);
      if constexpr (CLS == LC_C2C_OP) {
        if (op.op && op.side == 1) op.template apply<RAD>(op.line(otile, c.m0 + w), j, st.nb, x);
      }
    } else if constexpr (CLS == LC_R2C) {
      // the real pairs (x_2j, x_2j+1) as complex points
      if (sk == 1) {
#pragma unroll
        for (int r = 0; r < RAD; ++r) x[r] = *(const cpx<R>*)(base + r * step + off);
      } else {
        const char* base1 = base + a.sk_in * (int64_t)sizeof(R);
#pragma unroll
        for (int r = 0; r < RAD; ++r)
          x[r] = mk(*(const R*)(base + r * step + off), *(const R*)(base1 + r * step + off));
      }
    } else if constexpr (CLS == LC_R2C_ODD) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) x[r] = mk(*(const R*)(base + r * step + off), R(0));
    } else if constexpr (CLS == LC_C2R) {
      // Hermitian merge of X_k and X_{M-k}, both from memory (the second
      // touch of a point comes from the caches); k = j + r nb, so M - k =
      // (RAD - 1 - r) nb + (nb - j)
      const uint32_t offb = (w * ls + (st.nb - j) * sk) * esz;
      const cpx<R>* aux = (const cpx<R>*)a.aux;
      cpx<R> B[RAD];
#pragma unroll
      for (int r = 0; r < RAD; ++r) x[r] = *(const cpx<R>*)(base + r * step + off);
#pragma unroll
      for (int r = 0; r < RAD; ++r)
        B[r] = *(const cpx<R>*)(base + (uint64_t)(RAD - 1 - r) * step + offb);
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        cpx<R> p = x[r], q = conj(B[r]);
        if (r == 0 && j == 0) { p.im = R(0); q.im = R(0); }   // Im of DC and Nyquist ignored
        else if (a.adjoint) { p = scl(p, R(0.5)); q = scl(q, R(0.5)); }   // X_k / w_k
        x[r] = (p + q) + mul_pi((p - q) * conj(aux[j + r * st.nb]));
      }
#if defined(__HIP_DEVICE_COMPILE__)
      // one butterfly's points and partners in registers at a time
      if (BPT > 1) __builtin_amdgcn_sched_barrier(0);
#endif
    } else if constexpr (CLS == LC_C2R_ODD) {
      // Hermitian extension: X_k below n / 2, conj X_{n-k} above
      const uint32_t n = (uint32_t)a.n;
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const uint32_t k = j + r * st.nb;
        const bool up = 2 * k > n;
        cpx<R> z = *(const cpx<R>*)(base + (w * ls + (up ? n - k : k) * sk) * esz);
        if (r == 0 && j == 0) z.im = R(0);   // Im of DC ignored
        else if (a.adjoint) z = scl(z, R(0.5));   // X_k / w_k
        x[r] = up ? conj(z) : z;
      }
    } else {
      static_assert(CLS != CLS, "the R2R kinds load through LDS (line_prime.hpp)");
    }
    if (cj) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) x[r] = conj(x[r]);
    }
  }
#pragma unroll
  for (int i = 0; i < BPT; ++i) dft<R, RAD>(v + i * RAD);
}

// ---- LDS slots ------------------------------------------------------------------
// Registers -> LDS after stage s: butterfly j = jq Ns + jj leaves point
// jq Ns RAD + jj + r Ns in register r; jf: as the butterflies were read.  fin:
// the last stage, with a backward transform's outer conjugation.
template <typename R, int PTS, int RAD>
PFFT_HD void line_put(const PassArgs& a, const LineArgs& b, const TileCtx& c, int s, bool jf,
                      bool fin, uint32_t tid, const cpx<R>* v, cpx<R>* W) {
  constexpr int BPT = line_bpt(RAD, PTS);
  const LineStage& st = b.st[s];
  const bool cj = fin && a.bwd;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    uint32_t w, j;
    if (!line_slot(b, st, c, tid + i * b.threads, jf, &w, &j)) continue;
    const uint32_t jq = line_div(j, st.m_ns), jj = j - jq * st.ns;
    cpx<R>* L = W + w * b.pitch;
    const uint32_t k = jq * st.ns * RAD + jj;
#pragma unroll
    for (int r = 0; r < RAD; ++r) {
      const cpx<R> z = v[i * RAD + r];
      lds_put(&L[wp(k + r * st.ns, b.sh)], cj ? conj(z) : z);
    }
  }
}

// LDS -> registers, twiddles, butterflies of stage s: point j + r nb of the
// line times w_(Ns RAD)^(r jj) (none in stage 0 of the lines loaded into LDS); jf: the last stage before a contiguous
// store.
template <typename R, int PTS, int RAD>
PFFT_HD void line_get(const LineArgs& b, const TileCtx& c, int s, bool jf, uint32_t tid, cpx<R>* v,
                      const cpx<R>* W) {
  constexpr int BPT = line_bpt(RAD, PTS);
  const LineStage& st = b.st[s];
  const cpx<R>* tw = (const cpx<R>*)b.tw + st.tw;
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    uint32_t w, j;
    line_slot(b, st, c, tid + i * b.threads, jf, &w, &j);
    const uint32_t jj = j - line_div(j, st.m_ns) * st.ns;
    const cpx<R>* L = W + w * b.pitch;
#pragma unroll
    for (int r = 0; r < RAD; ++r) v[i * RAD + r] = lds_get(&L[wp(j + r * st.nb, b.sh)]);
    if (s > 0) {
#pragma unroll
      for (int r = 1; r < RAD; ++r) v[i * RAD + r] = v[i * RAD + r] * tw[(r - 1) * st.ns + jj];
    }
  }
#pragma unroll
  for (int i = 0; i < BPT; ++i) dft<R, RAD>(v + i * RAD);
}

// ---- stores from the registers of the last stage ---------------------------------
// Register r of butterfly j holds point j + r nb.
template <typename R, int CLS, int PTS, int RAD>
PFFT_HD void line_store(const PassArgs& a, const LineArgs& b, const TileCtx& c,
                        const LineOp<R>& op, const OpLine<R>& otile, uint32_t tid,
                        const cpx<R>* v) {
  constexpr int BPT = line_bpt(RAD, PTS);
  const LineStage& st = b.st[b.S - 1];
  const uint32_t ls = (uint32_t)a.lsout[0], sk = (uint32_t)a.sk_out;
  const R sc = a.do_scale ? (R)a.scale : R(1);
  const R sci = a.bwd ? -sc : sc;
  constexpr uint32_t esz = sizeof(R) * (CLS == LC_C2R || CLS == LC_C2R_ODD ? 1 : 2);
  char* base = (char*)a.out + c.out_base * (int64_t)esz;
  const uint64_t step = opaque_s((uint64_t)st.nb * a.sk_out * esz * (CLS == LC_C2R ? 2 : 1));
#pragma unroll
  for (int i = 0; i < BPT; ++i) {
    uint32_t w, j;
    if (!line_slot(b, st, c, tid + i * b.threads, b.jf_out != 0, &w, &j)) continue;
    const uint32_t off = (w * ls + j * sk * (CLS == LC_C2R ? 2 : 1)) * esz;
    cpx<R> z[RAD];
#pragma unroll
    for (int r = 0; r < RAD; ++r) z[r] = mk(v[i * RAD + r].re * sc, v[i * RAD + r].im * sci);
    if constexpr (CLS == LC_C2R) {
      // z_m -> the real pair x_2m = Re z_m, x_2m+1 = Im z_m
      char* base1 = base + a.sk_out * (int64_t)sizeof(R);
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        if (sk == 1) {
          *(cpx<R>*)(base + r * step + off) = z[r];
        } else {
          *(R*)(base + r * step + off) = z[r].re;
          *(R*)(base1 + r * step + off) = z[r].im;
        }
      }
    } else if constexpr (CLS == LC_C2R_ODD) {
#pragma unroll
      for (int r = 0; r < RAD; ++r) *(R*)(base + r * step + off) = z[r].re;
    } else if constexpr (CLS == LC_R2C_ODD) {
      // the bins up to n / 2
#pragma unroll
      for (int r = 0; r < RAD; ++r) {
        const uint32_t k = j + r * st.nb;
        if (2 * k < (uint32_t)a.n)
          *(cpx<R>*)(base + r * step + off) = a.adjoint && k ? scl(z[r], R(2)) : z[r];
      }
    } else {
      if constexpr (CLS == LC_C2C_OP) {
        if (a.fs_M) {
          const cpx<R>* t = (const cpx<R>*)a.fs_tw;
#pragma unroll
          for (int r = 0; r < RAD; ++r) {
            const cpx<R> f = t[(c.m0 + w) * (j + r * st.nb)];
            z[r] = z[r] * (a.bwd ? conj(f) : f);
          }
        }
        if (op.op && op.side == 2) {
          op.template apply<RAD>(op.line(otile, c.m0 + w), j, st.nb, z);
          if (op.acc) {
#pragma unroll
            for (int r = 0; r < RAD; ++r) z[r] = z[r] + *(const cpx<R>*)(base + r * step + off);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < RAD; ++r) *(cpx<R>*)(base + r * step + off) = z[r];
    }
  }
}

// ---- post-processing of the even r2c ------------------------------------------------
// X_k and X_{M-k} from Z_k and Z_{M-k} of the line in LDS, both by one work
// item: E = (Z_k + conj Z_{M-k}) / 2, O = -i (Z_k - conj Z_{M-k}) / 2,
// X_k = E + w_n^k O.
template <typename R>
PFFT_HD void line_post_r2c(const PassArgs& a, const LineArgs& b, const TileCtx& c, uint32_t tid,
                           const cpx<R>* W) {
  const uint32_t M = (uint32_t)a.M, H = M / 2 + 1;
  const cpx<R>* aux = (const cpx<R>*)a.aux;
  const uint32_t count = b.jf_out ? (uint32_t)c.Tact * H : b.Tw * H;
  const R sc = a.do_scale ? (R)a.scale : R(1);
  cpx<R>* out = (cpx<R>*)a.out + c.out_base;
  for (uint32_t e = tid; e < count; e += b.threads) {
    uint32_t w, k;
    if (b.jf_out) {
      w = line_div(e, b.m_half);
      k = e - w * H;
    } else {
      w = e & (b.Tw - 1);
      k = e >> b.twlog;
      if (w >= (uint32_t)c.Tact) continue;
    }
    const cpx<R>* L = W + w * b.pitch;
    const cpx<R> p = lds_get(&L[wp(k == M ? 0 : k, b.sh)]);
    const cpx<R> q = lds_get(&L[wp(k == 0 ? 0 : M - k, b.sh)]);
    auto bin = [&](cpx<R> z, cpx<R> zc, uint32_t kk) {
      const cpx<R> E = scl(z + zc, R(0.5)), O = scl(mul_mi(z - zc), R(0.5));
      cpx<R> y = E + aux[kk] * O;
      if (a.adjoint) y = scl(y, R(herm_weight(kk, a.n)));
      return scl(y, sc);
    };
    const int64_t g = (int64_t)w * a.lsout[0];
    out[g + (int64_t)k * a.sk_out] = bin(p, conj(q), k);
    if (2 * k != M) out[g + (int64_t)(M - k) * a.sk_out] = bin(q, conj(p), M - k);
  }
}

// the kind's output from the transform in LDS
template <typename R, int CLS>
PFFT_HD void line_post(const PassArgs& a, const LineArgs& b, const TileCtx& c, uint32_t tid,
                       char* lds) {
  if constexpr (CLS == LC_R2C) line_post_r2c<R>(a, b, c, tid, (const cpx<R>*)lds);
  else phase_store<R>(a, c, (const cpx<R>*)lds, nullptr, b.pitch, b.sh, (int)tid, (int)b.threads);
}

// direct: the last stage's registers hold the output
constexpr bool line_direct(int cls) { return cls != LC_R2C && cls != LC_R2R; }

// F<radix> for a run-time radix; _POW2: for the powers of two
#define PFFT_LINE_RADIX_POW2(rad, F) \
  switch (rad) {                     \
    case 2: F(2); break;             \
    case 4: F(4); break;             \
    case 8: F(8); break;             \
    default: F(16); break;           \
  }
#define PFFT_LINE_RADIX(rad, F) \
  switch (rad) {                \
    case 2: F(2); break;        \
    case 3: F(3); break;        \
    case 4: F(4); break;        \
    case 5: F(5); break;        \
    case 6: F(6); break;        \
    case 7: F(7); break;        \
    case 8: F(8); break;        \
    case 9: F(9); break;        \
    case 10: F(10); break;      \
    case 11: F(11); break;      \
    case 12: F(12); break;      \
    case 13: F(13); break;      \
    case 14: F(14); break;      \
    case 15: F(15); break;      \
    default: F(16); break;      \
  }

}  // namespace pfft
