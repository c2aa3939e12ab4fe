// Forward DFTs of 2 to 20 points in registers (natural order in and out),
// for host and device: the butterflies of every pass kernel.  Radices 6, 10,
// 12, 14, 15 and 20 are prime-factor DFTs of two coprime ones, 9 and 16
// two-step Cooley-Tukey, 7, 11 and 13 the symmetric form of a prime length.
#pragma once

#include "common.hpp"

namespace pfft {

template <typename R>
PFFT_HD void dft2(cpx<R>* v) {
  const cpx<R> a = v[0], b = v[1];
  v[0] = a + b; v[1] = a - b;
}
template <typename R>
PFFT_HD void dft3(cpx<R>* v) {
  const R c = R(-0.5), s = R(0.86602540378443864676372317075294);
  const cpx<R> t = v[1] + v[2];
  const cpx<R> d = v[1] - v[2];
  const cpx<R> m = v[0] + scl(t, c);
  const cpx<R> u = mk(d.im * s, -d.re * s);  // -i s d
  v[0] = v[0] + t;
  v[1] = m + u;
  v[2] = m - u;
}
template <typename R>
PFFT_HD void dft4(cpx<R>* v) {
  const cpx<R> t0 = v[0] + v[2], t1 = v[0] - v[2];
  const cpx<R> t2 = v[1] + v[3], t3 = mul_mi(v[1] - v[3]);
  v[0] = t0 + t2; v[2] = t0 - t2; v[1] = t1 + t3; v[3] = t1 - t3;
}
template <typename R>
PFFT_HD void dft5(cpx<R>* v) {
  const R c1 = R(0.30901699437494742410229341718282);
  const R c2 = R(-0.80901699437494742410229341718282);
  const R s1 = R(0.95105651629515357211643933337938);
  const R s2 = R(0.58778525229247312916870595463907);
  const cpx<R> a0 = v[0];
  const cpx<R> sa = v[1] + v[4], da = v[1] - v[4];
  const cpx<R> sb = v[2] + v[3], db = v[2] - v[3];
  const cpx<R> p1 = a0 + scl(sa, c1) + scl(sb, c2);
  const cpx<R> p2 = a0 + scl(sa, c2) + scl(sb, c1);
  const cpx<R> q1 = scl(da, s1) + scl(db, s2);   // times -i
  const cpx<R> q2 = scl(da, s2) - scl(db, s1);   // times -i
  v[0] = a0 + sa + sb;
  v[1] = p1 + mul_mi(q1);
  v[4] = p1 - mul_mi(q1);
  v[2] = p2 + mul_mi(q2);
  v[3] = p2 - mul_mi(q2);
}
template <typename R>
PFFT_HD void dft8(cpx<R>* v) {
  const R h = R(0.70710678118654752440084436210485);
  cpx<R> b[4], c[4];
  for (int r = 0; r < 4; ++r) { b[r] = v[r] + v[r + 4]; c[r] = v[r] - v[r + 4]; }
  c[1] = mk((c[1].re + c[1].im) * h, (c[1].im - c[1].re) * h);   // * (1-i)/sqrt2
  c[2] = mul_mi(c[2]);                                           // * -i
  c[3] = mk((c[3].im - c[3].re) * h, -(c[3].re + c[3].im) * h);  // * (-1-i)/sqrt2
  dft4(b); dft4(c);
  v[0] = b[0]; v[2] = b[1]; v[4] = b[2]; v[6] = b[3];
  v[1] = c[0]; v[3] = c[1]; v[5] = c[2]; v[7] = c[3];
}

template <typename R>
PFFT_HD void dft16(cpx<R>* v) {
  // 16 = 4 x 4: n = 4a + b, k = k1 + 4 k2
  const R c1 = R(0.92387953251128675612818318939679);  // cos(pi/8)
  const R s1 = R(0.38268343236508977172845998403040);  // sin(pi/8)
  const R h = R(0.70710678118654752440084436210485);
  cpx<R> y[16];
#pragma unroll
  for (int b = 0; b < 4; ++b) {
    cpx<R> t[4] = {v[b], v[4 + b], v[8 + b], v[12 + b]};
    dft4(t);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) y[4 * b + k1] = t[k1];
  }
  // twiddles w16^(b k1)
  y[5] = mk(y[5].re * c1 + y[5].im * s1, y[5].im * c1 - y[5].re * s1);      // w^1
  y[6] = mk((y[6].re + y[6].im) * h, (y[6].im - y[6].re) * h);              // w^2
  y[7] = mk(y[7].re * s1 + y[7].im * c1, y[7].im * s1 - y[7].re * c1);      // w^3
  y[9] = mk((y[9].re + y[9].im) * h, (y[9].im - y[9].re) * h);              // w^2
  y[10] = mul_mi(y[10]);                                                    // w^4
  y[11] = mk((y[11].im - y[11].re) * h, -(y[11].re + y[11].im) * h);        // w^6
  y[13] = mk(y[13].re * s1 + y[13].im * c1, y[13].im * s1 - y[13].re * c1); // w^3
  y[14] = mk((y[14].im - y[14].re) * h, -(y[14].re + y[14].im) * h);        // w^6
  y[15] = mk(-y[15].re * c1 - y[15].im * s1, -y[15].im * c1 + y[15].re * s1); // w^9
#pragma unroll
  for (int k1 = 0; k1 < 4; ++k1) {
    cpx<R> t[4] = {y[k1], y[4 + k1], y[8 + k1], y[12 + k1]};
    dft4(t);
#pragma unroll
    for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = t[k2];
  }
}

template <typename R>
PFFT_HD void dft9(cpx<R>* v) {
  // 9 = 3 x 3: n = 3a + b, k = k1 + 3 k2
  const R c1 = R(0.76604444311897803520239265055541667), s1 = R(0.64278760968653932632264340990726343);   // cos, sin of 2 pi / 9
  const R c2 = R(0.17364817766693034885171662676931480), s2 = R(0.98480775301220805936674302458952301);   // 4 pi / 9
  const R c4 = R(-0.93969262078590838405410927732473147), s4 = R(0.34202014332566873304409961468225958);  // 8 pi / 9
  cpx<R> y[9];
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    cpx<R> t[3] = {v[b], v[3 + b], v[6 + b]};
    dft3(t);
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) y[3 * b + k1] = t[k1];
  }
  y[4] = y[4] * mk(c1, -s1);
  y[5] = y[5] * mk(c2, -s2);
  y[7] = y[7] * mk(c2, -s2);
  y[8] = y[8] * mk(c4, -s4);
#pragma unroll
  for (int k1 = 0; k1 < 3; ++k1) {
    cpx<R> t[3] = {y[k1], y[3 + k1], y[6 + k1]};
    dft3(t);
#pragma unroll
    for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = t[k2];
  }
}

// Prime length P (7, 11, 13), symmetric form: with A_r = v_r + v_{P-r} and
// B_r = v_r - v_{P-r} (r, q = 1 .. (P-1)/2),
//   y_0 = v_0 + sum_r A_r,  y_q, y_{P-q} = P_q -+ i Q_q,
//   P_q = v_0 + sum_r A_r cos(2 pi q r / P),  Q_q = sum_r B_r sin(2 pi q r / P).
// cs: the cosines, sn: the sines of 2 pi m / P, m < P.
template <typename R, int P>
PFFT_HD void dft_prime(cpx<R>* v, const R (&cs)[P], const R (&sn)[P]) {
  constexpr int H = (P - 1) / 2;
  cpx<R> A[H + 1], B[H + 1];
  const cpx<R> v0 = v[0];
  cpx<R> y0 = v0;
#pragma unroll
  for (int r = 1; r <= H; ++r) {
    A[r] = v[r] + v[P - r];
    B[r] = v[r] - v[P - r];
    y0 = y0 + A[r];
  }
  v[0] = y0;
#pragma unroll
  for (int q = 1; q <= H; ++q) {
    cpx<R> p = v0, u = mk(R(0), R(0));
#pragma unroll
    for (int r = 1; r <= H; ++r) {
      const int m = (q * r) % P;
      p = p + scl(A[r], cs[m]);
      u = u + scl(B[r], sn[m]);
    }
    v[q] = p + mul_mi(u);
    v[P - q] = p - mul_mi(u);
  }
}
template <typename R>
PFFT_HD void dft7(cpx<R>* v) {
  const R cs[7] = {
      R(1.00000000000000000000000000000000000), R(0.62348980185873353052500488400423981),
      R(-0.22252093395631440428890256449679476), R(-0.90096886790241912623610231950744505),
      R(-0.90096886790241912623610231950744505), R(-0.22252093395631440428890256449679476),
      R(0.62348980185873353052500488400423981)};
  const R sn[7] = {
      R(0.00000000000000000000000000000000000), R(0.78183148246802980870844452667405775),
      R(0.97492791218182360701813168299393122), R(0.43388373911755812047576833284835875),
      R(-0.43388373911755812047576833284835875), R(-0.97492791218182360701813168299393122),
      R(-0.78183148246802980870844452667405775)};
  dft_prime<R, 7>(v, cs, sn);
}
template <typename R>
PFFT_HD void dft11(cpx<R>* v) {
  const R cs[11] = {
      R(1.00000000000000000000000000000000000), R(0.84125353283118116886181164891936772),
      R(0.41541501300188642552927414922962320), R(-0.14231483827328514044379266861636967),
      R(-0.65486073394528506405692507246629355), R(-0.95949297361449738989036805706632770),
      R(-0.95949297361449738989036805706632770), R(-0.65486073394528506405692507246629355),
      R(-0.14231483827328514044379266861636967), R(0.41541501300188642552927414922962320),
      R(0.84125353283118116886181164891936772)};
  const R sn[11] = {
      R(0.00000000000000000000000000000000000), R(0.54064081745559758210763595431869170),
      R(0.90963199535451837141171538307902846), R(0.98982144188093273237609203777671879),
      R(0.75574957435425828377403584397234442), R(0.28173255684142969771141791534661690),
      R(-0.28173255684142969771141791534661690), R(-0.75574957435425828377403584397234442),
      R(-0.98982144188093273237609203777671879), R(-0.90963199535451837141171538307902846),
      R(-0.54064081745559758210763595431869170)};
  dft_prime<R, 11>(v, cs, sn);
}
template <typename R>
PFFT_HD void dft13(cpx<R>* v) {
  const R cs[13] = {
      R(1.00000000000000000000000000000000000), R(0.88545602565320989590037552201509888),
      R(0.56806474673115580251180755912751662), R(0.12053668025532305334906768745254358),
      R(-0.35460488704253562596963789260001847), R(-0.74851074817110109863463059970135138),
      R(-0.97094181742605202715698227629378923), R(-0.97094181742605202715698227629378923),
      R(-0.74851074817110109863463059970135138), R(-0.35460488704253562596963789260001847),
      R(0.12053668025532305334906768745254358), R(0.56806474673115580251180755912751662),
      R(0.88545602565320989590037552201509888)};
  const R sn[13] = {
      R(0.00000000000000000000000000000000000), R(0.46472317204376854565601533513310478),
      R(0.82298386589365639457961742343938199), R(0.99270887409805399280075164949252018),
      R(0.93501624268541482343978459983783073), R(0.66312265824079520237678549266676628),
      R(0.23931566428755776714875372626021190), R(-0.23931566428755776714875372626021190),
      R(-0.66312265824079520237678549266676628), R(-0.93501624268541482343978459983783073),
      R(-0.99270887409805399280075164949252018), R(-0.82298386589365639457961742343938199),
      R(-0.46472317204376854565601533513310478)};
  dft_prime<R, 13>(v, cs, sn);
}

// Good-Thomas prime-factor DFT of N1 N2 points, N1 and N2 coprime: with the
// index maps n = (N2 n1 + N1 n2) mod N and k = (N2 <1/N2 mod N1> k1 + N1 <1/N1
// mod N2> k2) mod N it is N1 DFTs of N2 points, then N2 DFTs of N1 points,
// with no twiddles; the maps are compile-time register renamings.
constexpr int inv_mod(int a, int m) {
  for (int x = 1; x < m; ++x)
    if ((a * x) % m == 1) return x;
  return 1;
}
template <typename R, int RAD>
PFFT_HD void dft(cpx<R>* v);
template <typename R, int N1, int N2>
PFFT_HD void dft_pfa(cpx<R>* v) {
  constexpr int N = N1 * N2;
  constexpr int E1 = N2 * inv_mod(N2 % N1, N1), E2 = N1 * inv_mod(N1 % N2, N2);
  cpx<R> t[N1][N2];
#pragma unroll
  for (int n1 = 0; n1 < N1; ++n1)
#pragma unroll
    for (int n2 = 0; n2 < N2; ++n2) t[n1][n2] = v[(N2 * n1 + N1 * n2) % N];
#pragma unroll
  for (int n1 = 0; n1 < N1; ++n1) dft<R, N2>(t[n1]);
#pragma unroll
  for (int k2 = 0; k2 < N2; ++k2) {
    cpx<R> u[N1];
#pragma unroll
    for (int n1 = 0; n1 < N1; ++n1) u[n1] = t[n1][k2];
    dft<R, N1>(u);
#pragma unroll
    for (int k1 = 0; k1 < N1; ++k1) v[(E1 * k1 + E2 * k2) % N] = u[k1];
  }
}

template <typename R, int RAD>
PFFT_HD void dft(cpx<R>* v) {
  if constexpr (RAD == 2) dft2(v);
  else if constexpr (RAD == 3) dft3(v);
  else if constexpr (RAD == 4) dft4(v);
  else if constexpr (RAD == 5) dft5(v);
  else if constexpr (RAD == 8) dft8(v);
  else if constexpr (RAD == 16) dft16(v);
  else if constexpr (RAD == 7) dft7(v);
  else if constexpr (RAD == 9) dft9(v);
  else if constexpr (RAD == 11) dft11(v);
  else if constexpr (RAD == 13) dft13(v);
  else if constexpr (RAD == 6) dft_pfa<R, 2, 3>(v);
  else if constexpr (RAD == 10) dft_pfa<R, 2, 5>(v);
  else if constexpr (RAD == 12) dft_pfa<R, 4, 3>(v);
  else if constexpr (RAD == 14) dft_pfa<R, 2, 7>(v);
  else if constexpr (RAD == 15) dft_pfa<R, 3, 5>(v);
  else if constexpr (RAD == 20) dft_pfa<R, 4, 5>(v);
  else static_assert(RAD == 0, "no register DFT of this radix");
}

}  // namespace pfft
