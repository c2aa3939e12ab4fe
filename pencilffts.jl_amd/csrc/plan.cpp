// PLAN layer of the transform pipeline, restated in C++.
//
// Follows PencilFFTs.jl v0.15.3:
//   transform metadata      src/Transforms/{Transforms,c2c,r2c,r2r,no_transform}.jl
//   GlobalFFTParams         src/global_params.jl:50-62, input type :81-95
//   pencil chain            src/plans.jl:397-521
//   1D plans, binv, scale   src/plans.jl:523-553, product :268
// and then lowers every stage to one fused pass (transform + the transpose
// into the next pencil's memory order).
#include "plan.hpp"
#include "plane_pass.hpp"

#include <math.h>
#include <string.h>

#include <algorithm>
#include <sstream>

#include "../../include/pfft.h"

namespace pfft {

// ---- errors ----------------------------------------------------------------
static thread_local std::string g_last_error;

void set_error(int code, const std::string& msg) {
  (void)code;
  g_last_error = msg;
}
int fail(int code, const std::string& msg) {
  set_error(code, msg);
  return code;
}
const char* last_error() { return g_last_error.c_str(); }
void clear_error() { g_last_error.clear(); }

// ---- transform metadata ------------------------------------------------------
static const char* kR2RNames[11] = {"R2HC",    "HC2R",    "DHT",     "REDFT00",
                                    "REDFT01", "REDFT10", "REDFT11", "RODFT00",
                                    "RODFT01", "RODFT10", "RODFT11"};

int32_t kind_base(int32_t kind) { return kind & ~PFFT_INPLACE; }
bool kind_inplace(int32_t kind) { return (kind & PFFT_INPLACE) != 0; }

static bool is_r2r(int32_t b) { return b >= PFFT_R2R && b <= PFFT_R2R + PFFT_RODFT11; }
static bool is_c2c(int32_t b) { return b == PFFT_FFT || b == PFFT_BFFT; }
static bool is_c2r(int32_t b) { return b == PFFT_BRFFT_EVEN || b == PFFT_BRFFT_ODD; }

bool kind_valid(int32_t kind, std::string* why) {
  if (kind & ~(PFFT_INPLACE | 0xff)) {
    if (why) *why = "unknown transform kind " + std::to_string(kind);
    return false;
  }
  const int32_t b = kind_base(kind);
  if (b == PFFT_NOTRANSFORM || is_c2c(b) || b == PFFT_RFFT || is_c2r(b)) return true;
  if (is_r2r(b)) {
    const int32_t k = b - PFFT_R2R;
    if (k == PFFT_R2HC || k == PFFT_HC2R) {
      // r2r.jl:40-46
      if (why) *why = std::string("unsupported r2r transform kind: ") + kR2RNames[k];
      return false;
    }
    return true;
  }
  if (why) *why = "unknown transform kind " + std::to_string(kind);
  return false;
}

std::string kind_name(int32_t kind) {
  const int32_t b = kind_base(kind);
  const char* bang = kind_inplace(kind) ? "!" : "";
  switch (b) {
    case PFFT_NOTRANSFORM: return std::string("NoTransform") + bang;
    case PFFT_FFT: return std::string("FFT") + bang;
    case PFFT_BFFT: return std::string("BFFT") + bang;
    case PFFT_RFFT: return std::string("RFFT") + bang;
    case PFFT_BRFFT_EVEN: return std::string("BRFFT") + bang + "{even}";
    case PFFT_BRFFT_ODD: return std::string("BRFFT") + bang + "{odd}";
    default: break;
  }
  if (is_r2r(b)) return std::string("R2R") + bang + "{" + kR2RNames[b - PFFT_R2R] + "}";
  return "?";
}

std::string kind_type_name(int32_t kind) {
  const int32_t b = kind_base(kind);
  const char* bang = kind_inplace(kind) ? "!" : "";
  std::string base;
  switch (b) {
    case PFFT_NOTRANSFORM: base = "NoTransform"; break;
    case PFFT_FFT: base = "FFT"; break;
    case PFFT_BFFT: base = "BFFT"; break;
    case PFFT_RFFT: base = "RFFT"; break;
    case PFFT_BRFFT_EVEN:
    case PFFT_BRFFT_ODD: base = "BRFFT"; break;
    default:
      if (is_r2r(b))
        return std::string("PencilFFTs.Transforms.R2R") + bang + "{" +
               std::to_string(b - PFFT_R2R) + "}";
      base = "?";
  }
  return "PencilFFTs.Transforms." + base + bang;
}

std::string eltype_name(int32_t e) {
  switch (e) {
    case PFFT_F32: return "Float32";
    case PFFT_F64: return "Float64";
    case PFFT_C32: return "ComplexF32";
    case PFFT_C64: return "ComplexF64";
    default: return "Nothing";
  }
}

size_t eltype_bytes(int32_t e) {
  switch (e) {
    case PFFT_F32: return 4;
    case PFFT_F64: return 8;
    case PFFT_C32: return 8;
    case PFFT_C64: return 16;
    default: return 0;
  }
}

static bool eltype_is_complex(int32_t e) { return e == PFFT_C32 || e == PFFT_C64; }
static int32_t eltype_real(int32_t e) { return (e == PFFT_C32 || e == PFFT_F32) ? PFFT_F32 : PFFT_F64; }
static int32_t eltype_complex(int32_t e) { return eltype_real(e) == PFFT_F32 ? PFFT_C32 : PFFT_C64; }

// c2c.jl:49, r2c.jl:74-75, r2r.jl:82, no_transform.jl:23
int length_output(int32_t kind, int64_t n, int64_t* out) {
  std::string why;
  if (!kind_valid(kind, &why)) return fail(PFFT_ERR_ARGUMENT, why);
  const int32_t b = kind_base(kind);
  if (b == PFFT_RFFT) *out = n / 2 + 1;
  else if (b == PFFT_BRFFT_EVEN) *out = 2 * n - 2;
  else if (b == PFFT_BRFFT_ODD) *out = 2 * n - 1;
  else *out = n;
  return PFFT_OK;
}

// c2c.jl:58-61, r2c.jl:99-102 (BRFFT(d) = BRFFT(iseven(d)), r2c.jl:66),
// r2r.jl:103-131, no_transform.jl:21
int binv(int32_t kind, int64_t d, int32_t* inv) {
  std::string why;
  if (!kind_valid(kind, &why)) return fail(PFFT_ERR_ARGUMENT, why);
  const int32_t ip = kind & PFFT_INPLACE;
  const int32_t b = kind_base(kind);
  int32_t r;
  switch (b) {
    case PFFT_FFT: r = PFFT_BFFT; break;
    case PFFT_BFFT: r = PFFT_FFT; break;
    case PFFT_RFFT: r = (d % 2 == 0) ? PFFT_BRFFT_EVEN : PFFT_BRFFT_ODD; break;
    case PFFT_BRFFT_EVEN:
    case PFFT_BRFFT_ODD: r = PFFT_RFFT; break;
    case PFFT_NOTRANSFORM: r = PFFT_NOTRANSFORM; break;
    default: {
      const int32_t k = b - PFFT_R2R;
      int32_t ki = k;
      if (k == PFFT_REDFT01) ki = PFFT_REDFT10;
      else if (k == PFFT_REDFT10) ki = PFFT_REDFT01;
      else if (k == PFFT_RODFT01) ki = PFFT_RODFT10;
      else if (k == PFFT_RODFT10) ki = PFFT_RODFT01;
      r = PFFT_R2R + ki;
    }
  }
  *inv = r | ip;
  return PFFT_OK;
}

// Scale factor of a transform over one dimension whose input length is n:
// c2c.jl:71, r2c.jl:104-111 (c2r: the real output length), r2r.jl:96-101,
// no_transform.jl:25.
int scale_factor_1d(int32_t kind, int64_t n, int64_t* s) {
  std::string why;
  if (!kind_valid(kind, &why)) return fail(PFFT_ERR_ARGUMENT, why);
  const int32_t b = kind_base(kind);
  if (b == PFFT_NOTRANSFORM) *s = 1;
  else if (is_c2c(b) || b == PFFT_RFFT) *s = n;
  else if (is_c2r(b)) return length_output(kind, n, s);
  else {
    const int32_t k = b - PFFT_R2R;
    if (k == PFFT_REDFT00) *s = 2 * (n - 1);
    else if (k == PFFT_RODFT00) *s = 2 * (n + 1);
    else if (k == PFFT_DHT) *s = n;
    else *s = 2 * n;
  }
  return PFFT_OK;
}

// c2c.jl:51, r2c.jl:80-81, r2r.jl:83, no_transform.jl:24
int eltype_input(int32_t kind, int32_t real_type, int32_t* out) {
  std::string why;
  if (!kind_valid(kind, &why)) return fail(PFFT_ERR_ARGUMENT, why);
  if (real_type != PFFT_F32 && real_type != PFFT_F64)
    return fail(PFFT_ERR_ARGUMENT, "real type must be Float32 or Float64");
  const int32_t b = kind_base(kind);
  if (is_c2c(b) || is_c2r(b)) *out = eltype_complex(real_type);
  else if (b == PFFT_RFFT) *out = real_type;
  else *out = PFFT_NOTHING;
  return PFFT_OK;
}

// c2c.jl:50, r2c.jl:77-78, r2r.jl:84, no_transform.jl:22, error Transforms.jl:263-264
int eltype_output(int32_t kind, int32_t t, int32_t* out) {
  std::string why;
  if (!kind_valid(kind, &why)) return fail(PFFT_ERR_ARGUMENT, why);
  if (t < PFFT_F32 || t > PFFT_C64)
    return fail(PFFT_ERR_ARGUMENT, "invalid element type code " + std::to_string(t));
  const int32_t b = kind_base(kind);
  bool ok = true;
  int32_t r = t;
  if (is_c2c(b)) ok = eltype_is_complex(t);
  else if (b == PFFT_RFFT) { ok = !eltype_is_complex(t); r = eltype_complex(t); }
  else if (is_c2r(b)) { ok = eltype_is_complex(t); r = eltype_real(t); }
  if (!ok)
    return fail(PFFT_ERR_ARGUMENT, "invalid input data type for " + kind_type_name(kind) +
                                       ": " + eltype_name(t));
  *out = r;
  return PFFT_OK;
}

// ---- tables ------------------------------------------------------------------
// exp(-2 pi i num / den) with the argument reduced exactly in integers and the
// trigonometric functions evaluated in long double before rounding.
static void expm(int64_t num, int64_t den, double* re, double* im) {
  int64_t r = num % den;
  if (r < 0) r += den;
  // fold into [0, den/8] with symmetries so the long-double argument is small
  const long double tau = 6.283185307179586476925286766559005768L;
  const long double th = tau * (long double)r / (long double)den;
  *re = (double)cosl(th);
  *im = (double)(-sinl(th));
  // exact values at multiples of quarter turns
  if ((4 * r) % den == 0) {
    const int64_t q = (4 * r) / den;
    const double c[4] = {1, 0, -1, 0}, s[4] = {0, -1, 0, 1};
    *re = c[q & 3];
    *im = s[q & 3];
  } else if ((8 * r) % den == 0) {
    const double h = 0.70710678118654752440084436210485;
    const int64_t q = (8 * r) / den;  // odd
    const double c[8] = {1, h, 0, -h, -1, -h, 0, h};
    const double s[8] = {0, -h, -1, -h, 0, h, 1, h};
    *re = c[q & 7];
    *im = s[q & 7];
  }
}

// the plan's table of that key, -1 if there is none yet
static int find_table(const Plan& p, const std::string& key) {
  for (size_t i = 0; i < p.tables.size(); ++i)
    if (p.tables[i].key == key) return (int)i;
  return -1;
}

static int add_table(Plan& p, const std::string& key, std::vector<double>&& vals) {
  Table t;
  t.key = key;
  t.real_bytes = p.real_type == PFFT_F32 ? 4 : 8;
  t.values = std::move(vals);
  const size_t n = t.values.size();
  t.host.resize(n * t.real_bytes);
  if (t.real_bytes == 4) {
    float* f = (float*)t.host.data();
    for (size_t i = 0; i < n; ++i) f[i] = (float)t.values[i];
  } else {
    memcpy(t.host.data(), t.values.data(), n * 8);
  }
  p.tables.push_back(std::move(t));
  return (int)p.tables.size() - 1;
}

static int twiddle_table(Plan& p, int64_t M) {
  const std::string key = "tw" + std::to_string(M);
  const int have = find_table(p, key);
  if (have >= 0) return have;
  std::vector<double> v(2 * M);
  for (int64_t k = 0; k < M; ++k) expm(k, M, &v[2 * k], &v[2 * k + 1]);
  return add_table(p, key, std::move(v));
}

// Tables of the Bluestein form of an M-point FFT convolved at Mb points:
// the chirp c_j = exp(-i pi j^2 / M), j < M (argument j^2 mod 2M reduced
// exactly), and the Mb-point DFT of b_m = conj(c_|m|) (|m| < M, index m mod
// Mb, zero elsewhere) divided by Mb, from an FFT in long double.
// The kernel's forward convolution FFT runs in place, decimation in frequency
// over the radix schedule rad[0..ns): its output position
// p = q0 Mb/r0 + q1 Mb/(r0 r1) + ... holds bin q0 + r0 (q1 + r1 (q2 + ...)).
// The transform of b is stored in that order, so the pointwise product
// needs no reordering and the in-place inverse (decimation in time) returns
// natural order.
static int64_t dif_bin(int64_t pos, int64_t Mb, const int32_t* rad, int ns) {
  int64_t k = 0, w = 1, B = Mb;
  for (int s = 0; s < ns; ++s) {
    B /= rad[s];
    const int64_t q = (pos / B) % rad[s];
    k += q * w;
    w *= rad[s];
  }
  return k;
}

// Forward DFT in long double, by the smallest prime factor of the length.
static std::vector<std::complex<long double>> fft_long(
    const std::vector<std::complex<long double>>& x) {
  using Z = std::complex<long double>;
  const size_t n = x.size();
  const long double tau = 6.283185307179586476925286766559005768L;
  std::vector<Z> w(n), a = x, t(n);
  for (size_t k = 0; k < n; ++k)
    w[k] = {cosl(tau * (long double)k / (long double)n), -sinl(tau * (long double)k / (long double)n)};
  // Stockham: ns points done, radix q
  for (size_t ns = 1; ns < n;) {
    size_t q = 2;
    while ((n / ns) % q) ++q;
    const size_t nb = n / q;
    for (size_t j = 0; j < nb; ++j) {
      const size_t jj = j % ns, o = j / ns * ns * q + jj;
      for (size_t k = 0; k < q; ++k) {
        Z acc = 0;
        for (size_t r = 0; r < q; ++r)
          acc += a[j + r * nb] * w[(r * jj * (nb / ns) + r * k % q * nb) % n];
        t[o + k * ns] = acc;
      }
    }
    std::swap(a, t);
    ns *= q;
  }
  return a;
}

static void bluestein_tables(Plan& p, int64_t M, int64_t Mb, const int32_t* rad, int ns,
                             int32_t* chirp_id, int32_t* bhat_id) {
  std::string key = std::to_string(M) + ":" + std::to_string(Mb);
  for (int i = 0; i < ns; ++i) key += "," + std::to_string(rad[i]);
  *chirp_id = find_table(p, "bs_chirp" + key);
  *bhat_id = find_table(p, "bs_bhat" + key);
  if (*chirp_id >= 0 && *bhat_id >= 0) return;
  std::vector<double> ch(2 * M);
  for (int64_t j = 0; j < M; ++j) expm((j * j) % (2 * M), 2 * M, &ch[2 * j], &ch[2 * j + 1]);
  std::vector<long double> re(Mb, 0.0L), im(Mb, 0.0L);
  for (int64_t m = 0; m < M; ++m) {
    re[m] = ch[2 * m];
    im[m] = -(long double)ch[2 * m + 1];
    if (m) { re[Mb - m] = re[m]; im[Mb - m] = im[m]; }
  }
  std::vector<std::complex<long double>> x(Mb);
  for (int64_t m = 0; m < Mb; ++m) x[m] = {re[m], im[m]};
  x = fft_long(x);
  std::vector<double> bh(2 * Mb);
  for (int64_t pos = 0; pos < Mb; ++pos) {
    const int64_t k = dif_bin(pos, Mb, rad, ns);
    bh[2 * pos] = (double)(x[k].real() / (long double)Mb);
    bh[2 * pos + 1] = (double)(x[k].imag() / (long double)Mb);
  }
  *chirp_id = add_table(p, "bs_chirp" + key, std::move(ch));
  *bhat_id = add_table(p, "bs_bhat" + key, std::move(bh));
}

// LDS pitch (complex slots) of a generic-pass work line of Mw points: one
// pad slot after every 8 points, odd so that neighbouring lines start on
// other banks (the kernels' wp())
static int64_t line_pitch_slots(int64_t Mw) {
  if (Mw <= 0) return 0;
  const int64_t span = Mw + (Mw - 1) / 8;
  return span % 2 == 0 ? span + 1 : span;
}

static int64_t largest_prime_factor(int64_t m) {
  int64_t best = 1;
  for (int64_t q = 2; q * q <= m; ++q)
    while (m % q == 0) { best = q; m /= q; }
  return m > 1 ? std::max(best, m) : best;
}

// ---- radix schedule ----------------------------------------------------------
static int radix_schedule(int64_t M, int32_t* rad) {
  int ns = 0;
  int64_t m = M;
  for (int r : {8, 4, 2}) {
    while (m > 1 && m % r == 0) { rad[ns++] = r; m /= r; }
  }
  for (int r : {3, 5}) {
    while (m % r == 0) { rad[ns++] = r; m /= r; }
  }
  for (int64_t q = 7; m > 1; q += 2) {
    while (m % q == 0) {
      if (ns >= kMaxStages) return -1;
      rad[ns++] = (int32_t)q;
      m /= q;
    }
    if (q * q > m && m > 1) {
      if (ns >= kMaxStages) return -1;
      rad[ns++] = (int32_t)m;
      m = 1;
    }
  }
  return ns;
}

// ---- layouts -----------------------------------------------------------------
// Strides (in elements) of each logical dim and of the extra dim for a memory
// permutation `perm` of the N logical dims with sizes `dims`.
// Strides of the layout `perm` over `dims`; a nonzero pad0 is the padded
// length of memory axis 0 (the real view of an in-place r2c buffer holds
// 2 (n/2 + 1) reals per line, multiarrays_r2c.jl:75-86).
static void layout_strides(int N, const int32_t* perm, const int64_t* dims, int64_t* stride,
                           int64_t* stride_extra, int64_t pad0 = 0) {
  int64_t s = 1;
  for (int i = 0; i < N; ++i) {
    stride[perm[i]] = s;
    s *= (i == 0 && pad0 > dims[perm[i]]) ? pad0 : dims[perm[i]];
  }
  *stride_extra = s;
}

static void chain_perm(int N, int n, bool permute, int32_t* perm) {
  // plans.jl:503-521: stage n (0-based) reads data permuted as
  // (n, 0..n-1, n+1..N-1), the last stage fully reversed; stage 0 unpermuted.
  for (int i = 0; i < N; ++i) perm[i] = i;
  if (!permute || n == 0) return;
  if (n == N - 1) {
    for (int i = 0; i < N; ++i) perm[i] = N - 1 - i;
    return;
  }
  perm[0] = n;
  for (int i = 1; i <= n; ++i) perm[i] = i - 1;
  for (int i = n + 1; i < N; ++i) perm[i] = i;
}

// ---- line pass (line_pass.hpp) ------------------------------------------------
static int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

constexpr int64_t kLineSmallThreads = 128 * 1024;

// Threads per line of a schedule: the stage with the most butterflies per
// thread slot decides.
static double line_load(int64_t M, const int32_t* rad, int ns) {
  double worst = 0;
  for (int s = 0; s < ns; ++s)
    worst = std::max(worst, (double)(M / rad[s]) / (kLinePoints / rad[s]));
  return worst;
}
// Points a thread goes through in all stages, a stage's barrier and index
// arithmetic counted as ten more: what a launch of few wavefronts takes.
static double line_depth(const int32_t* rad, int ns) {
  double d = 10 * ns;
  for (int s = 0; s < ns; ++s) d += rad[s];
  return d;
}

// Radices of an M-point line: its prime factors of 17 to 61 first, then radices
// of 2 to 16, descending: the fewest stages (each one more is another trip of
// the line through LDS), then the fewest threads per line (a stage with fewer
// points per thread than the others leaves threads idle); small: the shortest
// line_depth.  0 where M does not factor that way.
static int line_schedule(int64_t M, int32_t* best, bool small = false) {
  int primes = 0;
  int64_t rest = M;
  for (int32_t q : {61, 59, 53, 47, 43, 41, 37, 31, 29, 23, 19, 17})
    while (rest % q == 0) {
      if (primes == kLineStages) return 0;
      best[primes++] = q;
      rest /= q;
    }
  if (primes && rest == 1) return primes;
  int n_best = 0;
  double load = 0;
  int32_t cur[kLineStages];
  auto rec = [&](auto&& self, int64_t m, int32_t top, int ns) -> void {
    if (m == 1) {
      const double l = small ? line_depth(cur, ns) : line_load(M, cur, ns);
      if (!n_best || (!small && ns < n_best) || ((small || ns == n_best) && l < load)) {
        n_best = ns;
        load = l;
        std::copy(cur, cur + ns, best + primes);
      }
      return;
    }
    if (primes + ns == kLineStages || (n_best && !small && ns >= n_best)) return;
    for (int32_t r = top; r >= 2; --r)
      if (m % r == 0) {
        cur[ns] = r;
        self(self, m / r, r, ns + 1);
      }
  };
  if (M > 1) rec(rec, rest, 16, 0);
  return n_best ? primes + n_best : 0;
}

static uint32_t reciprocal(int64_t d) {
  return d <= 1 ? 0u : (uint32_t)((((uint64_t)1 << 32) + d - 1) / d);
}

static int line_class(int kind) {
  return kind == L_C2C        ? LC_C2C
         : kind == L_R2C_HALF ? LC_R2C
         : kind == L_C2R_HALF ? LC_C2R
         : kind == L_R2C_FULL ? LC_R2C_ODD
         : kind == L_C2R_FULL ? LC_C2R_ODD
                              : LC_R2R;
}

// Convolution length of the Bluestein form of an M-point line FFT, the power of
// two at or above 2M - 1: 0 where M has no prime factor above kBluesteinPrime or
// one line of the convolution does not fit the workgroup.
static int64_t bluestein_length(const Plan& p, const PassArgs& a) {
  const int64_t M = a.M;
  if (largest_prime_factor(M) <= kBluesteinPrime) return 0;
  int64_t Mb = 1;
  while (Mb < 2 * M - 1) Mb *= 2;
  // one line (two for the parts of complex data): the checks of line_setup
  const int64_t Tw = a.r2r_cplx && !a.pair_real ? 2 : 1;
  const bool f32 = p.real_type == PFFT_F32;
  int32_t rad[kLineStages];
  const int S = line_schedule(Mb, rad);
  const int64_t points = Mb + (Mb >> (f32 ? 5 : 4)) + 32;
  if (!S || Tw * points * (f32 ? 8 : 16) > kMaxLds ||
      Tw * line_load(Mb, rad, S) > line_max_threads(line_class(a.kind), LF_BLUESTEIN, f32))
    return 0;
  return Mb;
}

// Build the pass for transforming logical dim `dim` from (perm_in, dims_in)
// into (perm_out, dims_out).
// Radix schedule, twiddles and per-kind tables of a pass's M-point line
// FFT (a.kind, a.n, a.M set); bluestein: in that form where it applies.
static int line_fft(Plan& p, PassPlan& pp, bool bluestein = true) {
  PassArgs& a = pp.args;
  const int lk = a.kind;
  const int64_t M = a.M, n = a.n;
  // Two real R2R lines share one complex FFT as its real and imaginary
  // parts: DCT-I / DST-I (real transforms), DCT-II / DST-II and DHT (split
  // by Hermitian symmetry afterwards) and DCT-III / DST-III (Hermitian
  // input, real transforms)
  a.pair_real = (lk == L_DCT1 || lk == L_DST1 || lk == L_DCT2 || lk == L_DST2 ||
                 lk == L_DCT3 || lk == L_DST3 || lk == L_DHT) ? 1 : 0;
  a.bs_M = bluestein ? bluestein_length(p, a) : 0;
  if (a.bs_M) {
    int32_t rad[kLineStages];
    const int S = line_schedule(a.bs_M, rad);
    bluestein_tables(p, M, a.bs_M, rad, S, &pp.bs_chirp_id, &pp.bs_bhat_id);
  } else {
    const int ns = radix_schedule(M, a.radix);
    if (ns < 0) return fail(PFFT_ERR_UNSUPPORTED, "too many radix stages");
    a.nstages = ns;
    pp.tw_id = twiddle_table(p, M);
  }
  // aux tables (one per kind family, n and M)
  const int fam = lk == L_C2R_HALF ? L_R2C_HALF
                  : lk == L_DST2 || lk == L_DCT3 || lk == L_DST3 ? L_DCT2
                  : lk == L_DST4 ? L_DCT4 : lk == L_DST4H ? L_DCT4H : lk;
  const std::string aux_key = "aux" + std::to_string(fam) + ":" + std::to_string(n) + ":" +
                              std::to_string(M);
  pp.aux_id = find_table(p, aux_key);
  if (pp.aux_id >= 0) return PFFT_OK;
  std::vector<double> aux;
  if (lk == L_R2C_HALF || lk == L_C2R_HALF) {
    aux.resize(2 * (M + 1));
    for (int64_t k = 0; k <= M; ++k) expm(k, n, &aux[2 * k], &aux[2 * k + 1]);
  } else if (lk == L_DCT2 || lk == L_DST2 || lk == L_DCT3 || lk == L_DST3) {
    aux.resize(2 * n);
    for (int64_t k = 0; k < n; ++k) expm(k, 4 * n, &aux[2 * k], &aux[2 * k + 1]);
  } else if (lk == L_DCT4 || lk == L_DST4) {
    aux.resize(4 * n);
    for (int64_t k = 0; k < n; ++k) expm(k, 4 * n, &aux[2 * k], &aux[2 * k + 1]);
    for (int64_t k = 0; k < n; ++k)
      expm(2 * k + 1, 8 * n, &aux[2 * (n + k)], &aux[2 * (n + k) + 1]);
  } else if (lk == L_DCT4H || lk == L_DST4H) {
    // entries m < n/2: the pre-twiddle c_m = exp(-i pi (4m + 1) / 4n) of the
    // half z_m; entries n/2 + m: e_m = exp(i pi m / n), the post-twiddle
    // conj(e_m) of Z_m and the split factor w_n^-m folded into it
    aux.resize(2 * n);
    const int64_t h = n / 2;
    for (int64_t m = 0; m < h; ++m) {
      expm(4 * m + 1, 8 * n, &aux[2 * m], &aux[2 * m + 1]);
      expm(-m, 2 * n, &aux[2 * (h + m)], &aux[2 * (h + m) + 1]);
    }
  } else if (lk == L_C2C && M == 1024 && p.real_type == PFFT_F32) {
    // middle twiddles of the 32 x 32 MFMA form of 1024-point lines, in the
    // order its lanes read them: entry 64 i + l is w1024^(k2 n1) with
    // k2 = l mod 32 and n1 = (i mod 4) + 8 (i div 4) + 4 (l div 32), the
    // row of accumulator register i of lane l
    aux.resize(2 * 1024);
    for (int i = 0; i < 16; ++i)
      for (int l = 0; l < 64; ++l) {
        const int64_t k2 = l & 31, n1 = (i & 3) + 8 * (i >> 2) + 4 * (l >> 5);
        expm(k2 * n1, 1024, &aux[2 * (64 * i + l)], &aux[2 * (64 * i + l) + 1]);
      }
  }
  if (!aux.empty()) pp.aux_id = add_table(p, aux_key, std::move(aux));
  return PFFT_OK;
}

// Line dims of a pass: length and input / output strides (elements), and the
// logical dim (N: the flattened extra dims, -1: none).
struct LineDim {
  int64_t len, si, so;
  int logical;
};

// Makes the generic form of a pass a line pass where it can be one: fills
// pp.line, the tile, threads, LDS and twiddles.  A pass stays with the phases
// of the generic kernel when it copies, when its FFT length has a prime
// factor above 61 whose convolution does not fit (bluestein_length), when one
// line takes more than kLineMaxThreads threads (past about 8000 points) or
// the LDS, or when a lane's offset within a tile would pass 2^31 bytes (the
// other two forms' offsets are 64-bit).
static bool line_setup(Plan& p, PassPlan& pp) {
  PassArgs& a = pp.args;
  LineArgs b = {};
  if (a.kind == L_COPY || a.M < 2) return false;
  const int64_t M = a.bs_M ? a.bs_M : a.M;   // points per work line
  int32_t rad[kLineStages];
  int S = line_schedule(M, rad);
  if (!S) return false;
  int64_t pts = kLinePoints;   // points a thread holds
  b.cls = line_class(a.kind);
  b.form = a.bs_M ? LF_BLUESTEIN : rad[0] > 16 || b.cls == LC_R2R ? LF_PRIME : LF_DIRECT;
  const int64_t max_threads = line_max_threads(b.cls, b.form, p.real_type == PFFT_F32);
  const int64_t rs = p.real_type == PFFT_F32 ? 4 : 8, cs = 2 * rs;
  const bool direct = b.cls != LC_R2C && b.cls != LC_R2R;
  b.jf_in = a.sk_in == 1;
  b.jf_out = a.sk_out == 1;
  // One pad slot per bank round (32 slots of 8 bytes, 16 of 16) spreads the
  // even strides of the first stage's writes; the line pitch puts the lines
  // of a tile side by side within a round, so that neighbouring threads on
  // neighbouring lines, a butterfly apart, meet different banks.
  b.sh = rs == 4 ? 5 : 4;
  const int64_t round = rs == 4 ? 32 : 16;
  const int64_t span = M + ((M - 1) >> b.sh);
  auto lines = [&](int64_t T) {
    const int64_t nreal = a.r2r_cplx ? 2 * T : T;
    return a.pair_real ? (nreal + 1) / 2 : nreal;
  };
  auto pitch = [&](int64_t Tw) {
    const int64_t want = Tw >= round ? 1 : round / Tw;
    int64_t q = span;
    while (q % round != want % round) ++q;
    return q * 4 > span * 5 ? (span | 1) : q;   // short lines: odd will do
  };
  auto threads = [&](int64_t Tw) {
    int64_t t = 0;
    for (int s = 0; s < S; ++s) {
      const int64_t n = Tw * (M / rad[s]);   // butterflies
      t = std::max(t, rad[s] > 16 ? ceil_div(n, 64) * 64 * ceil_div((rad[s] - 1) / 2, kPrimePairs)
                                  : ceil_div(n, std::max<int64_t>(pts / rad[s], 1)));
    }
    return ceil_div(t, 64) * 64;
  };
  auto bytes = [&](int64_t Tw) {
    return S == 1 && direct && (b.form == LF_DIRECT || b.form == LF_SMALL) ? 0 : Tw * pitch(Tw) * cs;
  };
  // lane offsets: 32 bits within a tile
  auto reach = [&](int64_t T) -> int64_t {
    if (b.form == LF_BLUESTEIN || b.form == LF_PRIME) return 0;
    const int64_t nb = M / rad[0], nbo = M / rad[S - 1];
    const int64_t ein = a.in_cplx ? cs : rs, eout = a.out_cplx ? cs : rs;
    const int64_t pin = b.cls == LC_R2C ? 2 : b.cls == LC_C2R_ODD ? rad[0] : 1;
    const int64_t pout = b.cls == LC_C2R ? 2 : 1;
    return std::max(((T - 1) * a.lsin[0] + pin * nb * a.sk_in) * ein,
                    ((T - 1) * a.lsout[0] + pout * nbo * a.sk_out) * eout);
  };
  // Tile: 128-byte runs on a transposed side and about 256 threads, more where
  // they cost no threads (a prime stage works in whole wavefronts); fewer
  // lines where threads or LDS run out (two workgroups per CU at least), where
  // the grid would not fill the chip, or where the last tile would be mostly
  // empty.  Runs stay at 32 bytes or more.
  const int64_t elt = (!b.jf_in && !a.in_cplx) || (!b.jf_out && !a.out_cplx) ? rs : cs;
  const bool moved = !b.jf_in || !b.jf_out;
  const int64_t run = moved ? 128 / elt : 1, run_min = moved ? 32 / elt : 1;
  const int64_t least = a.pair_real && !a.r2r_cplx ? 2 : 1;
  auto tiles = [&](int64_t t) {
    int64_t n = ceil_div(a.ldim[0], t);
    for (int i = 1; i < a.D; ++i) n *= a.ldim[i];
    return n;
  };
  int64_t cap = 1;
  while (cap < a.ldim[0]) cap *= 2;
  auto fits = [&](int64_t t) {
    return threads(lines(t)) <= max_threads && bytes(lines(t)) <= 80 * 1024;
  };
  auto tile = [&](int64_t grid) {
    int64_t t = std::max(run, least);
    while (t < 64 && threads(lines(t)) < 256) t *= 2;
    while (t < 64 && threads(lines(2 * t)) == threads(lines(t)) && fits(2 * t)) t *= 2;
    t = std::min(t, std::max(cap, least));
    while (t > least && !fits(t)) t /= 2;
    while (t > std::max(run_min, least) && threads(lines(t / 2)) < threads(lines(t)) &&
           (tiles(t) < grid || (a.ldim[0] * 5 < ceil_div(a.ldim[0], t) * t * 4)))
      t /= 2;
    return t;
  };
  int64_t T = tile(1024);
  // Arrays that leave most of the chip idle: the time is that of one wavefront's
  // instructions, so one butterfly a thread, of radices that keep them few
  // (below half of the 1024 threads a CU holds at 4 wavefronts per SIMD).
  if (b.form == LF_DIRECT && tiles(T) * threads(lines(T)) < kLineSmallThreads) {
    b.form = LF_SMALL;
    pts = 1;
    S = line_schedule(M, rad, true);
    T = tile(512);
  }
  b.S = S;
  const int64_t Tw = lines(T);
  if (threads(Tw) > max_threads || bytes(Tw) > kMaxLds || reach(T) >= ((int64_t)1 << 31) ||
      tiles(T) >= ((int64_t)1 << 31))
    return false;
  b.threads = (uint32_t)threads(Tw);
  // The load and store loops of the R2R kinds, on such arrays, in one round of
  // four points a thread (420 x 56 x 60 Float32, 56-point RODFT11 pass: 30.9 us
  // with the stages' threads, 28.3 us; a prime's stage bounds the lines that have one)
  if (b.form == LF_PRIME && rad[0] <= 16 && tiles(T) * threads(Tw) < kLineSmallThreads)
    b.threads = (uint32_t)std::max(threads(Tw), std::min(max_threads, ceil_div(Tw * M, 256) * 64));
  b.Tw = (uint32_t)Tw;
  while (((int64_t)1 << b.twlog) < Tw) ++b.twlog;
  b.pitch = (uint32_t)pitch(Tw);
  b.m_half = reciprocal(a.M / 2 + 1);
  b.m_line = reciprocal(a.M);
  auto reciprocal64 = [](int64_t d) -> uint64_t {   // ceil(2^64 / d)
    return d <= 1 ? 0 : ~(uint64_t)0 / (uint64_t)d + 1;
  };
  b.blocks = (uint32_t)ceil_div(a.ldim[0], T);
  b.m_blocks = reciprocal64(b.blocks);
  for (int i = 1; i < a.D; ++i) b.m_dim[i] = reciprocal64(a.ldim[i]);
  // Stages and their twiddles: entries of the M-point table in the order the
  // kernel reads them (Bluestein: of the convolution's FFTs, decimation in
  // frequency, ns the distance of a butterfly's points).
  std::string key = (a.bs_M ? "bs_line" : "line") + std::to_string(M);
  int64_t done = 1;
  uint32_t entries = 0;
  for (int s = 0; s < S; ++s) {
    LineStage& st = b.st[s];
    st.rad = (uint32_t)rad[s];
    st.nb = (uint32_t)(M / rad[s]);
    st.ns = (uint32_t)(a.bs_M ? M / (done * rad[s]) : done);
    st.m_nb = reciprocal(st.nb);
    st.m_ns = reciprocal(st.ns);
    st.tw = entries;
    if (rad[s] > 16) entries += (uint32_t)rad[s];   // its roots
    if (a.bs_M ? s < S - 1 : s > 0) entries += (uint32_t)((rad[s] - 1) * st.ns);
    done *= rad[s];
    key += "," + std::to_string(rad[s]);
  }
  if (entries) {
    pp.line_tw_id = find_table(p, key);
    if (pp.line_tw_id < 0) {
      std::vector<double> w(2 * M);
      if (!a.bs_M) w = p.tables[pp.tw_id].values;
      else
        for (int64_t k = 0; k < M; ++k) expm(k, M, &w[2 * k], &w[2 * k + 1]);
      std::vector<double> tw;
      tw.reserve(2 * entries);
      for (int s = 0; s < S; ++s) {
        const LineStage& st = b.st[s];
        if (st.rad > 16)
          for (int64_t m = 0; m < st.rad; ++m) {
            tw.push_back(w[2 * m * st.nb]);
            tw.push_back(w[2 * m * st.nb + 1]);
          }
        if (a.bs_M ? s == S - 1 : s == 0) continue;
        const int64_t step = M / ((int64_t)st.ns * st.rad);
        for (int64_t r = 1; r < st.rad; ++r)
          for (int64_t jj = 0; jj < st.ns; ++jj) {
            const size_t k = 2 * (size_t)(r * jj * step);   // r jj < rad ns
            tw.push_back(w[k]);
            tw.push_back(w[k + 1]);
          }
      }
      pp.line_tw_id = add_table(p, key, std::move(tw));
    }
  }
  pp.line = b;
  a.T = (int32_t)T;
  pp.threads = (int32_t)b.threads;
  pp.lds_bytes = bytes(Tw);
  a.ntiles = tiles(T);
  pp.grid = std::min<int64_t>(a.ntiles, 1 << 20);
  return true;
}

// LDS budget of one generic-pass tile (the tile size T halves until it fits)
#ifndef PFFT_GENERIC_TILE_LDS
#define PFFT_GENERIC_TILE_LDS (64 * 1024)
#endif
constexpr int64_t kGenericTileLds = PFFT_GENERIC_TILE_LDS;

// Line-dim order, tile size and LDS footprint of the generic pass (`dim`:
// the logical dim transformed).  *fits = false when one line does not fit
// the LDS.
static int line_layout(Plan& p, PassPlan& pp, std::vector<LineDim> lds, int dim, bool* fits) {
  PassArgs& a = pp.args;
  const int N = p.N;
  const int lk = a.kind;
  const int64_t M = a.M;
  const int64_t rs = p.real_type == PFFT_F32 ? 4 : 8;
  const int64_t cs = 2 * rs;
  using LD = LineDim;
  *fits = true;
  // Line dims in input-memory order; then the tile axis goes first: the
  // output's contiguous axis when the store transposes, else the input's
  // contiguous axis when the load is strided, else the line dim nearest in
  // input memory (consecutive lines are then adjacent in memory).
  std::stable_sort(lds.begin(), lds.end(), [](const LD& x, const LD& y) { return x.si < y.si; });
  int tile = -1;
  for (size_t i = 0; i < lds.size() && tile < 0; ++i)
    if (a.sk_out != 1 && lds[i].so == 1 && lds[i].len > 1) tile = (int)i;
  for (size_t i = 0; i < lds.size() && tile < 0; ++i)
    if (a.sk_in != 1 && lds[i].si == 1 && lds[i].len > 1) tile = (int)i;
  if (tile > 0) {
    const LD t = lds[tile];
    lds.erase(lds.begin() + tile);
    lds.insert(lds.begin(), t);
  }
  // drop unit dims except the first
  std::vector<LD> keep;
  for (size_t i = 0; i < lds.size(); ++i)
    if (i == 0 || lds[i].len > 1) keep.push_back(lds[i]);
  if ((int)keep.size() > kMaxDims) return fail(PFFT_ERR_UNSUPPORTED, "too many dimensions");
  a.D = (int32_t)keep.size();
  for (int i = 0; i < a.D; ++i) {
    a.ldim[i] = keep[i].len;
    a.lsin[i] = keep[i].si;
    a.lsout[i] = keep[i].so;
    a.llog[i] = (keep[i].logical >= 0 && keep[i].logical < N) ? keep[i].logical : -1;
  }
  a.pdim = dim;

  a.scale = 1.0;
  a.do_scale = 0;
  auto keep_generic = [&]() {
    pp.gen_args = a;
    pp.gen_threads = pp.threads;
    pp.gen_lds = pp.lds_bytes;
    pp.gen_grid = pp.grid;
    return PFFT_OK;
  };
  if (line_setup(p, pp)) return keep_generic();
  if (a.bs_M) {   // (no line pass after all: direct stages)
    pp.bs_chirp_id = pp.bs_bhat_id = -1;
    const int r = line_fft(p, pp, false);
    if (r) return r;
  }
  // tile size and LDS footprint of the generic pass
  a.Mp = line_pitch_slots(M);
  // c2c lines (and the real pairs of an even r2c, the Hermitian merge of an
  // even c2r) load straight into the work lines: no raw tile, no pre phase
  a.load_w0 = (lk == L_C2C || lk == L_R2C_HALF || lk == L_C2R_HALF) ? 1 : 0;
  auto footprint = [&](int64_t T, int64_t* w1off) {
    const int64_t nreal = a.r2r_cplx ? 2 * T : T;
    const int64_t Tw = a.pair_real ? (nreal + 1) / 2 : nreal;
    const int64_t w0 = lk == L_COPY ? 0 : Tw * a.Mp * cs;
    const int64_t w1 = (lk == L_COPY || a.nstages == 0) ? 0 : Tw * a.Mp * cs;
    const int64_t raw = a.load_w0 ? 0 : T * a.raw_pitch * rs;
    *w1off = (w0 + 255) / 256 * 256;
    return *w1off + std::max(w1, raw);
  };
  int64_t T = 1;
  while (T < 64 && T < a.ldim[0]) T *= 2;
  int64_t off = 0;
  int64_t bytes = footprint(T, &off);
  while (bytes > kGenericTileLds && T > 1) {
    T /= 2;
    bytes = footprint(T, &off);
  }
  if (bytes > kMaxLds) {
    *fits = false;
    return PFFT_OK;
  }
  a.T = (int32_t)T;
  a.lds_w1_off = off;
  pp.lds_bytes = bytes;
  // Lines whose FFT has a direct prime stage (radix 7 and up) are
  // arithmetic-heavy: twice the threads per tile hide more of it (measured
  // 13-30 % faster on such passes; the power-of-two and 3/5-smooth passes
  // measured 3-15 % slower that way)
  bool direct_prime = false;
  for (int i = 0; i < a.nstages; ++i) direct_prime = direct_prime || (a.radix[i] > 5 && a.radix[i] != 8);
  pp.threads = direct_prime ? kBlockThreadsHeavy : kBlockThreads;
  int64_t nt = (a.ldim[0] + T - 1) / T;
  for (int i = 1; i < a.D; ++i) nt *= a.ldim[i];
  a.ntiles = nt;
  pp.grid = std::min<int64_t>(nt, 1 << 20);
  return keep_generic();
}

// Four-step form of a c2c line too long for one LDS-resident pass: M = M1 M2
// with j = M2 j1 + j2 and k = k1 + M1 k2,
//   pass A: for each j2, the M1-point FFT over j1, times w_M^(j2 k1), written
//           to an intermediate Y[j2 + M2 (k1 + M1 r)] (r: the other line dims,
//           dense);
//   pass B: for each k1, the M2-point FFT over j2 of Y, written at k.
// Pass A's line dim 0 is j2 (its store's contiguous axis), which the kernel
// reads back as the tile's first line index for the twiddle.
static int split_pass(Plan& p, const PassPlan& whole, const std::vector<LineDim>& lds, int dim,
                      std::vector<PassPlan>& out) {
  const PassArgs& w = whole.args;
  const int64_t M = w.M;
  int64_t M2 = 0;
  for (int64_t f = 2; f <= M / 2; ++f)
    if (M % f == 0 && f * f >= M) { M2 = f; break; }
  if (!M2 || w.op || w.r2r_cplx)
    return fail(PFFT_ERR_UNSUPPORTED,
                "line of length " + std::to_string(M) + " does not fit the LDS-resident pass");
  const int64_t M1 = M / M2;
  int64_t rest = 1;
  std::vector<int64_t> R;
  for (const LineDim& d : lds) {
    R.push_back(rest);
    rest *= d.len;
  }
  PassPlan A = whole, B = whole;
  for (PassPlan* q : {&A, &B}) {
    q->tw_id = q->aux_id = q->bs_chirp_id = q->bs_bhat_id = q->fs_tw_id = q->line_tw_id = -1;
    PassArgs& a = q->args;
    a.bs_M = 0;
    a.fs_M = 0;
  }
  const int64_t mid = M * rest;   // intermediate elements
  // pass A
  {
    PassArgs& a = A.args;
    a.n = a.M = a.L_in = a.L_out = M1;
    a.sk_in = M2 * w.sk_in;
    a.sk_out = M2;
    a.raw_pitch = 2 * M1 + 2;
    a.fs_M = M;
    A.fs_tw_id = twiddle_table(p, M);
    A.out_elems = mid;
    A.elt_out = whole.elt_in;
    std::vector<LineDim> la = {{M2, w.sk_in, 1, -1}};
    for (size_t i = 0; i < lds.size(); ++i) la.push_back({lds[i].len, lds[i].si, M * R[i], lds[i].logical});
    int r = line_fft(p, A);
    bool fits = true;
    if (!r) r = line_layout(p, A, la, dim, &fits);
    if (r) return r;
    if (!fits || A.args.ldim[0] != M2)
      return fail(PFFT_ERR_UNSUPPORTED,
                  "line of length " + std::to_string(M) + " does not fit the LDS-resident pass");
  }
  // pass B
  {
    PassArgs& a = B.args;
    a.n = a.M = a.L_in = a.L_out = M2;
    a.sk_in = 1;
    a.sk_out = M1 * w.sk_out;
    a.raw_pitch = 2 * M2 + 2;
    B.in_elems = mid;
    B.elt_in = whole.elt_out;
    std::vector<LineDim> lb = {{M1, M2, w.sk_out, -1}};
    for (size_t i = 0; i < lds.size(); ++i) lb.push_back({lds[i].len, M * R[i], lds[i].so, lds[i].logical});
    int r = line_fft(p, B);
    bool fits = true;
    if (!r) r = line_layout(p, B, lb, dim, &fits);
    if (r) return r;
    if (!fits)
      return fail(PFFT_ERR_UNSUPPORTED,
                  "line of length " + std::to_string(M) + " does not fit the LDS-resident pass");
  }
  A.split_part = 1;
  B.split_part = 2;
  out.push_back(A);
  out.push_back(B);
  return PFFT_OK;
}

static int build_pass(Plan& p, int dim, int32_t kind, int32_t elt_in, int32_t elt_out,
                      const int32_t* perm_in, const int64_t* dims_in, const int32_t* perm_out,
                      const int64_t* dims_out, std::vector<PassPlan>& out,
                      int64_t pad_in = 0, int64_t pad_out = 0) {
  const int N = p.N;
  PassPlan pp;
  PassArgs& a = pp.args;
  memset(&a, 0, sizeof(a));
  pp.elt_in = elt_in;
  pp.elt_out = elt_out;
  pp.tw_id = -1;
  pp.aux_id = -1;
  pp.variant = 0;

  int64_t sin_[kMaxDims], sout[kMaxDims], sin_e, sout_e;
  layout_strides(N, perm_in, dims_in, sin_, &sin_e, pad_in);
  layout_strides(N, perm_out, dims_out, sout, &sout_e, pad_out);
  // element counts of the arrays the pass touches (padding included)
  pp.in_elems = p.E * sin_e;
  pp.out_elems = p.E * sout_e;

  a.L_in = dims_in[dim];
  a.L_out = dims_out[dim];
  a.sk_in = sin_[dim];
  a.sk_out = sout[dim];
  a.in_cplx = eltype_is_complex(elt_in);
  a.out_cplx = eltype_is_complex(elt_out);

  // line kind, logical length, FFT length
  const int32_t b = kind_base(kind);
  int64_t n = a.L_in, M = 0;
  int lk = L_COPY;
  int fft_bwd = 0;
  if (b == PFFT_NOTRANSFORM) {
    lk = L_COPY;
  } else if (is_c2c(b)) {
    lk = L_C2C;
    M = n;
    fft_bwd = b == PFFT_BFFT;
  } else if (b == PFFT_RFFT) {
    if (n % 2 == 0) { lk = L_R2C_HALF; M = n / 2; }
    else { lk = L_R2C_FULL; M = n; }
  } else if (is_c2r(b)) {
    n = a.L_out;
    if (n % 2 == 0) { lk = L_C2R_HALF; M = n / 2; }
    else { lk = L_C2R_FULL; M = n; }
    fft_bwd = 1;
  } else {
    const int32_t k = b - PFFT_R2R;
    a.r2r_cplx = a.in_cplx;
    switch (k) {
      case PFFT_REDFT00:
        if (n < 2) return fail(PFFT_ERR_ARGUMENT, "REDFT00 requires a length of at least 2");
        lk = L_DCT1; M = 2 * (n - 1); break;
      case PFFT_REDFT10: lk = L_DCT2; M = n; break;
      case PFFT_REDFT01: lk = L_DCT3; M = n; fft_bwd = 1; break;
      // even lengths: one n-point FFT holds two real lines' n/2-point FFTs
      case PFFT_REDFT11:
        if (n % 2 == 0) { lk = L_DCT4H; M = n; }
        else { lk = L_DCT4; M = 2 * n; }
        break;
      case PFFT_RODFT00: lk = L_DST1; M = 2 * (n + 1); break;
      case PFFT_RODFT10: lk = L_DST2; M = n; break;
      case PFFT_RODFT01: lk = L_DST3; M = n; fft_bwd = 1; break;
      case PFFT_RODFT11:
        if (n % 2 == 0) { lk = L_DST4H; M = n; }
        else { lk = L_DST4; M = 2 * n; }
        break;
      case PFFT_DHT: lk = L_DHT; M = n; break;
      default: return fail(PFFT_ERR_ARGUMENT, "unsupported r2r kind");
    }
  }
  if (lk == L_COPY) a.r2r_cplx = 0;
  a.kind = lk;
  a.bwd = fft_bwd;
  a.n = n;
  a.M = M;

  const int comp_in = a.in_cplx ? 2 : 1;
  a.raw_pitch = comp_in * a.L_in + comp_in;
  // line dims: every logical dim but `dim`, plus the flattened extra dim
  using LD = LineDim;
  std::vector<LD> lds;
  for (int d = 0; d < N; ++d)
    if (d != dim) lds.push_back({dims_in[d], sin_[d], sout[d], d});
  if (p.E > 1) lds.push_back({p.E, sin_e, sout_e, N});
  if (lds.empty()) lds.push_back({1, 0, 0, -1});
  if (lk == L_C2C) {
    // one line of the direct form: two work buffers of M + 1 points
    const int64_t cs = p.real_type == PFFT_F32 ? 8 : 16;
    const int64_t w0 = (line_pitch_slots(M) * cs + 255) / 256 * 256;
    if (w0 + line_pitch_slots(M) * cs > kMaxLds) return split_pass(p, pp, lds, dim, out);
  }
  if (lk != L_COPY) {
    const int r = line_fft(p, pp);
    if (r) return r;
  }

  bool fits = true;
  int r = line_layout(p, pp, lds, dim, &fits);
  if (r) return r;
  if (!fits)
    return fail(PFFT_ERR_UNSUPPORTED,
                "line of length " + std::to_string(n) + " does not fit the LDS-resident pass");
  out.push_back(pp);
  return PFFT_OK;
}

// ---- plane pass (plane_pass.hpp) -----------------------------------------------
// Whether a plane pass is the better one: planes of X x Y points in LDS, `planes`
// of them, a workgroup each.  It saves a launch each way (a pair of calls is 23-25 us
// of host time in six launches, 17-18 in four) and gives up parallelism: a
// plane's work runs on one CU.
//   Small planes of small arrays, any length: 16 x 32 x 64 Float64 r2c pairs 25.6
//   -> 22.7 us, 32^3 26.8 -> 23.5, 32 x 32 x 256 complex 30.8 -> 28.2; past it 64^3
//   27.9 -> 31.6 us, 32 x 32 x 4096 147 -> 202.
//   Lengths the specialised kernels lack (odd part above 3) take the line pass, which
//   a plane pass also beats with more points, while the planes are not few: r2c
//   pairs of 40^3 Float64 30.0 -> 26.6 us, 90^3 55.6 -> 45.4, 100^3 63.2 -> 53.2; past
//   it 110 x 110 x 50 Float32 37.1 -> 38.1, 180 x 120 x 60 47.3 -> 50.0.
static bool plane_fits(int64_t X, int64_t Y, int64_t n, int64_t planes) {
  auto odd_part = [](int64_t k) { while (k % 2 == 0) k /= 2; return k; };
  if (X * Y <= 1088 && X * Y * planes <= 1 << 18) return true;
  return (odd_part(n) > 3 || odd_part(Y) > 3) && X * Y <= 8192 && planes <= 256 &&
         planes * 100 >= X * Y;
}

// Stages of one dim of a plane pass; their twiddles are appended to `tw`.  False
// where the length has no register radices or a stage's butterflies do not
// fit the threads.
static bool plane_dim(Plan& p, int64_t M, int64_t lines, bool bwd, int64_t max_threads,
                      PlaneDim* d, std::vector<double>* tw, int64_t* threads) {
  int32_t rad[kLineStages];
  for (bool small : {true, false}) {
    const int S = line_schedule(M, rad, small);
    if (!S || rad[0] > 16) return false;
    // one butterfly a thread where the workgroup is large enough for it
    int64_t want = 0;
    bool ok = true;
    for (int s = 0; s < S; ++s) {
      const int64_t n = lines * (M / rad[s]);
      want = std::max(want, std::min(max_threads, ceil_div(n, 64) * 64));
      ok = ok && ceil_div(n, max_threads) <= line_bpt(rad[s]);
    }
    if (!ok) continue;
    d->S = S;
    d->bwd = bwd;
    d->lines = (uint32_t)lines;
    d->m_lines = reciprocal(lines);
    *threads = std::max(*threads, want);
    const std::vector<double> w = p.tables[twiddle_table(p, M)].values;
    int64_t ns = 1;
    for (int s = 0; s < S; ++s) {
      LineStage& st = d->st[s];
      st.rad = (uint32_t)rad[s];
      st.nb = (uint32_t)(M / rad[s]);
      st.ns = (uint32_t)ns;
      st.m_nb = reciprocal(st.nb);
      st.m_ns = reciprocal(ns);
      st.tw = (uint32_t)(tw->size() / 2);
      const int64_t step = M / (ns * rad[s]);
      if (s)
        for (int64_t r = 1; r < rad[s]; ++r)
          for (int64_t jj = 0; jj < ns; ++jj) {
            const size_t k = 2 * (size_t)(r * jj * step);
            tw->push_back(w[k]);
            tw->push_back(w[k + 1]);
          }
      ns *= rad[s];
    }
    return true;
  }
  return false;
}

// The pass over dims 0 and 1 of a 3D out-of-place plan (fwd: from the input
// pencil, else into it), the other side in natural order; false where it does
// not apply.
static bool plane_pass(Plan& p, bool fwd, PassPlan* out) {
  const Stage &sx = p.stages[0], &sy = p.stages[1];
  const int32_t kx = kind_base(fwd ? sx.kind_fwd : sx.kind_bwd);
  const int32_t ky = kind_base(fwd ? sy.kind_fwd : sy.kind_bwd);
  if (!is_c2c(ky)) return false;
  PassPlan pp;
  PassArgs& a = pp.args;
  memset(&a, 0, sizeof(a));
  const int64_t nx = p.size_in[0], mx = p.size_out[0], Y = p.size_in[1];
  a.n = nx;
  a.M = nx;
  a.kind = L_C2C;
  if (fwd ? kx == PFFT_RFFT : is_c2r(kx)) {
    const bool even = nx % 2 == 0;
    a.kind = fwd ? (even ? L_R2C_HALF : L_R2C_FULL) : (even ? L_C2R_HALF : L_C2R_FULL);
    if (even) a.M = nx / 2;
  } else if (!is_c2c(kx)) {
    return false;
  }
  if (a.M < 2 || Y < 2 || largest_prime_factor(a.M) > 13 || largest_prime_factor(Y) > 13)
    return false;
  a.bwd = kx == PFFT_BFFT || is_c2r(kx);
  pp.elt_in = fwd ? sx.elt_in : sy.elt_out;
  pp.elt_out = fwd ? sy.elt_out : sx.elt_in;
  a.in_cplx = eltype_is_complex(pp.elt_in);
  a.out_cplx = eltype_is_complex(pp.elt_out);
  const bool f32 = p.real_type == PFFT_F32;
  const int64_t rs = f32 ? 4 : 8, cs = 2 * rs;
  PlaneArgs& q = pp.plane;
  q.on = 1;
  q.fwd = fwd;
  q.cls = line_class(a.kind);
  // the plane in LDS: rows of the longer of the stored and the transformed line
  const int64_t row = std::max(a.M, mx);
  q.sh = f32 ? 5 : 4;
  q.pitch = (uint32_t)((row + ((row - 1) >> q.sh)) | 1);
  pp.lds_bytes = Y * (int64_t)q.pitch * cs;
  if (pp.lds_bytes > kMaxLds) return false;
  const int64_t planes = p.size_in[2] * p.E;
  if (planes >= ((int64_t)1 << 31) || !plane_fits(mx, Y, nx, planes) ||
      Y * cs >= 2048 || p.size_in[2] * cs >= 8192) return false;
  pp.tw_id = pp.aux_id = -1;
  pp.variant = 0;
  std::vector<double> tw;
  int64_t threads = 0;
  if (!plane_dim(p, a.M, Y, a.bwd != 0, plane_max_threads(f32), &q.x, &tw, &threads) ||
      !plane_dim(p, Y, mx, ky == PFFT_BFFT, plane_max_threads(f32), &q.y, &tw, &threads) ||
      line_fft(p, pp, false) != PFFT_OK)
    return false;
  q.threads = (uint32_t)threads;
  q.m_pairs = reciprocal(a.M / 2 + 1);
  if (!tw.empty()) {
    std::string key = "plane";
    for (const PlaneDim* d : {&q.x, &q.y})
      for (int s = 0; s < d->S; ++s) key += "," + std::to_string(d->st[s].rad);
    pp.line_tw_id = find_table(p, key);
    if (pp.line_tw_id < 0) pp.line_tw_id = add_table(p, key, std::move(tw));
  }
  const int64_t in_x = fwd ? nx : mx, out_x = fwd ? mx : nx;
  q.sx_in = q.sx_out = 1;
  q.sy_in = in_x;
  q.sy_out = out_x;
  a.L_in = in_x;
  a.L_out = out_x;
  a.sk_in = a.sk_out = 1;
  a.T = 1;
  a.D = p.E > 1 ? 2 : 1;
  a.ldim[0] = p.size_in[2];
  a.lsin[0] = in_x * Y;
  a.lsout[0] = out_x * Y;
  a.llog[0] = 2;
  a.ldim[1] = p.E;
  a.lsin[1] = a.lsin[0] * p.size_in[2];
  a.lsout[1] = a.lsout[0] * p.size_in[2];
  a.llog[1] = -1;
  for (int d = 0; d < a.D; ++d)
    q.m_dim[d] = a.ldim[d] <= 1 ? 0 : ~(uint64_t)0 / (uint64_t)a.ldim[d] + 1;
  a.scale = 1.0;
  a.ntiles = planes;
  pp.in_elems = planes * in_x * Y;
  pp.out_elems = planes * out_x * Y;
  pp.grid = std::min<int64_t>(planes, 1 << 20);
  pp.threads = (int32_t)threads;
  pp.gen_args = a;
  pp.gen_threads = pp.threads;
  pp.gen_lds = pp.lds_bytes;
  pp.gen_grid = pp.grid;
  *out = pp;
  return true;
}

// ---- spectral operators (pfft_execute_op) ------------------------------------
int op_setup(const Plan& p, int dir, const pfft_spectral_op& op, int* pass, int* side) {
  if (op.op < PFFT_OP_DERIVATIVE || op.op > PFFT_OP_DEALIAS)
    return fail(PFFT_ERR_ARGUMENT, "unknown spectral operator " + std::to_string(op.op));
  if (op.op == PFFT_OP_DERIVATIVE && (op.dim < 0 || op.dim >= p.N))
    return fail(PFFT_ERR_ARGUMENT, "derivative dimension out of range");
  for (int d = 0; d < p.N; ++d) {
    const int32_t b = kind_base(p.kinds[d]);
    if (b != PFFT_FFT && b != PFFT_BFFT && b != PFFT_RFFT)
      return fail(PFFT_ERR_UNSUPPORTED,
                  "spectral operators need wavenumbers: FFT/BFFT/RFFT dimensions only");
  }
  // mul! and the transpose of bmul! write the spectrum in the last forward
  // pass; bmul!/ldiv! and the transpose of mul! read it in the first
  // backward pass
  const bool writes = dir == PFFT_FORWARD || dir == PFFT_ADJOINT_BACKWARD;
  const std::vector<PassPlan>& list = writes ? p.fwd : p.bwd;
  *pass = writes ? (int)list.size() - 1 : 0;
  *side = writes ? 2 : 1;
  if (op.accumulate && !writes)
    return fail(PFFT_ERR_ARGUMENT,
                "accumulate applies where the spectrum is written (forward, adjoint of bmul!)");
  if (list[*pass].args.kind != L_C2C)
    return fail(PFFT_ERR_UNSUPPORTED,
                "the pass carrying a spectral operator must be a c2c one (two or more "
                "transformed dimensions)");
  if (list[*pass].split_part)
    return fail(PFFT_ERR_UNSUPPORTED,
                "a spectral operator cannot ride on a line split into two passes");
  return PFFT_OK;
}

void op_fill(const Plan& p, int dir, const pfft_spectral_op& op, int side, PassArgs& a) {
  a.op = op.op;
  a.op_side = side;
  a.op_dim = op.dim;
  a.op_conj = (dir == PFFT_ADJOINT_FORWARD || dir == PFFT_ADJOINT_BACKWARD) ? 1 : 0;
  a.op_acc = op.accumulate ? 1 : 0;
  a.op_alpha = op.alpha;
  a.kN = p.N;
  for (int d = 0; d < p.N; ++d) {
    const bool r2c = kind_base(p.kinds[d]) == PFFT_RFFT;
    a.kmode[d] = r2c ? 1 : 0;
    a.kn[d] = p.size_out[d];
    a.kmax[d] = r2c ? (double)(p.size_out[d] - 1) : (double)(p.size_out[d] / 2);
  }
}

// ---- plan construction -----------------------------------------------------
int plan_build(Plan& p, int32_t N, const int64_t* dims, const int32_t* kinds,
               int32_t real_type, int32_t permute, int32_t n_extra, const int64_t* extra,
               uint32_t flags) {
  if (N < 1 || N > kMaxDims - 1)
    return fail(PFFT_ERR_ARGUMENT, "number of transformed dimensions must be in 1.." +
                                       std::to_string(kMaxDims - 1));
  if (n_extra < 0 || n_extra > kMaxDims) return fail(PFFT_ERR_ARGUMENT, "too many extra dims");
  if (real_type != PFFT_F32 && real_type != PFFT_F64)
    return fail(PFFT_ERR_ARGUMENT, "real type must be Float32 or Float64");
  p.N = N;
  p.Ne = n_extra;
  p.real_type = real_type;
  p.permute = permute != 0;
  p.flags = flags;
  p.E = 1;
  for (int i = 0; i < n_extra; ++i) {
    if (extra[i] < 1) return fail(PFFT_ERR_ARGUMENT, "extra dims must be positive");
    p.extra[i] = extra[i];
    p.E *= extra[i];
  }
  for (int d = 0; d < N; ++d) {
    std::string why;
    if (!kind_valid(kinds[d], &why)) return fail(PFFT_ERR_ARGUMENT, why);
    if (dims[d] < 1) return fail(PFFT_ERR_ARGUMENT, "global dimensions must be positive");
    p.kinds[d] = kinds[d];
    p.size_in[d] = dims[d];
  }
  // GlobalFFTParams: in-place consistency (global_params.jl:56-60)
  bool ip0 = kind_inplace(kinds[0]);
  for (int d = 1; d < N; ++d) {
    if (kind_inplace(kinds[d]) != ip0) {
      std::string s = "cannot combine in-place and out-of-place transforms: (";
      for (int e = 0; e < N; ++e) s += (e ? ", " : "") + kind_name(kinds[e]);
      s += ")";
      return fail(PFFT_ERR_ARGUMENT, s);
    }
  }
  p.inplace = ip0;
  p.adjoint_ok = true;
  for (int d = 0; d < N; ++d)
    if (is_r2r(kind_base(kinds[d]))) p.adjoint_ok = false;
  for (int d = 0; d < N; ++d) {
    int r = length_output(kinds[d], dims[d], &p.size_out[d]);
    if (r) return r;
    if (p.size_out[d] < 1) return fail(PFFT_ERR_ARGUMENT, "transform output length is zero");
  }
  // input element type (global_params.jl:81-95)
  int32_t T = real_type;
  for (int d = 0; d < N; ++d) {
    int32_t t;
    int r = eltype_input(kinds[d], real_type, &t);
    if (r) return r;
    if (t != PFFT_NOTHING) { T = t; break; }
  }
  p.elt_in = T;

  // stages (plans.jl:406-446, 523-553)
  p.stages.clear();
  p.scale = 1.0;
  int32_t Ti = T;
  for (int n = 0; n < N; ++n) {
    Stage s;
    memset(&s, 0, sizeof(s));
    s.dim = n;
    s.kind_fwd = kinds[n];
    int r = eltype_output(kinds[n], Ti, &s.elt_out);
    if (r) return r;
    s.elt_in = Ti;
    chain_perm(N, n, p.permute, s.perm);
    for (int j = 0; j < N; ++j) {
      s.dims_before[j] = j < n ? p.size_out[j] : p.size_in[j];
      s.dims_after[j] = j <= n ? p.size_out[j] : p.size_in[j];
    }
    for (int i = 0; i < N; ++i) if (s.perm[i] == n) s.mem_axis = i;
    s.n_in = p.size_in[n];
    s.n_out = p.size_out[n];
    // binv with the input length along the transformed dimension
    r = binv(kinds[n], s.n_in, &s.kind_bwd);
    if (r) return r;
    int64_t sc;
    r = scale_factor_1d(s.kind_bwd, s.n_out, &sc);
    if (r) return r;
    p.scale *= (double)sc;
    p.stages.push_back(s);
    Ti = s.elt_out;
  }
  p.elt_out = Ti;

  // In-place plans (allocate.jl:57-83): chains that keep the element type
  // (FFT!, BFFT!, R2R!, NoTransform!) over one buffer of the largest pencil,
  // and RFFT! followed by FFT!s over the padded real layout of
  // multiarrays_r2c.jl (2 (n/2 + 1) reals per first-axis line).
  int64_t pad_real = 0;
  if (p.inplace) {
    const int32_t b0 = kind_base(kinds[0]);
    bool ok = true;
    if (b0 == PFFT_RFFT) {
      for (int d = 1; d < N; ++d) ok = ok && kind_base(kinds[d]) == PFFT_FFT;
      pad_real = 2 * (p.size_in[0] / 2 + 1);
    } else {
      for (int d = 0; d < N; ++d)
        ok = ok && kind_base(kinds[d]) != PFFT_RFFT && !is_c2r(kind_base(kinds[d]));
    }
    if (!ok)
      return fail(PFFT_ERR_UNSUPPORTED,
                  "in-place plans take FFT!/BFFT!/R2R!/NoTransform! chains, or RFFT! "
                  "followed by FFT!s (allocate.jl:57-83)");
  }
  p.pad_in0 = pad_real;

  // passes
  p.tables.clear();
  p.fwd.clear();
  p.bwd.clear();
  // Intermediate buffers are internal, so their memory order is free.  The
  // default is the reference chain (pass n writes the pencil of stage n+1);
  // when that layout would make an odd-length axis the fastest one (e.g. the
  // n/2+1 axis after an r2c), the store's runs would be misaligned, and the
  // pass keeps its input's order instead (the next pass then loads strided).
  // Not where the next pass would then read along one axis and write along
  // another, with its own lines along a third: neither side of it would move
  // in runs (315x225x189 Float32: the backward y pass 82.5 us, 35 us with
  // runs).  `next`: the dim it transforms, `def`: the order it writes by default.
  auto choose = [&](const int32_t* perm_in, const int32_t* perm_def, const int64_t* dims,
                    int next, const int32_t* def, const int64_t* dims_next, int32_t* perm_out) {
    memcpy(perm_out, perm_def, sizeof(int32_t) * N);
    auto odd = [](int64_t len) { return len > 1 && (len & 1); };
    if (!odd(dims[perm_def[0]]) || memcmp(perm_in, perm_def, sizeof(int32_t) * N) == 0) return;
    const int32_t p0 = perm_in[0];
    if (p0 != next && def && def[0] != next && def[0] != p0 && !odd(dims_next[def[0]])) return;
    memcpy(perm_out, perm_in, sizeof(int32_t) * N);
  };
  // Padded rows of intermediate buffers (the fastest dim grows by 32
  // elements).  Measured on MI355X: rows of 8 KiB and more (1024-point
  // complex lines) run 4 % faster per 1024^3 pair padded, whatever the
  // access; a buffer the next pass loads as tiles loads 6 % faster padded
  // (the 512^3 c2r pass, 4 KiB rows); a buffer of shorter rows written by
  // tile stores stores 6 % slower padded, so those keep dense rows, as do
  // rows under 2 KiB (small plans, where 32 elements would be a large
  // share).  In-place plans share one buffer between pencils and are never
  // padded.
  auto work_pad = [&](const int32_t* perm, const int64_t* dims, int32_t elt,
                      int consumer_dim) -> int64_t {
    if (p.inplace || (p.flags & PFFT_FLAG_DENSE_WORK)) return 0;
    const int64_t len = dims[perm[0]];
    const int64_t row = len * (int64_t)eltype_bytes(elt);
    const bool tile_load = perm[0] != consumer_dim;
    if (row < (tile_load ? 2048 : 8192)) return 0;
    return len + 32;
  };
  // The first two dims in one pass.  Not where a flag asks for particular kernels
  // of the single passes.
  const uint32_t single = PFFT_FLAG_GENERIC_ONLY | PFFT_FLAG_MFMA_SPLIT16 |
                          PFFT_FLAG_MFMA_BF16X3 | PFFT_FLAG_REVERSE_TILES |
                          PFFT_FLAG_STREAM_STORES | (0xffu << 16);
  PassPlan plane_fwd, plane_bwd;
  const bool planes = N == 3 && !p.inplace && !(p.flags & single) &&
                      plane_pass(p, true, &plane_fwd) && plane_pass(p, false, &plane_bwd);
  const int32_t natural[3] = {0, 1, 2};
  if (planes) {
    const Stage& s = p.stages[2];
    p.fwd.push_back(plane_fwd);
    int r = build_pass(p, 2, s.kind_fwd, s.elt_in, s.elt_out, natural, s.dims_before, s.perm,
                       s.dims_after, p.fwd);
    if (!r) r = build_pass(p, 2, s.kind_bwd, s.elt_out, s.elt_in, s.perm, s.dims_after, natural,
                           s.dims_before, p.bwd);
    if (r) return r;
    p.bwd.push_back(plane_bwd);
  }
  if (!planes) {
    int32_t cur[kMaxDims];
    int64_t cur_pad = pad_real;
    memcpy(cur, p.stages[0].perm, sizeof(cur));
    for (int n = 0; n < N; ++n) {
      const Stage& s = p.stages[n];
      int32_t outp[kMaxDims];
      if (n == N - 1) memcpy(outp, s.perm, sizeof(outp));
      else choose(cur, p.stages[n + 1].perm, s.dims_after, n + 1,
                  n + 2 < N ? p.stages[n + 2].perm : nullptr, p.stages[n + 1].dims_after, outp);
      const int64_t pad_out = n == N - 1 ? 0 : work_pad(outp, s.dims_after, s.elt_out, n + 1);
      int r = build_pass(p, n, s.kind_fwd, s.elt_in, s.elt_out, cur, s.dims_before, outp,
                         s.dims_after, p.fwd, cur_pad, pad_out);
      if (r) return r;
      memcpy(cur, outp, sizeof(cur));
      cur_pad = pad_out;
    }
  }
  if (!planes) {
    int32_t cur[kMaxDims];
    int64_t cur_pad = 0;
    memcpy(cur, p.stages[N - 1].perm, sizeof(cur));
    for (int n = N - 1; n >= 0; --n) {
      const Stage& s = p.stages[n];
      int32_t outp[kMaxDims];
      if (n == 0) memcpy(outp, s.perm, sizeof(outp));
      else choose(cur, p.stages[n - 1].perm, s.dims_before, n - 1,
                  n >= 2 ? p.stages[n - 2].perm : nullptr, p.stages[n - 1].dims_before, outp);
      const int64_t pad_out = n == 0 ? pad_real : work_pad(outp, s.dims_before, s.elt_in, n - 1);
      int r = build_pass(p, n, s.kind_bwd, s.elt_out, s.elt_in, cur, s.dims_after, outp,
                         s.dims_before, p.bwd, cur_pad, pad_out);
      if (r) return r;
      memcpy(cur, outp, sizeof(cur));
      cur_pad = pad_out;
    }
  }
  size_t w[2] = {0, 0};
  auto use = [&](PassPlan& pp) {
    if (pp.dst) {
      const size_t bytes = (size_t)pp.out_elems * eltype_bytes(pp.elt_out);
      w[pp.dst - 1] = std::max(w[pp.dst - 1], bytes);
    }
  };
  if (!p.inplace) {
    // buffers: user in -> work0 -> work1 -> work0 ... -> user out
    for (auto* list : {&p.fwd, &p.bwd}) {
      const int np = (int)list->size();
      for (int i = 0; i < np; ++i) {
        PassPlan& pp = (*list)[i];
        pp.src = i == 0 ? 0 : 1 + ((i - 1) & 1);
        pp.dst = i == np - 1 ? 0 : 1 + (i & 1);
        use(pp);
      }
    }
    p.in_bytes = (size_t)p.fwd.front().in_elems * eltype_bytes(p.elt_in);
    p.out_bytes = (size_t)p.fwd.back().out_elems * eltype_bytes(p.elt_out);
  } else {
    // One user buffer U holds every pencil (ManyPencilArray, the largest
    // pencil's size).  A pass whose input and output lines occupy the same
    // bytes (contiguous on both sides, same line strides in bytes) may run in
    // place, each line read whole before it is written; any other pass moves
    // data between U and the scratch W.  The chain starts and ends in U, so
    // the moves must be even: an odd count turns one in-place-capable pass
    // into a move, and failing that the chain uses two scratch buffers.
    size_t ubytes = 0;
    for (auto* list : {&p.fwd, &p.bwd})
      for (const PassPlan& pp : *list) {
        ubytes = std::max(ubytes, (size_t)pp.in_elems * eltype_bytes(pp.elt_in));
        ubytes = std::max(ubytes, (size_t)pp.out_elems * eltype_bytes(pp.elt_out));
      }
    for (auto* list : {&p.fwd, &p.bwd}) {
      const int np = (int)list->size();
      std::vector<bool> same(np);
      int moves = 0, first_same = -1;
      for (int i = 0; i < np; ++i) {
        const PassArgs& a = (*list)[i].args;
        const int64_t bi = eltype_bytes((*list)[i].elt_in), bo = eltype_bytes((*list)[i].elt_out);
        bool ok = a.sk_in == 1 && a.sk_out == 1;
        for (int d = 0; d < a.D && ok; ++d) ok = a.lsin[d] * bi == a.lsout[d] * bo;
        same[i] = ok;
        if (!ok) ++moves;
        else if (first_same < 0) first_same = i;
      }
      if (moves % 2 == 0 || first_same >= 0) {
        int cur = 0;   // 0 = U, 1 = W
        for (int i = 0; i < np; ++i) {
          PassPlan& pp = (*list)[i];
          const bool move = !same[i] || (moves % 2 == 1 && i == first_same);
          pp.src = cur;
          pp.dst = move ? 1 - cur : cur;
          cur = pp.dst;
          use(pp);
        }
      } else {
        if (np < 2)
          return fail(PFFT_ERR_UNSUPPORTED, "in-place plan with a single transposing pass");
        for (int i = 0; i < np; ++i) {   // U -> W0 -> W1 -> W0 ... -> U
          PassPlan& pp = (*list)[i];
          pp.src = i == 0 ? 0 : 1 + ((i - 1) & 1);
          pp.dst = i == np - 1 ? 0 : 1 + (i & 1);
          use(pp);
        }
      }
    }
    p.in_bytes = p.out_bytes = ubytes;
  }
  w[0] = (w[0] + 255) / 256 * 256;
  w[1] = (w[1] + 255) / 256 * 256;
  p.work_bytes = w[0] + w[1];
  p.work0_bytes = w[0];
  return PFFT_OK;
}

std::string plan_describe(const Plan& p) {
  // GlobalFFTParams show (global_params.jl:69-75) + extra dims (plans.jl:555-562)
  std::ostringstream o;
  o << "Transforms: (";
  for (int d = 0; d < p.N; ++d) o << (d ? ", " : "") << kind_name(p.kinds[d]);
  o << (p.N == 1 ? ",)" : ")");
  o << "\nInput type: " << eltype_name(p.elt_in);
  auto tup = [&](const int64_t* v, int n) {
    o << "(";
    for (int i = 0; i < n; ++i) o << (i ? ", " : "") << v[i];
    o << (n == 1 ? ",)" : ")");
  };
  o << "\nGlobal dimensions: ";
  tup(p.size_in, p.N);
  o << " -> ";
  tup(p.size_out, p.N);
  if (p.Ne) {
    o << "\nExtra dimensions: ";
    tup(p.extra, p.Ne);
  }
  o << "\nMPI topology: 1D decomposition (1 processes), one GPU";
  return o.str();
}

}  // namespace pfft
