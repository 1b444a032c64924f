// or_math.h -- accurate FP64 log, exp and pow for the FP64 path, host and device.
//
// The reference engine evaluates X**Y, LOG and EXP with the host C library,
// whose results are correctly rounded in all but a tiny fraction of cases.
// The device math library's pow / log / exp are accurate to about one ulp, so
// their last bit differs from the host's often enough to drift FP64 trajectories
// by 1e-12 over a few hundred cycles.  These routines compute the function in
// double-double arithmetic with about 2^-70 relative error before the final
// rounding, so the returned double is the correctly rounded value except when
// the exact result lies within ~2^-17 ulp of a rounding boundary.
//
// Method: table-driven argument reduction (P. T. P. Tang, "Table-driven
// implementation of the logarithm function in IEEE floating-point arithmetic",
// ACM TOMS 16(4), 1990, and "... of the exponential function", ACM TOMS 15(2),
// 1989) carried out in double-double arithmetic (Dekker 1971; Muller et al.,
// Handbook of Floating-Point Arithmetic, ch. 14).  Tables are generated by
// gen_math_tables.py with 60-digit decimal arithmetic.
//
// Domain: log for normal finite x > 0; exp for |z| < 708 (normal results); pow
// for normal finite x > 0, finite y and |y ln x| < 708, plus x == 0 with y > 0
// and the exact cases y == 0, x == 1.  Other arguments (subnormal, infinite or
// NaN input, results outside the normal range) fall back to the library of the
// compiling side; they do not occur on this path.
//
// The device tries a shorter evaluation first (log_fast, exp_fast: fewer polynomial terms,
// the low word in plain double, fused multiply-adds) and keeps its result only when every
// value within kFastErr of it rounds to the same double (Ziv's rounding test, ACM TOMS
// 17(3), 1991); the double-double value lies within that distance, so both give the same
// bits.  Over the path's ranges the test fails for 1 argument in 8,000 (exp, pow) or 41,000 (log), which
// takes the double-double path.
// What it is for: a plastic shell point calls log and exp five times in one dependent
// chain, and a wave's chain, not the issue rate, bounds the shell kernel.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#define OR_TABLE constexpr
#include "or_math_tables.h"

namespace ormath {

struct dd {
  double hi, lo;
};

// Where an evaluation reads the tables: GlobalTab, the constant arrays, or another type with
// the same members (the FP64 shell kernel's copy in LDS).  need(cond) comes before evaluations
// that the caller makes where cond holds.
struct GlobalTab {
  __host__ __device__ __forceinline__ void need(bool) const {}
  __host__ __device__ __forceinline__ double lg(int i, int k) const { return or_log_tab[i][k]; }
  __host__ __device__ __forceinline__ double ex(int j, int k) const { return or_exp_tab[j][k]; }
};

constexpr int kLogWords = 193 * 3, kExpWords = 128 * 2;
constexpr int kTabWords = (kLogWords + kExpWords + 3) / 4 * 4; // 32-byte multiple
struct MathTab {
  double v[kTabWords];
};
constexpr MathTab make_math_tab() {
  MathTab t{};
  for (int i = 0; i < kLogWords; ++i) t.v[i] = or_log_tab[i / 3][i % 3];
  for (int j = 0; j < kExpWords; ++j) t.v[kLogWords + j] = or_exp_tab[j / 2][j % 2];
  return t;
}

__host__ __device__ __forceinline__ dd two_sum(double a, double b) {
  double s = a + b;
  double bb = s - a;
  double e = (a - (s - bb)) + (b - bb);
  return {s, e};
}
__host__ __device__ __forceinline__ dd fast_two_sum(double a, double b) {
  double s = a + b;
  double e = b - (s - a);
  return {s, e};
}
__host__ __device__ __forceinline__ dd two_prod(double a, double b) {
  double p = a * b;
  double e = fma(a, b, -p);
  return {p, e};
}
__host__ __device__ __forceinline__ dd dd_add(dd a, dd b) {
  dd s = two_sum(a.hi, b.hi);
  double lo = s.lo + (a.lo + b.lo);
  return fast_two_sum(s.hi, lo);
}

// ln(x) as a double-double, x finite > 0 and normal.
template <class T = GlobalTab>
__host__ __device__ inline dd log_dd(double x, const T tab = T{}) {
  int64_t bits;
  __builtin_memcpy(&bits, &x, 8);
  int e = (int)((bits >> 52) & 0x7ff) - 1023;
  int64_t mb = (bits & 0x000fffffffffffffLL) | 0x3ff0000000000000LL; // m in [1,2)
  double m;
  __builtin_memcpy(&m, &mb, 8);
  if (m >= 1.5) { m = 0.5 * m; e += 1; }                       // m in [0.75, 1.5)
  const int i = (int)rint((m - 0.75) * 256.0);                  // cell center c_i = 0.75 + i/256
  const double r = tab.lg(i, 0);
  // t = m*r - 1 exactly as a double-double (p - 1 is exact since p is in [0.5, 2])
  dd p = two_prod(m, r);
  dd t = two_sum(p.hi - 1.0, p.lo);
  // log1p(t) = t - t^2/2 + t^3/3 - ..., |t| < 2^-8.5; t^2 term in double-double
  dd t2 = two_prod(t.hi, t.hi);
  t2.lo = t2.lo + 2.0 * t.hi * t.lo;
  const double th = t.hi;
  double q = -1.0 / 12.0;
  q = 1.0 / 11.0 + th * q;
  q = -1.0 / 10.0 + th * q;
  q = 1.0 / 9.0 + th * q;
  q = -1.0 / 8.0 + th * q;
  q = 1.0 / 7.0 + th * q;
  q = -1.0 / 6.0 + th * q;
  q = 1.0 / 5.0 + th * q;
  q = -1.0 / 4.0 + th * q;
  q = 1.0 / 3.0 + th * q;
  const double cub = th * th * th * q;
  dd l1p = dd_add(t, dd{-0.5 * t2.hi, -0.5 * t2.lo});
  l1p = dd_add(l1p, dd{cub, 0.0});
  dd tl = {tab.lg(i, 1), tab.lg(i, 2)};
  dd el = {(double)e * OR_LN2_HI, (double)e * OR_LN2_LO};    // e*LN2_HI exact (42-bit LN2_HI)
  dd s = dd_add(el, tl);
  return dd_add(s, l1p);
}

// exp(z) for z = zh + zl (double-double), |zh| < 708: the correctly rounded double in all but
// a tiny fraction of cases.
template <class T = GlobalTab>
__host__ __device__ inline double exp_dd(double zh, double zl, const T tab = T{}) {
  const double kd = rint(zh * OR_INVLN2N);
  const int k = (int)kd;
  // r = z - k*ln2/128, with k*LN2N_HI exact (35-bit LN2N_HI, |k| < 2^17)
  dd s = two_sum(zh, -kd * OR_LN2N_HI);
  const double rl = s.lo + (zl - kd * OR_LN2N_LO);
  dd r = fast_two_sum(s.hi, rl);
  const double rh = r.hi;
  double q = 1.0 / 5040.0;
  q = 1.0 / 720.0 + rh * q;
  q = 1.0 / 120.0 + rh * q;
  q = 1.0 / 24.0 + rh * q;
  q = 1.0 / 6.0 + rh * q;
  q = 0.5 + rh * q;
  const double poly = rh * rh * q;
  dd er = fast_two_sum(1.0, rh);
  er.lo = er.lo + (r.lo + poly);
  const int j = k & 127;
  const int sc = (k - j) / 128;
  dd tj = {tab.ex(j, 0), tab.ex(j, 1)};
  dd pr = two_prod(tj.hi, er.hi);
  pr.lo = pr.lo + (tj.hi * er.lo + tj.lo * er.hi);
  double res = pr.hi + pr.lo;
  // scale by 2^sc (the result stays normal on this domain)
  int64_t eb = (int64_t)(1023 + sc) << 52;
  double two_sc;
  __builtin_memcpy(&two_sc, &eb, 8);
  return res * two_sc;
}

// ---- the short evaluation and its rounding test ----
// Bound on |short value - exact value| + |double-double value - exact value|: absolute for
// log, relative to the unscaled result (in [1, 2)) for exp.  The terms left out or rounded
// sum to less than 2^-68.2 (log: t^8/8 at |t| < 2^-8.5 is 2^-71, t^2 q in double 2^-70;
// exp: r^7/5040 at |r| < 2^-8.5 is 2^-72, T*plo in double 2^-70; pow adds |y| times the
// logarithm's, with |y| <= 1).
constexpr double kFastErr = 0x1p-67;

// ln(x) as u + lo, |lo| < 2^-17, x finite > 0 and normal.
template <class T = GlobalTab>
__host__ __device__ __forceinline__ dd log_fast(double x, const T tab = T{}) {
  int64_t bits;
  __builtin_memcpy(&bits, &x, 8);
  int e = (int)((bits >> 52) & 0x7ff) - 1023;
  int64_t mb = (bits & 0x000fffffffffffffLL) | 0x3ff0000000000000LL;
  double m;
  __builtin_memcpy(&m, &mb, 8);
  if (m >= 1.5) { m = 0.5 * m; e += 1; }
  const int i = (int)rint((m - 0.75) * 256.0);
  const double r = tab.lg(i, 0), t_hi = tab.lg(i, 1), t_lo = tab.lg(i, 2);
  const double p = m * r;
  const dd t = fast_two_sum(p - 1.0, fma(m, r, -p));
  const double t2 = t.hi * t.hi;
  const double q = fma(t2, fma(t2, fma(t.hi, 1.0 / 7.0, -1.0 / 6.0), fma(t.hi, 1.0 / 5.0, -1.0 / 4.0)),
                       fma(t.hi, 1.0 / 3.0, -0.5));
  const double ed = (double)e;
  const dd s = fast_two_sum(ed * OR_LN2_HI, t_hi); // |e ln2| >= |t_hi|, or e = 0
  const dd u = fast_two_sum(s.hi, t.hi);          // |s| >= |t|, or s = 0
  return {u.hi, fma(t2, q, u.lo + (s.lo + (t.lo + fma(ed, OR_LN2_LO, t_lo))))};
}

// exp(zh + zl), |zl| < 2^-16, |zh| < 708; false when the result may round either way.
template <class T = GlobalTab>
__host__ __device__ __forceinline__ bool exp_fast(double zh, double zl, double &res, const T tab = T{}) {
  const double kd = rint(zh * OR_INVLN2N);
  const int k = (int)kd;
  const double rh = fma(-kd, OR_LN2N_HI, zh); // exact
  const double rl = fma(-kd, OR_LN2N_LO, zl);
  const double r = rh + rl;
  const double r2 = r * r;
  const double q = fma(r2, fma(r2, 1.0 / 720.0, fma(r, 1.0 / 120.0, 1.0 / 24.0)), fma(r, 1.0 / 6.0, 0.5));
  const double plo = fma(r2, q, rl);
  const int j = k & 127;
  const int sc = (k - j) / 128;
  const double th = tab.ex(j, 0), tl = tab.ex(j, 1);
  const double ph = th * rh;
  const dd hi = fast_two_sum(th, ph);
  const double lo = fma(th, plo, fma(tl, rh, tl)) + (fma(th, rh, -ph) + hi.lo);
  const double a = hi.hi + (lo - 2.0 * kFastErr), b = hi.hi + (lo + 2.0 * kFastErr);
  int64_t eb = (int64_t)(1023 + sc) << 52;
  double two_sc;
  __builtin_memcpy(&two_sc, &eb, 8);
  res = a * two_sc;
  return a == b;
}

// The short evaluations of log, exp and pow; false when the double-double path must decide.
template <class T = GlobalTab>
__host__ __device__ __forceinline__ bool try_log(double x, double &res, const T tab = T{}) {
  const dd l = log_fast(x, tab);
  res = l.hi + (l.lo - kFastErr);
  return res == l.hi + (l.lo + kFastErr);
}
template <class T = GlobalTab>
__host__ __device__ __forceinline__ bool try_pow_from_log(double y, dd l, double &res, const T tab = T{}) {
  const double zh = y * l.hi;
  if (!(y >= -1.0 && y <= 1.0) || y == 0.0 || !(zh > -700.0 && zh < 700.0)) return false;
  return exp_fast(zh, fma(y, l.hi, -zh) + y * l.lo, res, tab);
}
// FAST, of the functions below: the short evaluation is tried first.  The host build keeps to the
// double-double path unless it asks for the device's.
#if defined(__HIP_DEVICE_COMPILE__)
constexpr bool kTryFast = true;
#else
constexpr bool kTryFast = false;
#endif

// smallest normal and largest finite double
constexpr double kMinNormal = 0x1.0p-1022;
constexpr double kMaxFinite = 0x1.fffffffffffffp+1023;

template <class T = GlobalTab, bool FAST = kTryFast>
__host__ __device__ inline double or_log(double x, const T tab = T{}) {
  if (!(x >= kMinNormal && x <= kMaxFinite)) return log(x);
  double f;
  if (FAST && try_log(x, f, tab)) return f;
  // the rare path reads the constant arrays: through the shells' copy in LDS it costs them registers
  // that spill (28 bytes a lane)
  dd l = log_dd(x);
  return l.hi + l.lo;
}

template <class T = GlobalTab, bool FAST = kTryFast>
__host__ __device__ inline double or_exp(double z, const T tab = T{}) {
  if (!(z > -708.0 && z < 708.0)) return exp(z);
  double f;
  if (FAST && exp_fast(z, 0.0, f, tab)) return f;
  return exp_dd(z, 0.0, tab);
}

template <class T = GlobalTab, bool FAST = kTryFast>
__host__ __device__ inline double or_pow(double x, double y, const T tab = T{}) {
  if (x == 0.0 && y > 0.0) return 0.0;
  if (y == 0.0 || x == 1.0) return 1.0;
  if (!(x >= kMinNormal && x <= kMaxFinite) || !(y >= -kMaxFinite && y <= kMaxFinite)) return pow(x, y);
  double f;
  if (FAST && try_pow_from_log(y, log_fast(x, tab), f, tab)) return f;
  dd l = log_dd(x, tab);
  dd z = two_prod(y, l.hi);
  z.lo = z.lo + y * l.lo;
  z = fast_two_sum(z.hi, z.lo);
  if (!(z.hi > -708.0 && z.hi < 708.0)) return pow(x, y);
  return exp_dd(z.hi, z.lo, tab);
}

// x**y1 and x**y2 from one logarithm of x: the same two results as or_pow(x, y1) and
// or_pow(x, y2), for half the cost of the logarithms when the bases agree.
template <class T = GlobalTab>
__host__ __device__ inline double pow_from_log(double x, double y, dd l, const T tab = T{}) {
  if (y == 0.0) return 1.0;
  if (!(y >= -kMaxFinite && y <= kMaxFinite)) return pow(x, y);
  dd z = two_prod(y, l.hi);
  z.lo = z.lo + y * l.lo;
  z = fast_two_sum(z.hi, z.lo);
  if (!(z.hi > -708.0 && z.hi < 708.0)) return pow(x, y);
  return exp_dd(z.hi, z.lo, tab);
}
template <class T = GlobalTab, bool FAST = kTryFast>
__host__ __device__ inline void or_pow2(double x, double y1, double y2, double &r1, double &r2,
                                        const T tab = T{}) {
  if (!(x >= kMinNormal && x <= kMaxFinite) || x == 1.0) {
    r1 = or_pow<T, FAST>(x, y1, tab);
    r2 = or_pow<T, FAST>(x, y2, tab);
    return;
  }
  if (FAST) {
    const dd l = log_fast(x, tab);
    const bool ok1 = try_pow_from_log(y1, l, r1, tab), ok2 = try_pow_from_log(y2, l, r2, tab);
    if (ok1 && ok2) return;
  }
  const dd l = log_dd(x, tab);
  r1 = pow_from_log(x, y1, l, tab);
  r2 = pow_from_log(x, y2, l, tab);
}

} // namespace ormath
