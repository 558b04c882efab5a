// Nearly correctly rounded exp, log, log10 and pow in FP64 for the FP64 twin.
//
// The reference's FP64 build calls the host libm (glibc), whose exp, log and
// pow return the correctly rounded result in all but a tiny fraction of
// arguments.  The GPU's own libm is accurate to about one ulp, which differs
// from glibc in roughly one pow call in four and, through threshold
// branches, occasionally moves a column's result far more than an ulp.  These
// routines evaluate the function in double-double arithmetic with a relative
// error near 2^-77 and round once, so they agree with a correctly rounded
// libm except when the exact value lies within ~2^-77 relative of a rounding
// boundary.
//
// Methods (standard, from the literature):
//   error-free transformations two_sum / two_prod (Knuth; Dekker 1971, with
//   fused multiply-add for the product);
//   exp: Cody-Waite reduction by ln2/64 with a three-part constant, table of
//   2^(j/64) in double-double (Tang 1989), degree-8 Taylor polynomial whose
//   cubic and higher terms are summed in double;
//   log: frexp reduction to [1/sqrt2, sqrt2), a first approximation y from the
//   single-precision unit, corrected by the series of log1p(m e^-y - 1) with
//   e^-y in double-double;
//   pow: exp of y*log(x) with the product carried in double-double; whole
//   exponents known to the compiler by double-double products.
//
// Contraction is off in every function, so that the error-free
// transformations hold in the FP32 unit too.
//
// Everything here is straight-line code without a call: the step evaluates
// about a hundred of these per point, all inlined.  With the device libm's
// log for the first approximation and its exp, log and pow as the fallback
// for special arguments, each call site took several kilobytes and the FP64
// level physics 757 KB of code, which a compute unit's 64 KB instruction
// cache cannot hold: a single column waited 213 us in that kernel, most of
// it for instructions.  In this form it is 205 KB: by this alone a step of one
// column of 60 levels took 186 instead of 335 us, of 25,000 x 90 2.12 instead
// of 3.33 ms.  Special arguments (0, negative, infinite, NaN, 1) are a short
// block of selects, results near overflow or in the subnormal range come
// from the final scaling.
#pragma once

#include <hip/hip_runtime.h>

namespace tempo {
namespace crm {

#include "tempo_crmath_tables.inc"

struct dd {
  double hi, lo;
};

__device__ __host__ __forceinline__ dd two_sum(double a, double b) {
#pragma clang fp contract(off)
  const double s = a + b;
  const double bb = s - a;
  return {s, (a - (s - bb)) + (b - bb)};
}

__device__ __host__ __forceinline__ dd fast_two_sum(double a, double b) {  // |a| >= |b|
#pragma clang fp contract(off)
  const double s = a + b;
  return {s, b - (s - a)};
}

__device__ __host__ __forceinline__ dd two_prod(double a, double b) {
#pragma clang fp contract(off)
  const double p = a * b;
  return {p, fma(a, b, -p)};
}

// e^(zh + zl) = 2^k * (hi + lo) for |zh| <= 746, |zl| <= ulp(zh); kSmall:
// |zh| <= 0.35 and zl = 0 (the third part of the reduction's constant is then
// below 2^-85)
template <bool kSmall = false>
__device__ __host__ __forceinline__ dd exp_dd(double zh, double zl, int& k) {
#pragma clang fp contract(off)
  const double n = rint(zh * kInvLn2x64);
  const int ni = int(n);
  const double r1 = fma(-n, kLn2o64C1, zh);  // exact: n*c1 exact, Sterbenz
  const dd p2 = two_prod(n, kLn2o64C2);
  dd r = two_sum(r1, -p2.hi);
  r.lo = r.lo - p2.lo;
  if (!kSmall) r.lo = fma(-n, kLn2o64C3, r.lo) + zl;
  r = fast_two_sum(r.hi, r.lo);
  const int j = ni & 63;
  k = ni >> 6;
  const double x = r.hi;
  // e^x - 1 = x + x^2/2 + x^3 P(x), |x| <= ln2/128
  dd s = two_prod(x, x);
  s.hi *= 0.5;
  s.lo *= 0.5;
  const double P =
      fma(x, fma(x, fma(x, fma(x, fma(x, 1.0 / 40320.0, 1.0 / 5040.0), 1.0 / 720.0), 1.0 / 120.0), 1.0 / 24.0), 1.0 / 6.0);
  const dd a = fast_two_sum(x, s.hi);
  const double lo = fma(x * x * x, P, a.lo + s.lo) + fma(r.lo, x, r.lo);
  const dd pm1 = fast_two_sum(a.hi, lo);
  // 2^(j/64) * (1 + pm1)
  const double th = kExp2Tab[j][0], tl = kExp2Tab[j][1];
  const dd m1 = two_prod(th, pm1.hi);
  const double lo2 = tl + m1.lo + fma(th, pm1.lo, tl * pm1.hi);
  dd h = two_sum(th, m1.hi);
  h.lo += lo2;
  return fast_two_sum(h.hi, h.lo);
}

// log(x) = hi + lo for positive finite x: x = m 2^e with m in
// [1/sqrt2, sqrt2), y ~ log m from the single-precision unit (error near
// 2^-23), u = m e^-y - 1 in double-double, log m = y + log1p(u) with four
// terms of the series (u^5/5 < 2^-107 is dropped).
__device__ __host__ __forceinline__ dd log_dd(double x) {
#pragma clang fp contract(off)
  int e;
  double m = frexp(x, &e);
  if (m < 0.70710678118654752440) {
    m *= 2.0;
    e -= 1;
  }
#ifdef __HIP_DEVICE_COMPILE__
  const double y = double(__builtin_amdgcn_logf(float(m)) * 0.693147180559945309f);
#else
  const double y = double(logf(float(m)));
#endif
  int k;
  const dd E = exp_dd<true>(-y, 0.0, k);
  m = ldexp(m, k);
  const dd P = two_prod(m, E.hi);
  const double uh = P.hi - 1.0, ul = fma(m, E.lo, P.lo);  // P.hi - 1 is exact
  const double u = uh + ul;
  const double t = u * u * fma(u, fma(u, -0.25, 1.0 / 3.0), -0.5);
  const double ed = double(e);
  const dd h = two_sum(ed * kLn2Hi, y);
  const dd g = two_sum(h.hi, uh);
  return fast_two_sum(g.hi, g.lo + (h.lo + ((ul + t) + ed * kLn2Lo)));
}

// Results outside the normal range are formed by the final scaling (an
// argument past the clamps overflows to infinity or vanishes).
__device__ __host__ __forceinline__ double exp_cr(double x) {
#pragma clang fp contract(off)
  const double z = x > 710.0 ? 710.0 : (x < -746.0 ? -746.0 : x);
  int k;
  const dd r = exp_dd(z, 0.0, k);
  return ldexp(r.hi, k);  // r.hi is already the double nearest r.hi + r.lo
}

__device__ __host__ __forceinline__ bool positive_finite(double x) {
#pragma clang fp contract(off)
  return x > 0.0 && x <= 1.7976931348623157e308;
}

// log of 0, negative, infinite and NaN arguments, and of 1
__device__ __host__ __forceinline__ double log_special(double x) {
#pragma clang fp contract(off)
  return x == 1.0 ? 0.0 : x == 0.0 ? -__builtin_huge_val() : x > 0.0 ? x : __builtin_nan("");
}

__device__ __host__ __forceinline__ double log_cr(double x) {
#pragma clang fp contract(off)
  if (!positive_finite(x) || x == 1.0) return log_special(x);
  return log_dd(x).hi;
}

__device__ __host__ __forceinline__ double log10_cr(double x) {
#pragma clang fp contract(off)
  if (!positive_finite(x) || x == 1.0) return log_special(x);
  const dd l = log_dd(x);
  const dd p = two_prod(l.hi, kInvLn10Hi);
  const double lo = p.lo + l.hi * kInvLn10Lo + l.lo * kInvLn10Hi;
  return fast_two_sum(p.hi, lo).hi;
}

// pow where x is not a positive finite number other than 1, or y is zero,
// infinite or NaN: r = |x|**y as computed below, of use for negative x
__device__ __host__ __forceinline__ double pow_special(double x, double y, double r) {
#pragma clang fp contract(off)
  const double inf = __builtin_huge_val(), ax = fabs(x);
  if (x == 1.0 || y == 0.0) return 1.0;
  if (x != x || y != y) return x + y;
  const bool whole = rint(y) == y, odd = whole && fabs(y) < 9.0e15 && rint(0.5 * y) * 2.0 != y;
  if (fabs(y) == inf)
    r = ax == 1.0 ? 1.0 : ((ax > 1.0) == (y > 0.0) ? inf : 0.0);
  else if (ax == 0.0 || ax == inf)
    r = (ax == 0.0) == (y > 0.0) ? 0.0 : inf;
  else if (!whole)
    return __builtin_nan("");
  else if (ax == 1.0)
    r = 1.0;
  return odd ? copysign(r, x) : r;
}

// x^n for n = 1, 2, 3, 4, 5, 7, 8: products of the significand carried in
// double-double (relative error below 2^-100) and rounded once, as pow_cr
// rounds, at a tenth of its instructions.  The exponent goes in last, so that
// no product leaves the range in which its low part is exact; 0, infinities and
// NaN, whose low parts are none, take the plain product.
template <int n>
__device__ __host__ __forceinline__ dd pow_whole_dd(double x) {
#pragma clang fp contract(off)
  static_assert(n >= 1 && n <= 8, "small whole exponents");
  if constexpr (n == 1) return {x, 0.0};
  else if constexpr (n % 2 == 0) {
    const dd h = pow_whole_dd<n / 2>(x);
    const dd p = two_prod(h.hi, h.hi);
    return {p.hi, fma(2.0 * h.hi, h.lo, p.lo)};
  } else {
    const dd h = pow_whole_dd<n - 1>(x);
    const dd p = two_prod(h.hi, x);
    return {p.hi, fma(h.lo, x, p.lo)};
  }
}
template <int n>
__device__ __host__ __forceinline__ double pow_whole(double x) {
#pragma clang fp contract(off)
  int e;
  const double m = frexp(x, &e);
  const dd d = pow_whole_dd<(n < 0 ? -n : n)>(m);
  const bool in = fabs(d.hi) > 0.0 && fabs(d.hi) < 2.0;
  if constexpr (n < 0) {
    const double q = 1.0 / d.hi;
    const double r = fma(-q, d.hi, 1.0) - q * d.lo;
    return in ? ldexp(fma(q, r, q), n * e) : q;
  } else {
    return in ? ldexp(d.hi + d.lo, n * e) : d.hi;
  }
}

// x^(n + 1/2), and its inverse: the square root with its residual, times x^n,
// of the significand beside an even exponent
template <int n, bool kInverse = false>
__device__ __host__ __forceinline__ double pow_half(double x) {
#pragma clang fp contract(off)
  int e;
  double m = frexp(x, &e);
  const int half = e >> 1;
  m = ldexp(m, e - 2 * half);  // in [1/2, 2)
  const double s = sqrt(m);
  const double sl = fma(-s, s, m) * double(0.5f / float(s));
  const dd w = pow_whole_dd<n>(m);
  dd p = two_prod(w.hi, s);
  p.lo += fma(w.hi, sl, w.lo * s);
  const bool in = positive_finite(x);
  const int shift = half * (2 * n + 1);
  if (!kInverse) return in ? ldexp(p.hi + p.lo, shift) : w.hi * s;
  const double q = 1.0 / p.hi;
  return in ? ldexp(fma(q, fma(-q, p.hi, 1.0) - q * p.lo, q), -shift) : 1.0 / (w.hi * s);
}

// x^y for y = the double nearest 1/3 (1/3 - 1.85e-17): the cube root by
// Newton steps from the single-precision unit's first approximation, the
// last residual in double-double (relative error near 2^-95), times
// x^-1.85e-17 = 1 - 1.85e-17 log x.  Of use for positive finite x.
__device__ __host__ __forceinline__ dd pow_third_dd(double x, int& q) {
#pragma clang fp contract(off)
  int e;
  double m = frexp(x, &e);
  q = int(float(e + 1200) * (1.0f / 3.0f)) - 400;  // near e/3: m 2^(e - 3q) lies in [1/4, 8)
  m = ldexp(m, e - 3 * q);
#ifdef __HIP_DEVICE_COMPILE__
  const float l2 = __builtin_amdgcn_logf(float(m));
  const double y0 = double(__builtin_amdgcn_exp2f(l2 * (1.0f / 3.0f)));
  double rc = double(__builtin_amdgcn_rcpf(float(m)));
#else
  const float l2 = log2f(float(m));
  const double y0 = double(exp2f(l2 * (1.0f / 3.0f)));
  double rc = double(1.0f / float(m));
#endif
  rc = fma(rc, fma(-m, rc, 1.0), rc) * (1.0 / 3.0);  // 1/(3 m)
  const double r0 = fma(-(y0 * y0), y0, m) * rc;     // y0 has 24 bits: its square is exact
  const double y1 = fma(y0, fma(r0, -r0, r0), y0);   // error near 2^-53 (r0^3 is below it)
  const dd y2 = two_prod(y1, y1);
  const dd y3 = two_prod(y2.hi, y1);
  const double r1 = ((m - y3.hi) - fma(y2.lo, y1, y3.lo)) * rc;
  const double lnx = double((l2 + float(3 * q)) * 0.693147181f);
  return fast_two_sum(y1, y1 * fma(lnx, -1.850371707708594e-17, r1));
}

__device__ __host__ __forceinline__ double pow_cr(double x, double y) {
#pragma clang fp contract(off)
  // exponents known to the compiler
  if (__builtin_constant_p(y) && y == 1.0 / 3.0) {
    int q;
    const dd r = pow_third_dd(x, q);
    return positive_finite(x) ? ldexp(r.hi, q) : (x == 0.0 || x > 0.0 ? fabs(x) : __builtin_nan(""));
  }
  if (__builtin_constant_p(y)) {
    if (y == 1.0) return x;
    if (y == 2.0) return x * x;
    if (y == 3.0) return pow_whole<3>(x);
    if (y == 4.0) return pow_whole<4>(x);
    if (y == 7.0) return pow_whole<7>(x);
    if (y == 2.5) return pow_half<2>(x);
    if (y == 3.5) return pow_half<3>(x);
    if (y == 0.0) return 1.0;
    if (y == -3.5) return pow_half<3, true>(x);
    if (y == -3.0) return pow_whole<-3>(x);
    if (y == -4.0) return pow_whole<-4>(x);
    if (y == -5.0) return pow_whole<-5>(x);
    if (y == -7.0) return pow_whole<-7>(x);
  }
  const dd l = __builtin_constant_p(x) && x == 10.0 ? dd{kLn10Hi, kLn10Lo} : log_dd(fabs(x));
  const dd p = two_prod(y, l.hi);
  dd z = fast_two_sum(p.hi, fma(y, l.lo, p.lo));
  if (!(z.hi > -746.0 && z.hi < 710.0)) {
    z.hi = z.hi >= 710.0 ? 710.0 : (z.hi <= -746.0 ? -746.0 : z.hi);
    z.lo = 0.0;
  }
  int k;
  const dd r = exp_dd(z.hi, z.lo, k);
  const double v = ldexp(r.hi, k);
  if (!positive_finite(x) || x == 1.0 || y == 0.0 || !(fabs(y) < 1.0e300)) return pow_special(x, y, v);
  return v;
}

}  // namespace crm
}  // namespace tempo
