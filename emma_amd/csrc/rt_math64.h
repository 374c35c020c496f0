// rt_math64.h -- FP64 division and the logarithm / exponential pair of the
// FP64 rate fits.
//
// The FP64 chemistry is bound by its instructions and, in cells that take many
// sub-steps, by their latency.  Division: the compiler's IEEE sequence scales
// both operands and patches the special cases (11 instructions); the operands
// here are far from the range's ends, so the same two Newton steps and one
// residual correction without the scaling give the same correctly rounded
// quotient (operands and quotient within 2^-900 .. 2^900), and quotients by one
// divisor share its reciprocal.  div64 keeps the hardware's patch of the special
// cases: zeros, infinities and NaN divide as in IEEE arithmetic (64^3 cells with
// one group: 22.5 us a level step, 22.0 without the patch, 23.2 to 23.9 with
// plain divisions behind a test for NaN in its place).  quot64 leaves
// that out, for operands known to be ordinary or with a check of the result: a
// zero, infinite or denormal divisor, or an infinite numerator, gives NaN.
// Powers: the
// rate fits raise two numbers to six powers; pow() takes an extended-precision
// logarithm and a full range check each time.  Here a base's logarithm is taken once, as
// an unevaluated sum of two doubles good to about 2^-59, and products of
// powers are formed in the exponent and exponentiated once.
#pragma once

#include <hip/hip_runtime.h>

namespace emma {

// 1/b by the hardware estimate and two Newton steps
__device__ __forceinline__ double rcp64(double b) {
  double r = __builtin_amdgcn_rcp(b);
  r = fma(fma(-b, r, 1.0), r, r);
  r = fma(fma(-b, r, 1.0), r, r);
  return r;
}
// a/b correctly rounded, r = 1/b to about one ulp
__device__ __forceinline__ double quot64(double a, double b, double r) {
  const double q = a * r;
  return fma(fma(-q, b, a), r, q);
}
__device__ __forceinline__ double quot64(double a, double b) { return quot64(a, b, rcp64(b)); }
__device__ __forceinline__ double div64(double a, double b, double r) {
  return __builtin_amdgcn_div_fixup(quot64(a, b, r), b, a);
}
__device__ __forceinline__ double div64(double a, double b) { return div64(a, b, rcp64(b)); }

struct Dd {  // an unevaluated sum
  double h, l;
};

constexpr double kLn2Hi = 0x1.62e42fee00000p-1;  // ln 2 to 32 bits: k * kLn2Hi is exact
constexpr double kLn2Lo = 0x1.a39ef35793c76p-33;

// ln x, x > 0 and normal.  x = 2^k m, m in [1/sqrt 2, sqrt 2),
// s = (m - 1)/(m + 1) to twice the precision, ln m = 2 s + s^3 P(s^2) with
// the series' coefficients 2/3, 2/5, ... (the first left out is below 2^-60).
__device__ __forceinline__ Dd log_dd(double x) {
  double m = __builtin_amdgcn_frexp_mant(x);
  int k = __builtin_amdgcn_frexp_exp(x);
  const bool low = m < 0x1.6a09e667f3bcdp-1;
  m = low ? m + m : m;
  k = low ? k - 1 : k;
  const double f = m - 1., d = m + 1.;
  const double dl = m - (d - 1.);
  const double r = rcp64(d);
  const double s = f * r;
  const double sl = fma(-s, dl, fma(-s, d, f)) * r;
  const double z = s * s;
  double p = 2. / 21.;
  p = fma(p, z, 2. / 19.);
  p = fma(p, z, 2. / 17.);
  p = fma(p, z, 2. / 15.);
  p = fma(p, z, 2. / 13.);
  p = fma(p, z, 2. / 11.);
  p = fma(p, z, 2. / 9.);
  p = fma(p, z, 2. / 7.);
  p = fma(p, z, 2. / 5.);
  p = fma(p, z, 2. / 3.);
  const double t = s * z * p;
  const double a = (double)k * kLn2Hi, b = s + s;
  const double h0 = a + b;
  const double l0 = (b - (h0 - a)) + fma((double)k, kLn2Lo, fma(2., sl, t));
  Dd o;
  o.h = h0 + l0;
  o.l = l0 - (o.h - h0);
  return o;
}

// exp(h + l), h between about -800 and 700
__device__ __forceinline__ double exp_dd(double h, double l) {
  const double k = rint(h * 0x1.71547652b82fep+0);
  const double rh = fma(-k, kLn2Hi, h), rl = fma(-k, kLn2Lo, l);
  const double x = rh + rl;
  const double xl = (rh - x) + rl;
  double p = 1. / 6227020800.;
  p = fma(p, x, 1. / 479001600.);
  p = fma(p, x, 1. / 39916800.);
  p = fma(p, x, 1. / 3628800.);
  p = fma(p, x, 1. / 362880.);
  p = fma(p, x, 1. / 40320.);
  p = fma(p, x, 1. / 5040.);
  p = fma(p, x, 1. / 720.);
  p = fma(p, x, 1. / 120.);
  p = fma(p, x, 1. / 24.);
  p = fma(p, x, 1. / 6.);
  p = fma(p, x, 0.5);
  return ldexp(1. + (x + fma(x * x, p, xl)), (int)k);
}
__device__ __forceinline__ double exp64(double x) { return exp_dd(fmax(x, -800.), 0.); }

__device__ __forceinline__ Dd dd_scale(double y, Dd a) {
  Dd o;
  o.h = y * a.h;
  o.l = fma(y, a.h, -o.h) + y * a.l;
  return o;
}
__device__ __forceinline__ Dd dd_sub(Dd a, Dd b) {
  Dd o;
  o.h = a.h - b.h;
  const double bb = o.h - a.h;
  o.l = ((a.h - (o.h - bb)) - (b.h + bb)) + (a.l - b.l);
  return o;
}
__device__ __forceinline__ double exp_of(Dd a) { return exp_dd(a.h, a.l); }

}  // namespace emma
