// Stands in for hip/hip_runtime.h where a test compiles a device header for
// the host: the qualifiers, and the gfx950 instructions behind the builtins the
// FP64 physics uses, as the instruction set's manual gives them.
#pragma once
#include <math.h>
#include <stdint.h>
#include <string.h>

#define __device__
#define __forceinline__ inline

// v_rcp_f64 is good to 2^29 units in the last place: the reciprocal with a
// relative error of rcp_error (a test sets up to 2^-23 either way)
inline double rcp_error = 0.;
inline double __builtin_amdgcn_rcp(double b) { return 1. / b * (1. + rcp_error); }

// v_div_fixup_f64: the special cases of numerator / denominator
inline double __builtin_amdgcn_div_fixup(double quotient, double den, double num) {
  auto exponent = [](double x) {
    uint64_t u;
    memcpy(&u, &x, 8);
    return (int)(u >> 52 & 2047);
  };
  const double sign = signbit(num) != signbit(den) ? -1. : 1.;
  if (isnan(num)) return num;
  if (isnan(den)) return den;
  if (num == 0. && den == 0.) return NAN;
  if (isinf(num) && isinf(den)) return NAN;
  if (den == 0. || isinf(num)) return sign * INFINITY;
  if (isinf(den) || num == 0.) return sign * 0.;
  if (exponent(num) - exponent(den) < -1075) return sign * 0.;
  if (exponent(den) == 2047) return sign * INFINITY;
  return sign * fabs(quotient);
}

inline double __builtin_amdgcn_frexp_mant(double x) {
  int k;
  return frexp(x, &k);
}
inline int __builtin_amdgcn_frexp_exp(double x) {
  int k;
  frexp(x, &k);
  return k;
}
