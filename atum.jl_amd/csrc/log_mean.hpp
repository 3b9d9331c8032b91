// Logarithmic means of the box kernels: with f = (a-b)/(a+b), log_mean(a, b) = (a+b)/2 * f/atanh f.  The
// FAST kernels evaluate that; the reference-order ones the reference's own quotients (logavg of
// laws.hpp, src/numericalfluxes.jl:11-21), rounded as it rounds them, with a shorter logarithm.
#pragma once
#include "fast_flux.hpp"

namespace atm {

constexpr double LM_U = 0.01;  // the polynomials' range in u = f^2

// A constant in scalar registers (a literal is moved into vector registers at its use)
ATM_DEV double scalar(double c) {
  asm("" : "+s"(c));
  return c;
}

// f/atanh f and atanh(f)/f in u = f^2 <= LM_U: Chebyshev interpolants of degree 6 (3e-19 off)
ATM_DEV double lm_inverse(double u) {
#pragma clang fp contract(fast)
  double s = u * -0.017268601586902934 + -0.02179015140718188;
  s = s * u + -0.030194049011152555;
  s = s * u + -0.04656084640141071;
  s = s * u + -0.08888888888915485;
  s = s * u + -0.33333333333333315;
  return s * u + 1.0;
}
ATM_DEV double lm_direct(double u) {
#pragma clang fp contract(fast)
  double s = u * 0.07930082527176203 + 0.09087619619304513;
  s = s * u + 0.11111133605096339;
  s = s * u + 0.1428571420685783;
  s = s * u + 0.2000000000013155;
  s = s * u + 0.33333333333333254;
  return s * u + 1.0;
}
// log z for z outside [0.8, 1.2]: 2 atanh((m-1)/(m+1)) + k log 2, z = 2^k m, m in [sqrt 1/2, sqrt 2)
// (at most 2 ulps off, 0.41 rms; the library's log takes 99 instructions and more registers than the
// rest of the kernel, this one 30).  Zero, infinity, negatives and NaN as log.
ATM_DEV double lm_log(double z) {
#pragma clang fp contract(fast)
  double m = __builtin_amdgcn_frexp_mant(z);
  int k = __builtin_amdgcn_frexp_exp(z);
  const bool lo = m < 0.70710678118654752;
  m = lo ? 2 * m : m;
  k = lo ? k - 1 : k;
  const double d = m - 1, s = m + 1;
  const double f = fast_div(d, s, fast_rcp(s));
  const double u = f * f, t = 2 * f, kd = k;
  double q = u * scalar(0.07404933786156531) + scalar(0.0765625655736915);
  q = q * u + scalar(0.09091816120808513);
  q = q * u + scalar(0.11111098523202137);
  q = q * u + scalar(0.1428571438036914);
  q = q * u + scalar(0.19999999999650955);
  q = q * u + scalar(0.33333333333333826);
  const double r = kd * 0.693147180559663 + ((kd * 2.8235290563031577e-13 + t) + t * u * q);
  if (z > 0 && z < HUGE_VAL) return r;
  return z == 0 ? -HUGE_VAL : (z > 0 ? z : __builtin_nan(""));
}
// atanh(f)/f = log(a/b) / 2f for a and b that far apart, f = (a-b)/(a+b)
ATM_DEV double lm_far(double a, double b) {
  const double d = a - b, s = a + b, z = fast_div(a, b, fast_rcp(b)), h = 2 * fast_div(d, s, fast_rcp(s));
  const double l = lm_log(z);
  return fast_div(l, h, fast_rcp(h));
}

// f/atanh f and atanh(f)/f of a and b, f = (a-b)/(a+b), u = f^2
ATM_DEV double lm_g(double a, double b, double u) { return u < LM_U ? lm_inverse(u) : fast_rcp(lm_far(a, b)); }
ATM_DEV double lm_f(double a, double b, double u) { return u < LM_U ? lm_direct(u) : lm_far(a, b); }

// (atanh(f)/f - 1) / u on u <= 0.0295 (|f| up to that of sqrt 2): the interpolant of degree 7 of atanh(f)/f
ATM_DEV double lm_tail(double u) {
#pragma clang fp contract(fast)
  double q = u * scalar(0.07404933786156531) + scalar(0.0765625655736915);
  q = q * u + scalar(0.09091816120808513);
  q = q * u + scalar(0.11111098523202137);
  q = q * u + scalar(0.1428571438036914);
  q = q * u + scalar(0.19999999999650955);
  return q * u + scalar(0.33333333333333826);
}
constexpr double LM_NEAR = 0.0294;

// log m - 2f for m in [sqrt 1/2, sqrt 2], f the rounded (m-1)/s, s the rounded m+1, is = fast_rcp(s), u = f^2:
// what the two roundings left out of f, and the terms from f^3 on.  The sum with 2f is
// the logarithm to 0.51 ulp.
ATM_DEV double lm_rest(double m, double s, double is, double f, double u) {
#pragma clang fp contract(fast)
  const double ds = m - (s - 1);  // m + 1 - s, exactly
  const double df = (fma(-f, s, m - 1) - f * ds) * is;
  const double t = 2 * f;
  return fma(t * u, lm_tail(u), 2 * df);
}

// log z of any z, to 0.51 ulp: k log 2 + log m.  Zero, infinity, negatives and NaN as log.
ATM_DEV double lm_log_far(double z) {
#pragma clang fp contract(off)
  double m = __builtin_amdgcn_frexp_mant(z);
  int k = __builtin_amdgcn_frexp_exp(z);
  const bool lo = m < 0.70710678118654752;
  m = lo ? 2 * m : m;
  k = lo ? k - 1 : k;
  const double s = m + 1, is = fast_rcp(s), f = fast_div(m - 1, s, is), t = 2 * f, kd = k;
  const double c = fma(kd, 2.8235290563031577e-13, lm_rest(m, s, is, f, f * f));
  const double hi = kd * 0.693147180559663;  // exact: the constant ends in 12 zero bits
  const double sum = hi + t;
  const double r = sum + ((hi - sum) + t + c);
  if (z > 0 && z < HUGE_VAL) return r;
  return z == 0 ? -HUGE_VAL : (z > 0 ? z : __builtin_nan(""));
}

// logavg(a0, b0) and logavg(a1, b1) of the reference.  Reciprocals are taken in pairs, of the
// product of the two means' divisors (the hardware's takes four times an FMA): good to 46 bits, which
// fast_div corrects.
ATM_DEV void lm_logavg2(double a0, double b0, double a1, double b1, double* m0, double* m1) {
#pragma clang fp contract(off)
  constexpr double EPS = 2.220446049250313e-16;
  const double ib = rcp_div(b0 * b1);
  const double z0 = fast_div(a0, b0, b1 * ib), z1 = fast_div(a1, b1, b0 * ib);
  const double s0 = z0 + 1, s1 = z1 + 1, is = rcp_div(s0 * s1), is0 = s1 * is, is1 = s0 * is;
  const double f0 = fast_div(z0 - 1, s0, is0), f1 = fast_div(z1 - 1, s1, is1);
  const double u0 = f0 * f0, u1 = f1 * f1;
  double l0, l1;
  if (u0 < LM_NEAR && u1 < LM_NEAR) {
    l0 = 2 * f0 + lm_rest(z0, s0, is0, f0, u0);
    l1 = 2 * f1 + lm_rest(z1, s1, is1, f1, u1);
  } else {
    l0 = lm_log_far(z0);
    l1 = lm_log_far(z1);
  }
  // below eps the reference's series in u is 1 after rounding: l/t with both 1
  const bool eq0 = u0 < EPS, eq1 = u1 < EPS;
  const double t0 = eq0 ? 1.0 : 2 * f0, t1 = eq1 ? 1.0 : 2 * f1;
  const double it = rcp_div(t0 * t1);
  const double F0 = 2 * fast_div(eq0 ? 1.0 : l0, t0, t1 * it), F1 = 2 * fast_div(eq1 ? 1.0 : l1, t1, t0 * it);
  const double iF = rcp_div(F0 * F1);
  *m0 = fast_div(a0 + b0, F0, F1 * iF);
  *m1 = fast_div(a1 + b1, F1, F0 * iF);
}

}  // namespace atm
