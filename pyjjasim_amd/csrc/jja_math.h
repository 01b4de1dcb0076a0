// jja_math.h -- double-precision sine and the parts of the Box-Muller transform for
// the step kernels, usable on host and device (host builds test them against the C
// library).
//
// What bounds the junction pass is the number of vector instructions: all but the
// reciprocals take the same four cycles of a wave, so a register move or a select
// costs as much as a fused multiply-add. Hence no branches (lanes take both sides),
// no classification of arguments that cannot occur, and constants read from scalar
// registers (JJA_K) instead of being moved into vector registers.
//
// Method (published, not derived from any GPU vendor library):
//   sine: argument reduction  x = n*(pi/2) + r. n = rint(x*2/pi) is formed by adding
//     1.5*2^52, which leaves n's low bits in the low word; pi/2 is split into P1 + P2
//     (P1 = pi/2 rounded to double). rh = x - n*P1 by one FMA is exact: whenever
//     n != 0 both terms are multiples of 2^-53 and the difference is below one. The
//     small term n*P2 is subtracted with one rounding, whose error is kept as a tail
//     rl. Accurate for |x| up to about 1e15; beyond, the neglected n*P3 term grows
//     like 1e-33 |x|.
//   kernels on |r| <= pi/4: the sine and cosine polynomials of Sun's fdlibm
//     (coefficients below), both evaluated by fused multiply-adds with the tail rl as
//     a first-order correction; the quadrant picks one.
//   sine and cosine of a fraction of a turn: the quarter turn nearest to it is
//     subtracted exactly.
//   -log(u): u = 2^k m, m in [sqrt(1/2), sqrt(2)), s = (m - 1) / (m + 1) with its
//     rounding error, log m = 2 atanh(s) by a polynomial fitted to Chebyshev nodes
//     (relative error 5e-18), summed with k log 2 without losing the sum's error.
// Measured against glibc (tests/test_jja_math.py, tests/test_box_muller.py): the sine
// at most 1 ulp for |x| <= 1e9; near the zeros k*pi/2, where the result is tiny, the
// absolute error stays below 1e-24; -log(u) at most 1 ulp.
//
// The polynomial coefficients of jja_ksin and jja_kcos are those of fdlibm's k_sin.c
// and k_cos.c, which carry this notice:
//
//   Copyright (C) 1993 by Sun Microsystems, Inc. All rights reserved.
//
//   Developed at SunPro, a Sun Microsystems, Inc. business.
//   Permission to use, copy, modify, and distribute this
//   software is freely granted, provided that this notice
//   is preserved.
#ifndef JJA_MATH_H
#define JJA_MATH_H

#include <math.h>
#include <stdint.h>
#include <string.h>

#if defined(__HIPCC__)
#define JJA_HD __host__ __device__ __forceinline__
#else
#define JJA_HD static inline
#endif

// A constant kept in a scalar register.
JJA_HD double JJA_K(double c) {
#if defined(__HIP_DEVICE_COMPILE__)
  __asm__("" : "+s"(c));
#endif
  return c;
}

JJA_HD uint64_t jja_bits(double x) {
  uint64_t b;
  memcpy(&b, &x, sizeof(b));
  return b;
}
JJA_HD double jja_from_bits(uint64_t b) {
  double x;
  memcpy(&x, &b, sizeof(x));
  return x;
}

// What the sine and cosine of x + y share (|x| <= pi/4, |y| << ulp(x)).
typedef struct {
  double x, y, z, h, w;  // z = x^2, h = z / 2, w = 1 - h
} jja_arg;

JJA_HD jja_arg jja_make_arg(double x, double y) {
  jja_arg a;
  a.x = x;
  a.y = y;
  a.z = x * x;
  a.h = 0.5 * a.z;
  a.w = 1.0 - a.h;
  return a;
}

JJA_HD double jja_ksin(jja_arg a) {
  double p = a.z * JJA_K(1.58969099521155010221e-10);
  p = p + JJA_K(-2.50507602534068634195e-08);
  p = fma(a.z, p, JJA_K(2.75573137070700676789e-06));
  p = fma(a.z, p, JJA_K(-1.98412698298579493134e-04));
  p = fma(a.z, p, JJA_K(8.33333333332248946124e-03));
  p = fma(a.z, p, JJA_K(-1.66666666666666324348e-01));
  return a.x + fma(a.x, a.z * p, a.y * a.w);
}

JJA_HD double jja_kcos(jja_arg a) {
  double p = a.z * JJA_K(-1.13596475577881948265e-11);
  p = p + JJA_K(2.08757232129817482790e-09);
  p = fma(a.z, p, JJA_K(-2.75573143513906633035e-07));
  p = fma(a.z, p, JJA_K(2.48015872894767294178e-05));
  p = fma(a.z, p, JJA_K(-1.38888888888741095749e-03));
  p = fma(a.z, p, JJA_K(4.16666666666666019037e-02));
  return a.w + (((1.0 - a.w) - a.h) + fma(a.z, a.z * p, -(a.x * a.y)));
}

// x = q * pi/2 + the returned argument; q: quadrant (its low two bits count)
JJA_HD jja_arg jja_reduce(double x, uint32_t* q) {
  const double kMagic = JJA_K(6755399441055744.0);  // 1.5 * 2^52
  const double kP2 = JJA_K(6.12323399573676603587e-17);  // pi/2 - P1 rounded to double
  const double t = fma(x, JJA_K(6.36619772367581382433e-01), kMagic);
  const double n = t - kMagic;
  *q = (uint32_t)jja_bits(t);
  const double rh = fma(-n, JJA_K(1.57079632679489655800e+00), x);  // P1: pi/2 rounded to double
  const double r = fma(-n, kP2, rh);
  return jja_make_arg(r, fma(-n, kP2, rh - r));
}

// x, with its sign changed where bit 1 of q is set
JJA_HD double jja_flip(double x, uint32_t q) {
  return jja_from_bits(jja_bits(x) ^ ((uint64_t)((q << 30) & 0x80000000u) << 32));
}

JJA_HD double jja_sin(double x) {
  uint32_t q;
  const jja_arg a = jja_reduce(x, &q);
  const double s = jja_ksin(a), c = jja_kcos(a);
  return jja_flip((q & 1u) ? c : s, q);
}

// sin and cos of the argument a in quadrant q
JJA_HD void jja_quadrant(jja_arg a, uint32_t q, double* sn, double* cs) {
  const double s = jja_ksin(a), c = jja_kcos(a);
  *sn = jja_flip((q & 1u) ? c : s, q);
  *cs = jja_flip((q & 1u) ? s : c, q + 1u);
}

// sin(x) and cos(x) with one shared argument reduction (same method and accuracy as
// jja_sin; cos(x) = sin(x + pi/2) is quadrant n + 1).
JJA_HD void jja_sincos(double x, double* sn, double* cs) {
  uint32_t q;
  const jja_arg a = jja_reduce(x, &q);
  jja_quadrant(a, q, sn, cs);
}

// sin and cos of u turns, 0 <= u < 1
JJA_HD void jja_sincos_turn(double u, double* sn, double* cs) {
  const double kMagic = JJA_K(6755399441055744.0), kTwoPi_ = JJA_K(6.283185307179586);
  const double t = fma(u, 4.0, kMagic);
  const double f = fma(t - kMagic, -0.25, u);  // exact: within 1/8
  const double r = f * kTwoPi_;
  const double rl = fma(f, JJA_K(2.4492935982947064e-16), fma(f, kTwoPi_, -r));
  jja_quadrant(jja_make_arg(r, rl), (uint32_t)jja_bits(t), sn, cs);
}

// -log(u) for a normal u, 0 < u <= 1
JJA_HD double jja_neg_log(double u) {
  // the exponent that leaves m in [sqrt(1/2), sqrt(2)), by the high word
  const uint32_t kTop = 0x3fe6a09eu;  // that of sqrt(1/2)
  const uint64_t b = jja_bits(u);
  const uint32_t h = (uint32_t)(b >> 32) + (0x3ff00000u - kTop);
  const double m = jja_from_bits((uint64_t)((h & 0xfffffu) + kTop) << 32 | (uint32_t)b);
  const double k = (double)((int32_t)(h >> 20) - 0x3ff);
  const double f = m - 1.0, d = m + 1.0, dl = m - (d - 1.0);  // m + 1 = d + dl
#if defined(__HIP_DEVICE_COMPILE__)
  // the reciprocal to half the bits and one Newton step: the quotient's residual
  // below corrects what is left
  double r = __builtin_amdgcn_rcp(d);
  r = fma(fma(-d, r, 1.0), r, r);
#else
  const double r = 1.0 / d;
#endif
  const double s = f * r;
  const double sl = fma(-s, dl, fma(-d, s, f)) * r;  // (m - 1) / (m + 1) = s + sl
  const double z = s * s;
  double p = z * JJA_K(0.146167211662876);
  p = p + JJA_K(0.15331699634642276);
  p = fma(z, p, JJA_K(0.1818288978615799));
  p = fma(z, p, JJA_K(0.22222211125723262));
  p = fma(z, p, JJA_K(0.28571428626031065));
  p = fma(z, p, JJA_K(0.3999999999989938));
  p = fma(z, p, JJA_K(0.666666666666667));
  // log u = k log2 + 2 s + tail; k log2's first part (41 bits) is exact
  const double kh = k * JJA_K(0.693147180559663), s2 = s + s;
  const double tail = fma(s, z * p, fma(k, JJA_K(2.8235290563031577e-13), sl + sl));
  const double sum = kh + s2;  // |kh| > |s2| unless k = 0, so this loses (kh - sum) + s2
  return -(sum + (((kh - sum) + s2) + tail));
}

#endif  // JJA_MATH_H
