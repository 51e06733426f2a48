// FP64 2^x and log2 for the chemistry kernels, with a fixed, documented
// operation count (used by the FLOP accounting of the roofline).
//
// Rate constants are evaluated in base 2, k = A 2^(b log2 T + e log2(e) / (R T)):
// the reduction of the exponent to an integer and a fraction is then exact
// without the two-part product with ln 2 that base e needs: 15 instructions
// instead of 24, of which the right-hand side of GRI-3.0 has 13 per lane.  With
// both directions of a fall-off reaction in one pass (prodrates_wave) its wave
// evaluation went from 1,165 to 801 VALU instructions, and the guided step of
// 491,520 GRI-3.0 cells, which VALU issue bounds, from 347 to 306 ms.  Against
// 64-bit evaluation in another order the rates are as far off as before
// (3e-16 to 3e-15 of their norm).
//
// fexp2: k = rint(x), r = x - k (exact), 2^r on |r| <= 1/2 by a degree-11
//   polynomial 1 + r q(r), q interpolating (2^r - 1) / r at the Chebyshev points
//   (relative error 2e-17, mostly the rounding of the ln 2 coefficient),
//   result 2^k p by ldexp.
//   Finite x under- and overflow to 0 and +inf as they should, NaN propagates,
//   +-inf gives NaN (the exponents here are sums of finite terms; a rate at
//   T = 0 is undefined in any case).  Ops: 1 rint, 1 sub, 11 fma, 1 ldexp.
// flog2: x = 2^e m with m in [sqrt(1/2), sqrt(2)) (frexp); with f = m - 1 and
//   s = f/(1 + m), log2 m = (2 / ln 2) atanh(s) = s P(s^2), |s| <= 0.1716, P the
//   degree-7 interpolant at the Chebyshev points of [0, 0.0295] (relative
//   error 2e-18).  Arguments that are not positive and finite give NaN: they
//   have no rate constant, and Pr = 0 has none either (its log10 Pr = -inf makes
//   the Troe blending -inf / +inf).  Ops: 2 frexp, 1 ldexp, 2 add, 1 div, 1 mul,
//   8 fma.
#pragma once
#include "wave_target.h"

namespace tgr {

// Operation counts in the FLOP convention of the roofline (add, sub, mul,
// div, rint, ldexp, frexp = 1 flop; fma = 2 flops; compares and selects = 0).
constexpr double kFlopsExp = 1 + 1 + 11 * 2 + 1;           // 25
constexpr double kFlopsLog = 2 + 1 + 2 + 1 + 1 + 8 * 2;    // 23

constexpr double kLog2e = 1.4426950408889634074;
constexpr double kLn2 = 0.69314718055994530942;

// nearest integer of k as the hardware converts it: out of range saturates
__host__ __device__ __forceinline__ int sat_int(double k) {
#if defined(__HIP_DEVICE_COMPILE__)
  int i;
  asm("v_cvt_i32_f64 %0, %1" : "=v"(i) : "v"(k));
  return i;
#else
  return k >= 2147483647.0 ? 2147483647 : (k <= -2147483648.0 ? -2147483647 - 1 : (k == k ? (int)k : 0));
#endif
}

__host__ __device__ __forceinline__ double fexp2(double x) {
  const double k = rint(x);
  const double r = x - k;
  double p = 4.4549605981865186e-10;
  p = fma(p, r, 7.072585949269223e-09);
  p = fma(p, r, 1.0178062445845774e-07);
  p = fma(p, r, 1.321544258792169e-06);
  p = fma(p, r, 1.525273382983612e-05);
  p = fma(p, r, 0.0001540353044173605);
  p = fma(p, r, 0.0013333558146416936);
  p = fma(p, r, 0.009618129107606888);
  p = fma(p, r, 0.0555041086648216);
  p = fma(p, r, 0.24022650695910097);
  p = fma(p, r, 0.6931471805599453);
  p = fma(p, r, 1.0);
  return ldexp(p, sat_int(k));
}

__host__ __device__ __forceinline__ double flog2(double x) {
  int e;
  double m = frexp(x, &e);  // m in [0.5, 1)
  const int lo = m < 0.70710678118654752440 ? 1 : 0;
  m = ldexp(m, lo);
  e -= lo;
  const double s = (m - 1.0) / (m + 1.0);
  const double z = s * s;
  double p = 0.2136589569431927;
  p = fma(p, z, 0.2209130842311768);
  p = fma(p, z, 0.262334352504183);
  p = fma(p, z, 0.32059853491395984);
  p = fma(p, z, 0.4121985858409005);
  p = fma(p, z, 0.5770780163455203);
  p = fma(p, z, 0.9617966939259898);
  p = fma(p, z, 2.8853900817779268);
  const double y = fma(s, p, (double)e);
  return x > 0.0 && x < INFINITY ? y : NAN;
}

}  // namespace tgr
