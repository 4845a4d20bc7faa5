// exp, tanh and the logistic function of a binary32 argument, evaluated in binary64 and rounded
// once to binary32 as the reference does ((float)StrictMath.exp((double)t) and so on,
// CpuScalarReferenceKernel.java:1213-1217,1736-1737), without the library functions' handling of
// binary64's own range: a binary32 argument needs neither subnormal binary64 results nor a
// reduction that holds beyond |t| = 120.
//
// What bounds them on the GPU is the number of binary64 instructions (as many a cycle as binary32
// ones). The library's exp is 43 vector instructions and its tanh 167, a whole table's activation
// costing several times the memory traffic around it; these are about 24 and 39. An elementwise
// chain of 20000 x 1001 that ends in tanh went from 225 to 186 us on MI355X, a 3001 x 1531 x 2047
// layer with tanh, forward and backward, from 916 to 890 us; the results are the same bits.
//
// Method (Cody and Waite, "Software Manual for the Elementary Functions", 1980):
//   t = n ln2 + r, n = rint(t / ln2), |r| <= 0.3466; ln2 = H + L in two binary64 parts, so that
//   r is formed by two FMAs with an absolute error below 2^-54; exp(r) - 1 = r + r^2 Q(r), Q the
//   Taylor polynomial to r^11 / 13! (the first term left out, r^14 / 14!, is below 2^-57), which
//   keeps the relative error of exp(r) - 1 near 2^-52 for small r as well.
//   exp(t)     = 2^n + 2^n (exp(r) - 1), one FMA;
//   tanh(|t|)  = -E / (2 + E) with E = exp(-2 |t|) - 1 = 2^n (exp(r) - 1) + (2^n - 1);
//   sigmoid(t) = 1 / (1 + e) for t >= 0 and e / (1 + e) below, e = exp(-|t|): the stable form.
// The quotients have denominators in [1, 2]: a hardware reciprocal, one Newton step and a
// residual correction. The binary64 results are within a few units of 2^-52, so the rounding to
// binary32 differs from the exactly rounded value only when that lies within that distance of a
// tie (about one argument in 10^7).
//
// Plain C++ but for the reciprocal, so that the host tests can compare it with the library.
#pragma once
#include <stdint.h>
#include <string.h>
#include <math.h>

namespace shk {

struct ExpParts {
  double p;      // exp(r) - 1
  double scale;  // 2^n
};

// Of x in [-120, 120].
__host__ __device__ inline ExpParts exp_parts(double x) {
  const double kLog2e = 0x1.71547652b82fep+0;  // binary64(1 / ln 2)
  const double kLn2Hi = 0x1.62e42fefa39efp-1;  // H = binary64(ln 2)
  const double kLn2Lo = 0x1.abc9e3b39803fp-56; // L = binary64(ln 2 - H)
  const double kShift = 0x1.8p52;              // adding it rounds to an integer
  const double kd = fma(x, kLog2e, kShift);
  const double n = kd - kShift;                // exact
  double r = fma(-n, kLn2Hi, x);
  r = fma(-n, kLn2Lo, r);
  double q = 1.0 / 6227020800.0;               // 1/13!
  q = fma(q, r, 1.0 / 479001600.0);            // 1/12!
  q = fma(q, r, 1.0 / 39916800.0);
  q = fma(q, r, 1.0 / 3628800.0);
  q = fma(q, r, 1.0 / 362880.0);
  q = fma(q, r, 1.0 / 40320.0);
  q = fma(q, r, 1.0 / 5040.0);
  q = fma(q, r, 1.0 / 720.0);
  q = fma(q, r, 1.0 / 120.0);
  q = fma(q, r, 1.0 / 24.0);
  q = fma(q, r, 1.0 / 6.0);
  q = fma(q, r, 0.5);                          // 1/2!
  ExpParts e;
  e.p = fma(r * r, q, r);
  uint64_t kb;                                 // the low half of kd's pattern holds n
  memcpy(&kb, &kd, 8);
  const uint64_t sb = (uint64_t)(((uint32_t)kb + 1023u) << 20) << 32;
  memcpy(&e.scale, &sb, 8);
  return e;
}

// n / d for d in [1, 2] and |n| <= 1.
__host__ __device__ inline double quotient_12(double n, double d) {
#if defined(__HIP_DEVICE_COMPILE__)
  double y = __builtin_amdgcn_rcp(d);
  y = fma(fma(-d, y, 1.0), y, y);
  const double q = n * y;
  return fma(fma(-d, q, n), y, q);
#else
  return n / d;
#endif
}

// t in [lo, hi] (a NaN gives one of the two: the callers put it back).
__host__ __device__ inline float clamp_f(float t, float lo, float hi) {
  return fminf(fmaxf(t, lo), hi);
}

// (float)exp((double)t). Beyond the clamp the result is 0 or +inf either way.
__host__ __device__ inline float exp_rn(float t) {
  const ExpParts e = exp_parts((double)clamp_f(t, -110.0f, 90.0f));
  const float v = (float)fma(e.p, e.scale, e.scale);
  return t != t ? t : v;
}

// (float)tanh((double)t): odd, the sign of a zero kept; +-1 from |t| = 9.1 on.
__host__ __device__ inline float tanh_rn(float t) {
  const ExpParts e = exp_parts(-2.0 * (double)fminf(fabsf(t), 20.0f));
  const double E = fma(e.p, e.scale, e.scale - 1.0);
  const float v = copysignf((float)quotient_12(-E, 2.0 + E), t);
  return t != t ? t : v;
}

// (float)(1 / (1 + exp(-t))) by its stable two branches.
__host__ __device__ inline float sigmoid_rn(float t) {
  const ExpParts p = exp_parts(-(double)fminf(fabsf(t), 110.0f));
  const double e = fma(p.p, p.scale, p.scale);
  const float v = (float)quotient_12(t >= 0.0f ? 1.0 : e, 1.0 + e);
  return t != t ? t : v;
}

}  // namespace shk
