// pow64.h -- x^k in FP64 for x > 0, the |difference|^(q - p) of the qGGMRF
// potentials (device code of both libraries).
//
// Table-driven logarithm (P. T. P. Tang, "Table-driven implementation of the
// logarithm function in IEEE floating-point arithmetic", ACM TOMS 16, 1990)
// in base 2 and a polynomial 2^f:
//   x = 2^e m, m in [1/2, 1); i the top 7 bits of m's fraction, c the middle
//   of their interval, t[i] = (1/c rounded, -log2 of that); r = m t[i].x - 1,
//   |r| <= 2^-8, and log2 m = t[i].y + log2(1 + r) by its series to r^6
//   (the rest is below 2^-57);
//   k log2 x = n + f with n its nearest integer: f = (k e - n) + k log2 m,
//   formed with two fused multiply-adds, so that the part before the binary
//   point costs no digits of f; 2^f by its series to f^13 (rest below 2^-57).
// Against exp2(k * log2(x)), whose product rounds at the size of k log2 x,
// the largest error over x in [1e-12, 1e3], k in (0, 1] falls from 41 to
// 1.6 units in the last place, at about a third of the instructions.
#ifndef PHASECON_POW64_H
#define PHASECON_POW64_H
#include <cfloat>
#include <cmath>

constexpr int kPow64Tab = 128;

// Table entry i.
__host__ __device__ inline void pow64_entry(int i, double& inv, double& lg) {
  const double c = 0.5 + (i + 0.5) / 256.0;
  inv = 1.0 / c;
  lg = -log2(inv);
}

// log2(1 + r) / r for |r| <= 2^-8
__host__ __device__ inline double pow64_log(double r) {
  const double l = 1.4426950408889634074;  // log2 e
  double p = fma(r, -l / 6.0, l / 5.0);
  p = fma(p, r, -l / 4.0);
  p = fma(p, r, l / 3.0);
  p = fma(p, r, -l / 2.0);
  return fma(p, r, l);
}

// 2^f for |f| <= 1/2 (a little more does no harm): ln(2)^j / j!
__host__ __device__ inline double pow64_exp(double f) {
  double p = 1.3691488853904128881e-12;
  p = fma(p, f, 2.5678435993488205141e-11);
  p = fma(p, f, 4.4455382718708114976e-10);
  p = fma(p, f, 7.0549116208011233299e-9);
  p = fma(p, f, 1.0178086009239699728e-7);
  p = fma(p, f, 1.3215486790144309489e-6);
  p = fma(p, f, 1.5252733804059840280e-5);
  p = fma(p, f, 1.5403530393381609954e-4);
  p = fma(p, f, 1.3333558146428443424e-3);
  p = fma(p, f, 9.6181291076284771620e-3);
  p = fma(p, f, 5.5504108664821579953e-2);
  p = fma(p, f, 2.4022650695910071233e-1);
  p = fma(p, f, 6.9314718055994530942e-1);
  return fma(p, f, 1.0);
}

#ifdef __HIPCC__
// The table in LDS; a barrier before its first use is the caller's.
__device__ __forceinline__ void pow64_init(double2* t) {
  for (int i = threadIdx.x; i < kPow64Tab; i += blockDim.x) pow64_entry(i, t[i].x, t[i].y);
}

__device__ __forceinline__ double pow64(double x, double k, const double2* t) {
  if (!(x <= DBL_MAX)) return exp2(k * log2(x));  // infinity, NaN
  const double m = __builtin_amdgcn_frexp_mant(x);
  const double e = (double)__builtin_amdgcn_frexp_exp(x);
  const int i = (int)(__double2hiint(m) >> 13) & (kPow64Tab - 1);
  const double2 q = t[i];
  const double r = fma(m, q.x, -1.0);
  const double lm = fma(pow64_log(r), r, q.y);
  const double n = __builtin_rint(fma(k, lm, k * e));
  return ldexp(pow64_exp(fma(k, lm, fma(k, e, -n))), (int)n);
}
#endif
#endif
