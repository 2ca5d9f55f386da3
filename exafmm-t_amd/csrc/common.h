// Shared device-side definitions of the gfx950 FMM engine.
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>

namespace xfmm {

enum Kind { LAPLACE = 0, HELMHOLTZ = 1, YUKAWA = 2 };

constexpr double FOUR_PI_INV = 0.07957747154594766788;  // 1/(4 pi)
constexpr int NCHILD = 8;
constexpr int NM2L = 26;  // M2L relative positions of a target parent

template <typename R>
struct cplx {
  R x, y;
};

// Wave numbers as seen by the kernels.  Laplace ignores both, modified
// Helmholtz (Yukawa) uses re, Helmholtz uses re + i im.
struct Wavek {
  double re, im;
};

__device__ __forceinline__ double rsqrt_pos(double r2) { return r2 > 0.0 ? rsqrt(r2) : 0.0; }
__device__ __forceinline__ float rsqrt_pos(float r2) { return r2 > 0.0f ? rsqrtf(r2) : 0.0f; }

// 1/sqrt(r2) for r2 known to be positive and finite (well-separated surfaces):
// hardware estimate plus one second-order Newton correction,
// y (1 + e/2 + 3e^2/8) with e = 1 - r2 y^2.
__device__ __forceinline__ double rsqrt_sep(double r2) {
  const double y = __builtin_amdgcn_rsq(r2);
  const double e = fma(-r2 * y, y, 1.0);
  return fma(y * e, fma(e, 0.375, 0.5), y);
}
__device__ __forceinline__ float rsqrt_sep(float r2) { return __builtin_amdgcn_rsqf(r2); }
__device__ __forceinline__ double dexp(double x) { return exp(x); }
__device__ __forceinline__ void dsincos(double x, double* s, double* c) { sincos(x, s, c); }
// sin and cos for |x| < 2^30 in FP64.  x = n pi/2 + r with pi/2 as the sum of its
// rounding P1 and the rest P2 (Cody and Waite): h is exact, r + l is within
// n 2^-107 of the reduced argument; the Taylor series of sin r (to r^17) and cos r
// (to r^16) are truncated at 1e-19 and 2e-18 for |r| <= pi/4, and what rounds r
// and 1 - r^2/2 is added back (largest error over phases up to 1e9: 8.4e-17, the library's 8.7e-17).
// The library's sincos keeps a path for huge arguments beside it, a branch and
// registers (189 against 122 in the Helmholtz near field: half the waves).
__device__ __forceinline__ void sincos_near(double x, double* s, double* c) {
  const double n = __builtin_rint(x * 0.63661977236758134308);
  const double h = fma(-n, 1.57079632679489661923, x);
  const double r = fma(-n, 6.123233995736766036e-17, h);
  const double l = fma(-n, 6.123233995736766036e-17, h - r);  // what r was rounded by
  const double z = r * r, w = fma(z, -0.5, 1.0);
  double u = 1.0 / 355687428096000.0, v = 1.0 / 20922789888000.0;
  u = fma(u, z, -1.0 / 1307674368000.0);
  v = fma(v, z, -1.0 / 87178291200.0);
  u = fma(u, z, 1.0 / 6227020800.0);
  v = fma(v, z, 1.0 / 479001600.0);
  u = fma(u, z, -1.0 / 39916800.0);
  v = fma(v, z, -1.0 / 3628800.0);
  u = fma(u, z, 1.0 / 362880.0);
  v = fma(v, z, 1.0 / 40320.0);
  u = fma(u, z, -1.0 / 5040.0);
  v = fma(v, z, -1.0 / 720.0);
  u = fma(u, z, 1.0 / 120.0);
  v = fma(v, z, 1.0 / 24.0);
  u = fma(u, z, -1.0 / 6.0);
  const double sn = r + fma(u * z, r, l * w);
  const double cs = w + (fma(-0.5 * r, r, 1.0 - w) + fma(v * z, z, -r * l));
  const int q = int(n);
  const double a = q & 1 ? cs : sn, b = q & 1 ? sn : cs;
  *s = q & 2 ? -a : a;
  *c = (q + 1) & 2 ? -b : b;
}
// FP32 (mixed / FLOAT near field and surface evaluations): exp through the
// hardware 2^x, sine and cosine on the hardware units, whose argument is in
// revolutions, after reducing x / (2 pi) to [-1/2, 1/2].  The reductions
// cost a relative error of |x| 2^-24 (phase error |x| 6e-8 rad), the FP32
// rounding of the arguments themselves.
__device__ __forceinline__ float dexp(float x) { return __builtin_amdgcn_exp2f(x * 1.44269504088896341f); }
__device__ __forceinline__ void dsincos(float x, float* s, float* c) {
  const float t = x * 0.159154943091895336f;
  const float f = t - __builtin_rintf(t);
  *s = __builtin_amdgcn_sinf(f);
  *c = __builtin_amdgcn_cosf(f);
}

// Compensated (Kahan) accumulation of a partial sum into (s, c).
template <typename R>
__device__ __forceinline__ void kahan_add(R& s, R& c, R v) {
  const R y = v - c;
  const R t = s + y;
  c = (t - s) - y;
  s = t;
}

}  // namespace xfmm
