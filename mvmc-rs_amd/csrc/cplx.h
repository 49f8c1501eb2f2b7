// Complex double arithmetic of the complex Pfaffian kernels: num_complex's
// products and Julia's scaled division and reciprocal (built with
// -ffp-contract=off).
#pragma once
#include <hip/hip_runtime.h>

namespace mvmc_hip {

struct alignas(16) cz {
  double re, im;
};
__device__ __forceinline__ cz cz_mul(cz a, cz b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
__device__ __forceinline__ cz cz_add(cz a, cz b) { return {a.re + b.re, a.im + b.im}; }
__device__ __forceinline__ cz cz_sub(cz a, cz b) { return {a.re - b.re, a.im - b.im}; }
__device__ __forceinline__ cz cz_neg(cz a) { return {-a.re, -a.im}; }

// Julia's ComplexF64 reciprocal (crates/pfapack/src/julia_complex.rs:79-122).
__device__ inline cz julia_recip(cz w) {
  double c = w.re, d = w.im;
  const double absc = fabs(c), absd = fabs(d);
  const double cd = absc > absd ? absc : absd;
  const double dc = absc > absd ? absd : absc;
  // sqrt(DBL_MIN/2) <= cd <= sqrt(DBL_MAX/2)
  if (0x1.6a09e667f3bcdp-512 <= cd && cd <= 0x1.6a09e667f3bccp+511) {
    const double norm = fma(cd, cd, dc * dc);
    return {c / norm, -d / norm};
  }
  if (isinf(c) || isinf(d)) return {copysign(0.0, c), copysign(-0.0, -d)};
  const double bs = 0x1p+105;  // 2 / eps^2
  double scale = 1.0;
  if (cd >= 0x1.fffffffffffffp+1022) {  // DBL_MAX / 2
    c *= 0.5;
    d *= 0.5;
    scale = 0.5;
  } else if (cd <= 0x1p-969) {  // 2 DBL_MIN / eps
    c *= bs;
    d *= bs;
    scale = bs;
  }
  double p, q;
  if (absd <= absc) {
    const double r = d / c, z = fma(d, r, c);
    p = 1.0 / z;
    q = -r / z;
  } else {
    const double r = -c / -d, z = fma(-c, r, -d);
    q = 1.0 / z;
    p = -r / z;
  }
  return {p * scale, q * scale};
}

__device__ inline double julia_div_part(double a, double b, double c, double d, double r, double t) {
  if (r != 0.0) {
    const double br = b * r;
    return br != 0.0 ? (a + br) * t : a * t + (b * t) * r;
  }
  return (a + d * (b / c)) * t;
}

// Julia's scaled ComplexF64 division (julia_complex.rs:9-77).
__device__ inline cz julia_div(cz z, cz w) {
  double a = z.re, b = z.im, c = w.re, d = w.im;
  const double ab = fabs(a) >= fabs(b) ? fabs(a) : fabs(b);
  const double cdm = fabs(c) >= fabs(d) ? fabs(c) : fabs(d);
  if (isinf(c) || isinf(d)) {
    auto sgn = [](double x) { return (x == 0.0 || isnan(x)) ? x : copysign(1.0, x); };
    if (isfinite(a) && isfinite(b)) return {0.0 * sgn(a) * sgn(c), -0.0 * sgn(b) * sgn(d)};
    return {__builtin_nan(""), __builtin_nan("")};
  }
  const double halfov = 0x1.fffffffffffffp+1022, twouneps = 0x1p-969;
  double s = 1.0;
  const bool scaled = ab >= halfov || ab <= twouneps || cdm >= halfov || cdm <= twouneps;
  if (scaled) {
    const double bs = 0x1p+105;
    if (ab >= halfov) {
      a *= 0.5;
      b *= 0.5;
      s *= 2.0;
    } else if (ab <= twouneps) {
      a *= bs;
      b *= bs;
      s /= bs;
    }
    if (cdm >= halfov) {
      c *= 0.5;
      d *= 0.5;
      s *= 0.5;
    } else if (cdm <= twouneps) {
      c *= bs;
      d *= bs;
      s *= bs;
    }
  }
  bool swapped = false;
  if (!(fabs(d) <= fabs(c))) {
    double t0 = a;
    a = b;
    b = t0;
    t0 = c;
    c = d;
    d = t0;
    swapped = true;
  }
  const double r = d / c;
  const double t = 1.0 / (c + d * r);
  const double p = julia_div_part(a, b, c, d, r, t);
  double q = julia_div_part(b, -a, c, d, r, t);
  if (swapped) q = -q;
  if (scaled) return {p * s, q * s};
  return {p, q};
}

}  // namespace mvmc_hip
