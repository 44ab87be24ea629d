// nlm_sincos.hpp -- sine and cosine of small angles.
#pragma once

// sin and cos for |x| <= pi/4, without a branch, so that the points of a lane overlap.
// With z = x^2: sin x = x + x z S(z), cos x = (1 - z/2) + (z^2 C(z) + the rounding errors
// of 1 - z/2 and of z).  S (degree 6) and C (degree 5) interpolate the exact series at the
// Chebyshev nodes of [0, (pi/4)^2]; truncation below 1e-18.  Largest error over 4e6 points:
// sin 0.69 ulp, cos 0.56 (0.75 without the error of z); the library's sincos on the card
// 0.77 and 0.74.
__device__ __forceinline__ void sincos_small(double x, double* s, double* c) {
  const double z = x * x, zl = fma(x, x, -z);
  double p = -7.586691094197958e-13;
  p = fma(p, z, 1.6058531516797758e-10);
  p = fma(p, z, -2.5052106231802837e-08);
  p = fma(p, z, 2.7557319219337312e-06);
  p = fma(p, z, -0.00019841269841265063);
  p = fma(p, z, 0.008333333333333331);
  p = fma(p, z, -0.16666666666666666);
  *s = fma(x * z, p, x);
  double q = -1.1382623647474604e-11;
  q = fma(q, z, 2.087614614655861e-09);
  q = fma(q, z, -2.7557317271145144e-07);
  q = fma(q, z, 2.480158729876456e-05);
  q = fma(q, z, -0.0013888888888887398);
  q = fma(q, z, 0.041666666666666664);
  const double h = fma(-0.5, z, 1.0);
  *c = h + fma(z * z, q, fma(-0.5, zl, fma(-0.5, z, 1.0 - h)));
}
