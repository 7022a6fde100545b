// inv_gamma.h — 1 / sqrt(1 + p^2), the reciprocal Lorentz factor of the pushes and of
// their reverse, which replays the push's sub-steps and so needs the same bits.
#pragma once

#include <math.h>

#ifdef __HIPCC__
#define QSS_HD __host__ __device__
#else
#define QSS_HD
#endif

QSS_HD inline float inv_gamma(float px, float py, float pz) {
  return 1.0f / sqrtf(1.0f + px * px + py * py + pz * pz);
}

// On the device the hardware's estimate (about 2^-24) and two Newton steps on
// g = x y, h = y / 2 (Goldschmidt's coupled form), then a last correction: 14
// operations with an error under an ulp, where a square root and a division are 29
// with two roundings.  Where p^2 overflows the estimate is 0 and so is the result, as
// the division's: the steps then multiply that 0 by the largest double, not by infinity.
QSS_HD inline double inv_gamma(double px, double py, double pz) {
  double x = 1.0 + px * px + py * py + pz * pz;
#ifdef __HIP_DEVICE_COMPILE__
  double y = __builtin_amdgcn_rsq(x);   // of NaN: NaN, whatever the minimum gives
  x = __builtin_fmin(x, __DBL_MAX__);
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  y = __builtin_fma(h, __builtin_fma(-h, g, 0.5), h);   // half of 1/sqrt(x)
  y = y + y;
  return __builtin_fma(0.5 * y, __builtin_fma(-(x * y), y, 1.0), y);
#else
  return 1.0 / sqrt(x);
#endif
}
