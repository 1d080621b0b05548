// float64 arithmetic of the thermostat chain, shared by the kernels and a host test. Compiled without contraction:
// every operation rounds, fused ones are written out.
#pragma once

#include <math.h>

// a / b from r = 1 / b (rounded): the product, its remainder and one correction give the rounded quotient
// (Markstein's theorem; away from overflow and underflow). A non-finite a keeps a * r.
__host__ __device__ __forceinline__ double div_q(double a, double b, double r) {
  const double q = a * r;
  const double rem = fma(-q, b, a);
  return rem == rem ? fma(rem, r, q) : q;
}

// exp(x) for |x| < kExpSmall: the Taylor polynomial of degree 9 (the next term is below 2^-71), summed in pairs and
// added to 1 last. The last sum rounds by half a unit in the last place; the one before it rounds by 2^-59 below 2^-5
// and by 2^-58 above (x > 0 only), 2^-6 units of a result below or above 1, and the terms within it by less than
// 2^-9 units: at most 0.518 units off (0.516 measured).
constexpr double kExpSmall = 0.03125;

__host__ __device__ __forceinline__ double exp_small(double x) {
  const double x2 = x * x;
  const double a = fma(x, 1.0 / 6, 0.5), b = fma(x, 1.0 / 120, 1.0 / 24);
  const double c = fma(x, 1.0 / 5040, 1.0 / 720), d = fma(x, 1.0 / 362880, 1.0 / 40320);
  const double lo = fma(x2, b, a), hi = fma(x2, d, c);
  return 1.0 + fma(x2, fma(x2 * x2, hi, lo), x);
}
