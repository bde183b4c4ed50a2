// Division and square root of the Schur chase (k_texture.hip) from the
// hardware's seeds, which are within 2^29 units in the last place.  Operands
// must lie well inside the normal range (the chase takes steps whose vector has
// an entry of at least 2^-350 and whose matrix and first vector are at most
// 2^340): the results are then the correctly rounded ones.
#pragma once

namespace wnd {

// 1 / d by two Newton steps from the seed y
__device__ __forceinline__ double recip(double d, double y) {
  double e = __builtin_fma(-d, y, 1.0);
  y = __builtin_fma(y, e, y);
  e = __builtin_fma(-d, y, 1.0);
  return __builtin_fma(y, e, y);
}

// a / d with d's reciprocal y: the product corrected by its exact remainder
// (Markstein, Computation of elementary functions on the IBM RISC System/6000,
// 1990)
__device__ __forceinline__ double quot(double a, double d, double y) {
  const double q = a * y;
  const double r = __builtin_fma(-d, q, a);
  return __builtin_fma(r, y, q);
}

// sqrt(a) from the seed y of 1 / sqrt(a): one step of Goldschmidt's coupled
// iteration for sqrt and 1 / (2 sqrt), then two corrections by the exact
// remainder
__device__ __forceinline__ double root(double a, double y) {
  double g = a * y, h = y * 0.5;
  const double r = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, r, g);
  h = __builtin_fma(h, r, h);
  double d = __builtin_fma(-g, g, a);
  g = __builtin_fma(d, h, g);
  d = __builtin_fma(-g, g, a);
  return __builtin_fma(d, h, g);
}

}  // namespace wnd
