// Scalars of a Householder reflector with LAPACK's conventions (gfx950).
#pragma once

#include "kernels.hpp"

namespace qca {

// Scalars of one reflector (zlarfg): beta, tau and scale = 1 / (alpha - beta).
struct Larfg {
  double beta;
  c128 tau, scale;
};

// Squared norm of a column below its diagonal together with alpha, in the range
// where neither it nor the reciprocal of (alpha - beta)^2 over- or underflows.
// Columns outside are scaled by larfg_exponent first (LAPACK's zlarfg rescales
// likewise); a NaN is not.
__device__ __forceinline__ bool larfg_in_range(double s) { return !(s <= 1e-280 || s >= 1e280); }
// Binary exponent of the largest |re|, |im| of a column, 0 where there is none
// (all zero, or not finite).
__device__ __forceinline__ int larfg_exponent(double largest) {
  return largest > 0.0 && largest < __builtin_inf() ? ilogb(largest) : 0;
}

// alpha and the squared norm of what is below it, in range (or all zero).  Square
// root and divisions to the last bit: a refined reciprocal square root and a
// reciprocal in their place gave Q 4% more error and no time (512 x 256: 777
// against 784 us, splits equal).
__device__ __forceinline__ Larfg larfg(c128 alpha, double xnorm2) {
  Larfg h;
  h.beta = alpha.re;
  h.tau = c128{0.0, 0.0};
  h.scale = c128{1.0, 0.0};
  if (xnorm2 == 0.0 && alpha.im == 0.0) return h;
  const double s = alpha.re * alpha.re + alpha.im * alpha.im + xnorm2;
  const double nrm = sqrt(s);
  h.beta = (alpha.re >= 0.0) ? -nrm : nrm;
  const double dr = alpha.re - h.beta, di = alpha.im;
  const double den = dr * dr + di * di;
  h.scale = c128{dr / den, -di / den};
  h.tau = c128{-dr / h.beta, -di / h.beta};
  return h;
}

}  // namespace qca
