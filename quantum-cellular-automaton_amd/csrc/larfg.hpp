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

// alpha and the squared norm of what is below it, in range (or all zero).
__device__ __forceinline__ Larfg larfg(c128 alpha, double xnorm2) {
  Larfg h;
  h.beta = alpha.re;
  h.tau = c128{0.0, 0.0};
  h.scale = c128{1.0, 0.0};
  if (xnorm2 == 0.0 && alpha.im == 0.0) return h;
  const double s = alpha.re * alpha.re + alpha.im * alpha.im + xnorm2;
  // sqrt and 1 / sqrt from one reciprocal square root and Newton steps:
  // y (1 + e/2 + 3 e^2 / 8), e = 1 - s y^2, then one more step on each.  sqrt() and
  // divisions to the last bit are a longer serial chain: QR 32x32 67.3 us instead of
  // 65.8, 512x256 786 instead of 777, split 12x16 264 instead of 246 (left sweep), for
  // Q of 4.4e-16 instead of 4.6e-16 and R of 1.01e-16 instead of 1.04e-16 (25 shapes up
  // to 512x256; 4.9e-16 and 1.08e-16 with panel GEMMs in place of register panels)
  double y = __builtin_amdgcn_rsq(s);
  const double e = fma(-s * y, y, 1.0);
  y = fma(y, e * fma(0.375, e, 0.5), y);
  double nrm = s * y;
  nrm = fma(0.5 * y, fma(-nrm, nrm, s), nrm);
  const double inrm = fma(y, fma(-nrm, y, 1.0), y);
  h.beta = (alpha.re >= 0.0) ? -nrm : nrm;
  const double ib = (alpha.re >= 0.0) ? -inrm : inrm;
  const double dr = alpha.re - h.beta, di = alpha.im;
  const double id = 1.0 / (dr * dr + di * di);
  h.scale = c128{dr * id, -di * id};
  h.tau = c128{-dr * ib, -di * ib};
  return h;
}

}  // namespace qca
