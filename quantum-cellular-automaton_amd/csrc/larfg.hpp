// Scalars of a Householder reflector with LAPACK's conventions (gfx950).
#pragma once

#include "kernels.hpp"

namespace qca {

// Scalars of one reflector (zlarfg): beta, tau, scale = 1 / (alpha - beta), and
// gamma = conj(tau) |scale|^2 = 1 / (beta (beta - alpha)), the factor of the
// reflector in its unscaled form u = (alpha - beta, x): H^H = I - gamma u u^H.
struct Larfg {
  double beta;
  c128 tau, scale, gamma, u0;
};
// In the range where no square over- or underflows, sqrt and 1 / beta come from
// one reciprocal square root refined by Newton steps (half the serial latency
// of sqrt and a division).
__device__ __forceinline__ Larfg larfg(c128 alpha, double xnorm2) {
  Larfg h;
  h.beta = alpha.re;
  h.tau = h.gamma = c128{0.0, 0.0};
  h.scale = h.u0 = c128{1.0, 0.0};
  if (xnorm2 == 0.0 && alpha.im == 0.0) return h;
  const double s = alpha.re * alpha.re + alpha.im * alpha.im + xnorm2;
  double nrm, inrm;
  if (s > 1e-280 && s < 1e280) {
    // y (1 + e/2 + 3 e^2 / 8), e = 1 - s y^2, then one more step on sqrt and 1/sqrt
    double y = __builtin_amdgcn_rsq(s);
    const double e = fma(-s * y, y, 1.0);
    y = fma(y, e * fma(0.375, e, 0.5), y);
    nrm = s * y;
    nrm = fma(0.5 * y, fma(-nrm, nrm, s), nrm);
    inrm = fma(y, fma(-nrm, y, 1.0), y);
  } else {
    nrm = sqrt(s);
    inrm = 1.0 / nrm;
  }
  h.beta = (alpha.re >= 0.0) ? -nrm : nrm;
  const double ib = (alpha.re >= 0.0) ? -inrm : inrm;
  const double dr = alpha.re - h.beta, di = alpha.im;
  const double id = 1.0 / (dr * dr + di * di);
  h.u0 = c128{dr, di};
  h.scale = c128{dr * id, -di * id};
  h.tau = c128{-dr * ib, -di * ib};
  h.gamma = c128{-h.scale.re * ib, -h.scale.im * ib};
  return h;
}

}  // namespace qca
