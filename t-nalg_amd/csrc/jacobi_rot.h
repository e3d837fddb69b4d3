// Plane rotations of the one-sided Jacobi SVDs.
#pragma once
#include "tnx_common.h"

// The rotation of two columns x, y with norms^2 a, c and product g:
//   x' = x - s (y + tau x),  y' = y + s (x - tau y),  tau = s / (1 + cos),
// and with `swap` x'' = y', y'' = -x', so that the larger column comes first.
// rot: rotate (the caller's test; g is not zero); order: the pair may be
// swapped.  The tangent needs no more than the hardware's reciprocal and root
// (any angle is a rotation; an approximate one leaves 1e-7 of g); it is formed
// from the entries over a power of two near the larger one, so nothing over-
// or underflows (without SCALE the caller keeps their squares in range).  The cosine and tau are refined to working accuracy (third
// order: the cube of the approximation's 2^-20 or less), so the transformation
// is orthogonal; in this form its rounding errors are those of the small
// numbers s and tau, not of cos.
struct JacobiRot { double s, tau; bool swap; };

template <bool SCALE = true>
__device__ __forceinline__ JacobiRot jacobi_rot(double a, double c, double g, bool rot, bool order) {
  JacobiRot r;
  r.swap = order && c > a;
  double h = rot ? c - a : 0.0;
  if constexpr (SCALE) {
    const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(h), fabs(g)));
    h = __builtin_amdgcn_ldexp(h, ex);
    g = __builtin_amdgcn_ldexp(g, ex);
  }
  const double g2 = rot ? 2.0 * g : 1.0;
  const double w = fma(h, h, g2 * g2);
  const double den = fabs(h) + w * __builtin_amdgcn_rsq(w);
  const double t = (h >= 0.0 ? g2 : -g2) * __builtin_amdgcn_rcp(den);   // |t| <= 1
  const double x = fma(t, t, 1.0);
  double y = __builtin_amdgcn_rsq(x);              // cos = 1 / sqrt(1 + t^2)
  const double e = fma(-x * y, y, 1.0);
  y = fma(y * e, fma(0.375, e, 0.5), y);
  const double d = 1.0 + y;
  double q = __builtin_amdgcn_rcp(d);
  const double f = fma(-d, q, 1.0);
  q = fma(q, fma(f, f, f), q);
  r.s = rot ? y * t : 0.0;
  r.tau = r.s * q;
  return r;
}

__device__ __forceinline__ void jacobi_apply(const JacobiRot& r, double& x, double& y) {
  const double xn = fma(-r.s, fma(r.tau, x, y), x), yn = fma(r.s, fma(-r.tau, y, x), y);
  x = r.swap ? yn : xn;
  y = r.swap ? -xn : yn;
}
