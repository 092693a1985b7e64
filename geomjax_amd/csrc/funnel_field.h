// Closed-form vector field of RMHMC with the Monge metric on Neal's funnel
// (shared by the sampling and the tangent kernels; R may be float, double or
// a dual number).  See funnel_rmhmc.hip for the derivation.
#pragma once

#include "common.h"

namespace gjx {

// Per-chain scalar coefficients of the vector field at one iterate.
template <class R>
struct FieldCoef {
  R ce;   // u_x = p_x + ce * x
  R A, B; // dH/dq_x = A x + B p_x
  R uv;   // u_v
  R dHv;  // dH/dq_v
};

template <class R>
__device__ __forceinline__ FieldCoef<R> field_coef(R v, R pv, R sx, R xpx, R a2, R inv_s2, R halfDx) {
  const R e = exp(-v);
  const R gv = -v * inv_s2 - halfDx + R(0.5) * e * sx;
  const R gg = e * e * sx + gv * gv;
  const R gp = -e * xpx + gv * pv;
  const R L = R(1) + a2 * gg;
  const R k = a2 / L;
  const R c = gp * k;
  const R ce = c * e;
  const R uv = pv - c * gv;
  const R wv = gv - gp * uv;
  // x . w_x = -e Sx - (g.p) (x . u_x) = -e Sx - (g.p)(Xp + ce Sx)
  const R xw = -e * sx - gp * (xpx + ce * sx);
  const R hwv = e * xw - (inv_s2 + R(0.5) * e * sx) * wv;
  FieldCoef<R> f;
  f.ce = ce;
  f.A = e * (R(1) + k * (e + wv + gp * ce));
  f.B = e * k * gp;
  f.uv = uv;
  f.dHv = k * hwv - gv;
  return f;
}

// Whether the fixed-point iteration goes on, decided without the per-coordinate
// norm where that is certain.  The norm is the largest of |da x0_k + db p0_k| and
// |dg x0_k + dd p0_k| over the coordinates and of mv, the change of v and p_v.
// With |x0_k| <= X and |p0_k| <= P (2-norms, with slack for their rounding)
//   norm >= mv  and  norm <= max(|da| X + |db| P, |dg| X + |dd| P, mv),
// so mv > tol with the upper bound below the divergence limit goes on, an upper
// bound within tol has converged, and a non-finite change (norm NaN) stops.
// Everything else is kOpen: the norm itself has to be formed.
// A term of the upper bound is NaN only as 0 times an infinite X or P, and fmaxf drops
// it.  An infinite |x0|^2 makes the field's coefficients NaN (finite is false); with
// an infinite |p0|^2 and a step other than 0 the change's coefficient of p0 in x is not 0 in
// the first iterate, so the other term is infinite (kOpen), and the next iterate's field
// is NaN.  With a step of 0 all four coefficients are 0 and the norm is mv.
enum SpanDecision { kStop, kGoOn, kOpen };

struct SpanBound {
  float X, P;
  __device__ __forceinline__ SpanBound(float Sxx, float Spp) : X(1.001f * sqrtf(Sxx)), P(1.001f * sqrtf(Spp)) {}
  __device__ __forceinline__ SpanDecision operator()(bool finite, float mv, float da, float db, float dg, float dd,
                                                     double tol, double div_tol) const {
    const float up = 1.001f * fmaxf(fmaxf(fabsf(da) * X + fabsf(db) * P, fabsf(dg) * X + fabsf(dd) * P), mv);
    if (!finite || mv != mv) return kStop;
    if ((double)mv > tol && (double)up < div_tol) return kGoOn;
    if ((double)up <= tol) return kStop;
    return kOpen;
  }
};

// Whether a layout of LPC lanes with EPL coordinates each forms the bounds first.  They
// cost about forty instructions of every iteration's serial chain; the norm they
// save costs EPL steps and log2(LPC) exchanges, those past a row of 16 lanes through
// LDS.  Measured against the norm in every iteration, time ratio at 9 | 8192 chains,
// 18 steps, four transitions (LPC x EPL): 4x1 0.85 | 0.82, 4x4 0.96 | 0.93, 4x8 1.10 | 1.04,
// 8x4 0.97 | 0.99, 8x8 1.10 | 1.10, 8x16 1.20 | 1.22, 16x1 0.97 | 1.01, 16x2 1.00 | 1.09,
// 16x8 1.17 | 1.28, 32x1 1.01 | 1.05, 32x4 1.11 | 1.14, 64x1 1.12 | 1.12.
template <int LPC, int EPL>
__device__ constexpr bool span_screens() {
  return EPL >= 8 || LPC >= 32 || (LPC == 16 && EPL >= 2);
}

// Quadratic form p^T G^-1 p of the Monge metric G = I + a2 g g^T, written as
//   |p|^2 / L + (a2 |g|^2 / L) |p_perp|^2,   L = 1 + a2 |g|^2,
//   p_perp = p - (g.p / |g|^2) g   (formed component by component).
// Both terms are sums of squares, so the value is never negative and keeps its
// relative accuracy.  The textbook |p|^2 - a2 (g.p)^2 / L loses every digit to
// cancellation once a2 |g|^2 is large (a fixed-point iterate that ran away)
// and can come out hugely negative, which would make a run-away state look
// like a large energy gain.  The dense Cholesky form -log N(p; 0, G) never
// goes negative either.  With g = (-e x, gv) for the funnel,
// p_perp = (p_x + c e x, p_v - c gv) where c = monge_perp_coef(g.p, |g|^2).
template <class R>
__device__ __forceinline__ R monge_perp_coef(R gp, R gg) {
  return gg > R(0) ? gp / gg : R(0);
}
template <class R>
__device__ __forceinline__ R monge_quad(R pp, R perp2, R gg, R a2) {
  const R L = R(1) + a2 * gg;
  return pp / L + (a2 * gg / L) * perp2;
}

}  // namespace gjx
