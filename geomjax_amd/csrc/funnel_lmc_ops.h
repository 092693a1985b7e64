// Device building blocks of the LMC-Monge integrator on Neal's funnel, shared by
// the transition kernels (funnel_lmc.hip) and NUTS (funnel_nuts.hip).  R is
// float, double or a dual number; LPC lanes per chain hold EPL coordinates each.
//
// Reference: geomjax/lmcmonge/integrators.py:52-194 (lan_integrator,
// half_step_omega), geomjax/lmcmonge/metrics.py:104-284 (velocity draw,
// kinetic energy, weighted gradients), examples/funnel/main.py:34-39.
// The closed forms are derived at the top of funnel_lmc.hip.
#pragma once

#include "common.h"
#include "dual.h"
#include "funnel_lmc.h"

namespace gjx {
namespace lmc_ops {

template <class R>
struct PosScalars {
  R e, Sx, Smx, gv, L, sL, isL, dlv, Hdlv, igHdlv;
  R eL;          // e / sqrt(L)
  R Q1, Q2, Q3;  // eL sum mi x^2, eL^2 sum mi^2 x^2, eL^2 sum mi^3 x^2
};

// Sums over a position's coordinates: x^2, mi x^2, mi^2 x^2, mi^3 x^2.
template <class R>
struct PosSums {
  R x2 = R(0), mx2 = R(0), m2x2 = R(0), m3x2 = R(0);
  __device__ __forceinline__ void add(R x, R mi) {
    const R t = mi * x, u = mi * t;
    x2 += x * x;
    mx2 += t * x;
    m2x2 += t * t;
    m3x2 += u * t;
  }
  template <int LPC>
  __device__ __forceinline__ void reduce() {
    x2 = group_sum<LPC>(x2);
    mx2 = group_sum<LPC>(mx2);
    m2x2 = group_sum<LPC>(m2x2);
    m3x2 = group_sum<LPC>(m3x2);
  }
};

template <class R>
__device__ __forceinline__ PosScalars<R> pos_scalars(R v, const PosSums<R>& S, R a2, R inv_s2, R halfDx, R miv) {
  PosScalars<R> P;
  const R Sx = S.x2, Smx = S.mx2;
  P.e = exp(-v);
  P.Sx = Sx;
  P.Smx = Smx;
  P.gv = -v * inv_s2 - halfDx + R(0.5) * P.e * Sx;
  P.L = R(1) + a2 * (P.e * P.e * Smx + miv * P.gv * P.gv);  // normalizing_constant (metrics.py:193-197)
  P.sL = sqrt(P.L);
  P.isL = R(1) / P.sL;
  P.dlv = miv * P.gv * P.isL;
  // Hdl_v = (e (x . dl_x) - (1/sigma^2 + e Sx / 2) dl_v) / sqrt(L),  x . dl_x = -e Smx / sqrt(L)
  P.Hdlv = (-P.e * P.e * Smx * P.isL - (inv_s2 + R(0.5) * P.e * Sx) * P.dlv) * P.isL;
  P.igHdlv = miv * P.Hdlv;
  // eL meets a sum one factor at a time: its square alone may leave R's range
  P.eL = P.e * P.isL;
  P.Q1 = P.eL * Smx;
  P.Q2 = P.eL * (P.eL * S.m2x2);
  P.Q3 = P.eL * (P.eL * S.m3x2);
  return P;
}

// One half_step_omega (geomjax/lmcmonge/integrators.py:158-194) at the
// position described by P, updating the velocity (vx, vv) and dJ.
//
// Every vector of the half step is a combination of x, mi x, mi^2 x and the
// velocity (t = mi x, u = mi t below), so its dot products s0 .. s7 are
// combinations of the position's sums Q1 .. Q3, formed once per position for both
// half steps that meet there, and of four sums with the velocity.  VALU issue and the
// chain of group sums bound the kernel: a step takes 12 of them (18 with each dot
// product summed by itself) and about half the instructions per coordinate (8192 chains,
// 100 float32 coordinates, 4 transitions of 32 steps: 448 -> 368 us; the position's
// error against float64 arithmetic 6.0e-4 -> 5.3e-4).
//   dl = -eL t,  Hdl = eL (eL t + dlv x),  hv = eL (vv x - v),
//   dphi = g0 x + k1 eL^2 t,  dphi_ig = mi dphi,  g0 = eL (1 + k1 dlv), k1 = alpha2 / sqrt(L).
template <class R, int LPC, int EPL>
__device__ __forceinline__ void half_step(const PosScalars<R>& P, const R (&x)[EPL], const R (&mi)[EPL], R (&vx)[EPL],
                                          R& vv, double& dJ, R a2, R inv_s2, R h, bool exact_sm) {
  R xv = R(0), tv = R(0), uv = R(0), v2 = R(0);
#pragma unroll
  for (int k = 0; k < EPL; ++k) {
    const R t = mi[k] * x[k], u = mi[k] * t;
    xv += x[k] * vx[k];
    tv += t * vx[k];
    uv += u * vx[k];
    v2 += vx[k] * vx[k];
  }
  xv = group_sum<LPC>(xv);
  tv = group_sum<LPC>(tv);
  uv = group_sum<LPC>(uv);
  v2 = group_sum<LPC>(v2);
  const R eL = P.eL, k1 = a2 * P.isL, ke = k1 * eL;
  const R g0 = eL * (R(1) + k1 * P.dlv);
  const R m1 = eL * tv, m2 = eL * (eL * uv);
  const R w1 = vv * P.Q1 - m1, w2 = vv * P.Q2 - m2;  // eL sum t (vv x - v), eL^2 sum u (vv x - v)
  const R q2 = P.Q2 + P.dlv * P.Q1;
  const R s0 = -eL * w1;                                                    // hv . dl
  const R s1 = -(g0 * P.Q1 + ke * P.Q2);                                    // dphi . dl
  const R s3 = eL * (vv * xv - v2);                                         // v . hv
  const R s4 = g0 * w1 + ke * w2;                                           // dphi_ig . hv
  const R s5 = eL * (m1 + P.dlv * xv);                                      // Hdl . v
  const R s6 = g0 * q2 + ke * (eL * P.Q3 + P.dlv * P.Q2);                   // Hdl . dphi_ig
  const R s7 = -eL * q2;                                                    // Hdl . dl
  // log-scale coordinate contributions
  const R hv_v = (P.e * xv - (inv_s2 + R(0.5) * P.e * P.Sx) * vv) * P.isL;
  const R gn_v = P.gv * P.isL;
  const R dphi_v = -gn_v + a2 * P.Hdlv * P.isL;
  const R dphig_v = -P.dlv + a2 * P.igHdlv * P.isL;
  const R P1 = s0 + hv_v * P.dlv;     // hv . dl
  const R P2 = s1 + dphi_v * P.dlv;   // dphi . dl
  const R P3 = s3 + vv * hv_v;        // v . hv
  const R P4 = s4 + dphig_v * hv_v;   // dphi_ig . hv
  const R P5 = s5 + P.Hdlv * vv;      // Hdl . v
  const R P6 = s6 + P.Hdlv * dphig_v; // Hdl . dphi_ig
  const R P7 = s7 + P.Hdlv * P.dlv;   // Hdl . dl
  // 1st volume adjustment (:178-179)
  const R d1 = R(1) + h * a2 * P1;
  dJ -= log(fabs((double)val(d1)));
  // v_t = v - (eps/2) sqrt(L) (dphi_ig - alpha2 (dphi.dl) dl)   (:182-185)
  const R vtH = P3 - h * P.sL * (P4 - a2 * P2 * P1);
  R coef = h * vtH / d1;  // (:186-189); the reference has no alpha2 here
  if (exact_sm) coef *= a2;
  const R HdlVn = P5 - h * P.sL * (P6 - a2 * P2 * P7) - coef * P7;
  // 2nd volume adjustment (:192)
  dJ += log(fabs((double)val(R(1) - h * a2 * HdlVn)));
  const R kq = h * P.sL, kd = a2 * P2;
  const R ct = eL * (coef - kq * kd) - kq * g0, cu = kq * ke;
#pragma unroll
  for (int k = 0; k < EPL; ++k) {
    const R t = mi[k] * x[k], u = mi[k] * t;
    vx[k] = vx[k] + ct * t - cu * (eL * u);
  }
  vv = vv - kq * (dphig_v - kd * P.dlv) - coef * P.dlv;
}

// Scalars of the position (x, v) and the inclusive prefix of mi x^2 over the
// chain's coordinates in lane order (the velocity draw's running sums).
template <class R, int LPC, int EPL>
__device__ __forceinline__ PosScalars<R> position_scalars(const R (&x)[EPL], R v, const R (&mi)[EPL], R (&loc_inc)[EPL],
                                                          int lg, R a2, R inv_s2, R halfDx, R miv) {
  PosSums<R> S;
#pragma unroll
  for (int k = 0; k < EPL; ++k) {
    S.add(x[k], mi[k]);
    loc_inc[k] = S.mx2;
  }
  const R off = group_exclusive_scan<LPC>(S.mx2, lg);
#pragma unroll
  for (int k = 0; k < EPL; ++k) loc_inc[k] += off;
  S.template reduce<LPC>();
  return pos_scalars<R>(v, S, a2, inv_s2, halfDx, miv);
}

// The transition's standard normals for the velocity draw and its accept
// uniform: host-fed ([T, C, D] in storage type T, [T, C]) or the device Philox
// streams at counter + t.
template <class T, int EPL>
__device__ __forceinline__ void transition_noise(const FunnelLmcArgs& a, size_t c, int t, int j0, int Dx, bool live,
                                                 T (&z)[EPL], T& zv, double& uacc) {
  const int D = Dx + 1;
  const uint64_t tt = a.counter + (uint64_t)t;
  const uint32_t k0 = (uint32_t)a.seed, k1 = (uint32_t)(a.seed >> 32);
  if (a.z != nullptr) {
    const size_t base = ((size_t)t * a.C + c) * D;
#pragma unroll
    for (int k = 0; k < EPL; ++k) z[k] = (live && j0 + k < Dx) ? ld<T>(a.z, base + j0 + k) : T(0);
    zv = live ? ld<T>(a.z, base + Dx) : T(0);
    uacc = (live && a.u != nullptr) ? a.u[(size_t)t * a.C + c] : 1.0;
    return;
  }
#pragma unroll
  for (int k = 0; k < EPL; k += 2) {
    u32x4 r = philox4x32_10(u32x4{(uint32_t)c, (uint32_t)tt, kStreamMomentum + (uint32_t)(j0 + k), (uint32_t)(tt >> 32)},
                            k0, k1);
    T n0, n1;
    normal2(r, n0, n1);
    z[k] = j0 + k < Dx ? n0 : T(0);
    if (k + 1 < EPL) z[k + 1] = j0 + k + 1 < Dx ? n1 : T(0);
  }
  {
    u32x4 r = philox4x32_10(u32x4{(uint32_t)c, (uint32_t)tt, kStreamMomentumV, (uint32_t)(tt >> 32)}, k0, k1);
    T n0, n1;
    normal2(r, n0, n1);
    zv = n0;
  }
  u32x4 r = philox4x32_10(u32x4{(uint32_t)c, (uint32_t)tt, kStreamAccept, (uint32_t)(tt >> 32)}, k0, k1);
  uacc = u01_f64(r.x, r.y) - 0.5 * (1.0 / 9007199254740992.0);
}

// Velocity v0 = chol(M^-1 - alpha2 dl dl^T) z (geomjax/lmcmonge/metrics.py:155-166)
// with the exact lower factor of a diagonal-minus-rank-one matrix.
template <class R, int LPC, int EPL>
__device__ __forceinline__ void draw_velocity(const PosScalars<R>& P, const R (&x)[EPL], const R (&mi)[EPL],
                                              const R (&loc_inc)[EPL], const R (&z)[EPL], R zv, R a2, R alpha,
                                              R miv, int lg, int j0, int Dx, R (&vx)[EPL], R& vv) {
  // a_j^2 = alpha2 dl_j^2 / mi_j = (alpha2 e^2 / L) mi_j x_j^2
  const R w = a2 * P.e * P.e / P.L;
  R cj[EPL];
  R acc2 = R(0);
#pragma unroll
  for (int k = 0; k < EPL; ++k) {
    const R tj = R(1) - w * loc_inc[k];
    const R tjm = R(1) - w * (loc_inc[k] - mi[k] * x[k] * x[k]);
    const R aj = -alpha * P.e * sqrt(mi[k]) * x[k] * P.isL;
    cj[k] = aj * z[k] / sqrt(tj * tjm);
    vx[k] = sqrt(tj / tjm) * z[k];
    acc2 += cj[k];
  }
  const R off2 = group_exclusive_scan<LPC>(acc2, lg);
  const R tot2 = group_sum<LPC>(acc2);
  R run = off2;
#pragma unroll
  for (int k = 0; k < EPL; ++k) {
    const R aj = -alpha * P.e * sqrt(mi[k]) * x[k] * P.isL;
    vx[k] = j0 + k < Dx ? sqrt(mi[k]) * (vx[k] - aj * run) : R(0);
    run += cj[k];
  }
  // t after all x coordinates is 1 - alpha2 e^2 Smx / L; then the log-scale coordinate
  const R txe = R(1) - w * P.Smx;
  const R av = alpha * sqrt(miv) * P.gv * P.isL;
  const R tv = txe - av * av;
  vv = sqrt(miv) * (sqrt(tv / txe) * zv - av * tot2);
}

// One lan_integrator step (geomjax/lmcmonge/integrators.py:52-156): half step of
// the velocity, full step of the position, half step of the velocity.
template <class R, int LPC, int EPL>
__device__ __forceinline__ void lmc_step(PosScalars<R>& P, R (&xc)[EPL], R& vc, const R (&mi)[EPL], R (&vx)[EPL],
                                         R& vv, double& dJ, R eps, R h, R a2, R inv_s2, R halfDx, R miv,
                                         bool exact_sm) {
  half_step<R, LPC, EPL>(P, xc, mi, vx, vv, dJ, a2, inv_s2, h, exact_sm);
  PosSums<R> S;
#pragma unroll
  for (int k = 0; k < EPL; ++k) {
    xc[k] = xc[k] + eps * vx[k];
    S.add(xc[k], mi[k]);
  }
  vc = vc + eps * vv;
  S.template reduce<LPC>();
  P = pos_scalars<R>(vc, S, a2, inv_s2, halfDx, miv);
  half_step<R, LPC, EPL>(P, xc, mi, vx, vv, dJ, a2, inv_s2, h, exact_sm);
}


// Kinetic energy of the lmcmonge metric (geomjax/lmcmonge/metrics.py:168-186) in
// float64 sums: -(log L - sum log mi)/2 + |v|_M^2 / 2 + alpha2 (v . g)^2 / 2,
// g = (-e x, gv) the full gradient.
template <class R, int LPC, int EPL>
__device__ __forceinline__ double lmc_kinetic(const PosScalars<R>& Q, const R (&xx)[EPL], const R (&vel)[EPL], R velv,
                                              const R (&mi)[EPL], R miv, int j0, int Dx, double sum_log_mi,
                                              double alpha2) {
  double svm = 0.0, xv = 0.0;
#pragma unroll
  for (int k = 0; k < EPL; ++k) {
    if (j0 + k < Dx) svm += (double)val(vel[k]) * (double)val(vel[k]) / (double)val(mi[k]);
    xv += (double)val(xx[k]) * (double)val(vel[k]);
  }
  svm = group_sum<LPC>(svm) + (double)val(velv) * (double)val(velv) / (double)val(miv);
  xv = group_sum<LPC>(xv);
  const double vg = -(double)val(Q.e) * xv + (double)val(velv) * (double)val(Q.gv);  // v . g
  return -0.5 * (log((double)val(Q.L)) - sum_log_mi) + 0.5 * svm + 0.5 * alpha2 * vg * vg;
}

}  // namespace lmc_ops
}  // namespace gjx
