// The fused modes of the per-zone solve (compiled with
// -ffp-contract=fast-honor-pragmas): the FP64 residual in its identity form,
// the per-zone constants of the EMHD rows, and the Newton step by
// elimination instead of a dense Jacobian and LU.
//
// Identities (normal-observer split, beta^i = alpha^2 g^0i, gamma_ij = g_ij):
//   u^0 = gamma/alpha, u_i = gamma_ij utilde^j, u_0 = -alpha gamma + g_0j utilde^j
//   b^0 = B^i u_i,  b_mu = (B_mu + b^0 u_mu)/u^0  with B_mu = g_mu,j B^j
//   b^mu b_mu = (B^i B_i + (b^0)^2)/(u^0)^2
// so the t-row of the stress tensor needs no contravariant spatial vector,
// and with A_u = w u^0 + q b^0/|b| + u^0 dP/3, A_b = q u^0/|b| - b^0 (1 + dP/b^2)
//   T^0_nu = A_u u_nu + A_b b_nu + d_0nu (p + b^2/2 + dP/3).
//
// Newton step.  Write the variation of the momentum rows with the spatial
// unknowns lowered, x_i = gamma_ij d(utilde^j):
//   c2 x_i + S_u u_i + S_b b_i = r_i
// where c2 depends on the state only and S_u, S_b collect every scalar that
// multiplies u_i and b_i (they are linear in d(rho), d(u), d(q), d(dP) and in
// X = utilde^i x_i, Y = B^i x_i).  Contracting with utilde, B and beta gives
// X, Y and Z = beta^i x_i as affine functions of (S_u, S_b), the density row
// gives d(rho), the EMHD rows (diagonal in their own unknown) d(q), d(dP),
// and the definitions of S_u and S_b with the energy row leave 3 unknowns
// (S_u, S_b, d(u)) for EMHD and, after the terms in S_b cancel, one for ideal
// MHD.  The result is the solution of the dense 5x5 or 7x7 system of
// analyticJacobian to rounding.
//
// What it measured against the FP32 Jacobian, equilibration and 5x5 / 7x7 LU
// it replaced (those were bound by vector instruction issue: 1980 VALU
// instructions per wavefront of the ideal solve, 5566 of the EMHD torus
// phase; about 700 and 2800 static ones now): 2^22 ideal zones 252 -> 223 us
// (5.3 TB/s of the algorithmic bytes, above a large copy's 4.9), 70,001 EMHD
// zones 30.9 -> 19.2 us, 700,001 EMHD zones compacted 213 -> 171 us, error
// against the known roots unchanged or smaller.
//
// Every function fixes contraction to single expressions (contract(on)), so
// the kernels that inline them agree bit for bit.
#pragma once
#include <hip/hip_runtime.h>

#include "analytic.hpp"
#include "fast_ops.hpp"
#include "zone_physics.hpp"

namespace grim {

// Per-zone scales of the fused residual and step.
struct ZoneScale {
  double invAlpha;  // 1/alpha
  double scale;     // mask/dt
  double invDt;     // 1/dt
  double invGs;     // 1/(g mask/dt)
  double invDet;    // 1/det(gamma_ij)
};

// What the step reuses of the residual evaluated at the same primitives.
struct FusedPrimal {
  double lor, b0, BB;  // Lorentz factor, b^0, B^i B_i
  double ib, Kq, Kd;   // EMHD: 1/|b|, q = qTilde Kq, dP = dPTilde Kd
};

__device__ __forceinline__ double dot3(const double* a, const double* b) {
#pragma clang fp contract(on)
  return a[0] * b[0] + a[1] * b[1] + a[2] * b[2];
}

// gamma_ij v^j
__device__ __forceinline__ void lower3(const ZoneGeom& G, const double* v, double* out) {
#pragma clang fp contract(on)
#pragma unroll
  for (int i = 0; i < 3; i++)
    out[i] = G.cov(i + 1, 1) * v[0] + G.cov(i + 1, 2) * v[1] + G.cov(i + 1, 3) * v[2];
}

// Cofactors of gamma_ij: gamma^ij = cof / det, packed 11 12 13 22 23 33.
__device__ __forceinline__ void cofactors3(const ZoneGeom& G, double* c) {
#pragma clang fp contract(on)
  c[0] = G.cov(2, 2) * G.cov(3, 3) - G.cov(2, 3) * G.cov(2, 3);
  c[1] = G.cov(1, 3) * G.cov(2, 3) - G.cov(1, 2) * G.cov(3, 3);
  c[2] = G.cov(1, 2) * G.cov(2, 3) - G.cov(1, 3) * G.cov(2, 2);
  c[3] = G.cov(1, 1) * G.cov(3, 3) - G.cov(1, 3) * G.cov(1, 3);
  c[4] = G.cov(1, 2) * G.cov(1, 3) - G.cov(1, 1) * G.cov(2, 3);
  c[5] = G.cov(1, 1) * G.cov(2, 2) - G.cov(1, 2) * G.cov(1, 2);
}

__device__ __forceinline__ void zoneScale(const ZoneGeom& G, double mask, double dt, ZoneScale& s) {
#pragma clang fp contract(on)
  double c[6];
  cofactors3(G, c);
  s.invAlpha = fastRcp(G.alpha);
  s.invDt = fastRcp(dt);
  s.scale = mask * s.invDt;
  s.invGs = fastRcp(G.g * s.scale);
  s.invDet = fastRcp(G.cov(1, 1) * c[0] + G.cov(1, 2) * c[1] + G.cov(1, 3) * c[2]);
}

// The closure of one element (setFluidElementParameters; the torus form
// torus/problem.cpp:7-55) with fast quotients; chi and nu come divided by
// tau, which every consumer forms and in which tau itself cancels.
struct FastClosure {
  double tau, chiOverTau, nuOverTau;
};

template <class L>
__device__ __forceinline__ void fastClosure(double rho, double u, double p, double T, double bsq, double qTilde,
                                            double dPTilde, const DevParams& prm, double alphaC, double alphaV,
                                            double radius, FastClosure& c) {
#pragma clang fp contract(on)
  const double cs2 = prm.gam * p * fastRcp(rho + prm.gam * u);
  // locals, stored once below: members stored branch by branch are merged
  // into stores at a selected address, which keeps c in scratch memory
  double tau, chi, nu;
  if (prm.closure == GRIM_CLOSURE_LINEAR_MODES) {
    tau = 1.;
    chi = nu = cs2;
  } else if (prm.closure == GRIM_CLOSURE_PER_ZONE) {
    tau = prm.tau0;
    chi = alphaC * cs2;
    nu = alphaV * cs2;
  } else if (prm.closure == GRIM_CLOSURE_SHOCK_TESTS) {
    tau = 0.1;
    chi = prm.condAlpha * cs2;
    nu = prm.viscAlpha * cs2;
  } else if (prm.closure == GRIM_CLOSURE_BUOYANCY) {
    tau = fastDiv(1.2 * fastSqrt(radius), cs2);
    chi = cs2 * (1. / 1.2);
    nu = 0.;
  } else {
    const double dyn = radius * fastSqrt(radius);
    tau = dyn;
    if constexpr (L::COND_ON) {
      const double q = prm.highOrderCond ? qTilde * T * fastSqrt(rho * prm.condAlpha * cs2) : qTilde;
      double y = fastDiv(fabs(q), prm.condClosureFactor * rho * (cs2 * fastSqrt(cs2)));
      y = exp((1. - y) * 100.);
      tau = smin(tau, dyn * (fastDiv(y, y + 1.) + 1.e-5));
    }
    if constexpr (L::VISC_ON) {
      const double dP = prm.highOrderVisc ? dPTilde * fastSqrt(T * rho * prm.viscAlpha * cs2) : dPTilde;
      const double dPmod = fastDiv(smax(p - (2. / 3.) * dP, prm.bSqrFloor), smax(p + (1. / 3.) * dP, prm.bSqrFloor));
      const double dPmaxPlus = smin(prm.viscClosureFactor * bsq * 0.5 * dPmod, (1.49 / 1.07) * p);
      const double dPmaxMinus = smax(-prm.viscClosureFactor * bsq, (-2.99 / 1.07) * p);
      const double dPmax = (dP > 0.) ? dPmaxPlus : dPmaxMinus;
      double y = fastDiv(fabs(dP), fabs(dPmax) + prm.bSqrFloor);
      y = exp((1. - y) * 100.);
      tau = smin(tau, dyn * (fastDiv(y, y + 1.) + 1.e-5));
    }
    const double maxAlpha = fastDiv(1. - cs2, 2. * cs2 + 1.e-12);
    chi = smin(maxAlpha, prm.condAlpha) * cs2;
    nu = smin(maxAlpha, prm.viscAlpha) * cs2;
  }
  c.tau = tau;
  c.chiOverTau = chi;
  c.nuOverTau = nu;
}

// Coefficient and old elements of the EMHD rows (elemOld's u_mu and T; the
// weights of the time-derivative sources, emhdWeights): with s_c =
// sqrt(rho chi tau) and s_v = sqrt(rho nu tau / T) of the coefficient element,
//   K_Q rho chi T = s_c, normQ = T s_c, K_DP rho nu = s_v, normDP = T s_v
// for the high-order closure, so no quotient by chi or nu is formed.  The
// coefficient element is the old one when the caller passes the same planes
// (grim's half step), which is evaluated once then.
//
// loadEmhdPlanes takes what it reads from memory, so that the caller can issue
// those loads with its others.
template <class L>
struct EmhdPlanes {
  double old[5], coef[L::DOF];  // elemOld's rho, u, u~^i; the coefficient element's primitives
  double alphaC, alphaV, radius;
};

__device__ __forceinline__ bool coefIsOld(const grim_zone_batch& b) {
  return !b.prim_coef || b.prim_coef == b.prim_old;
}

template <class L>
__device__ __forceinline__ void loadEmhdPlanes(const grim_zone_batch& b, int64_t z, EmhdPlanes<L>& e) {
  const int64_t n = b.n;
  const double* coef = coefIsOld(b) ? b.prim_old : b.prim_coef;
#pragma unroll
  for (int v = 0; v < 5; v++) e.old[v] = b.prim_old[v * n + z];
#pragma unroll
  for (int v = 0; v < L::DOF; v++) e.coef[v] = coef[v * n + z];
  e.alphaC = b.closure ? b.closure[z] : 1.;
  e.alphaV = b.closure ? b.closure[n + z] : 1.;
  e.radius = b.radius ? b.radius[batchGeomIndex(b, z)] : 0.;
}

template <class L>
__device__ __forceinline__ void fusedEmhdConstants(const grim_zone_batch& b, const DevParams& prm, const ZoneGeom& G,
                                                   const EmhdPlanes<L>& e, double invDt, ZoneConst<L>& c,
                                                   EmhdWeights& w) {
#pragma clang fp contract(on)
  c.alphaC = e.alphaC;
  c.alphaV = e.alphaV;
  const double radius = e.radius;
  const double *old = e.old, *P = e.coef;
  double utLow[3];
  double rho = smax(old[RHO], prm.rhoFloor), u = smax(old[UU], prm.uFloor);
  double T = smax(fastDiv((prm.gam - 1.) * u, rho), prm.tFloor);
  lower3(G, old + U1, utLow);
  double lor = fastSqrt(1. + dot3(old + U1, utLow));
  c.oldUCov[0] = G.cov(0, 1) * old[U1] + G.cov(0, 2) * old[U2] + G.cov(0, 3) * old[U3] - G.alpha * lor;
#pragma unroll
  for (int i = 0; i < 3; i++) c.oldUCov[i + 1] = utLow[i];
  c.oldT = T;
  if (!coefIsOld(b)) {
    rho = smax(P[RHO], prm.rhoFloor);
    u = smax(P[UU], prm.uFloor);
    T = smax(fastDiv((prm.gam - 1.) * u, rho), prm.tFloor);
    lower3(G, P + U1, utLow);
    lor = fastSqrt(1. + dot3(P + U1, utLow));
  }
  double BLow[3];
  lower3(G, P + L::B1, BLow);
  const double u0 = fastDiv(lor, G.alpha), invU0 = fastDiv(G.alpha, lor);
  const double b0 = dot3(P + L::B1, utLow);
  const double bsq = (dot3(P + L::B1, BLow) + b0 * b0) * invU0 * invU0 + prm.bSqrFloor;
  const double ib = fastRsqrt(bsq);
  double bCon[4];
  bCon[0] = b0;
  const double ga = lor * G.alpha;
#pragma unroll
  for (int i = 0; i < 3; i++) bCon[i + 1] = (P[L::B1 + i] + b0 * (P[U1 + i] - ga * G.gcon0[i + 1])) * invU0;
  FastClosure cl;
  fastClosure<L>(rho, u, (prm.gam - 1.) * u, T, bsq, L::COND_ON ? P[L::Q] : 0., L::VISC_ON ? P[L::DP] : 0., prm,
                 c.alphaC, c.alphaV, radius, cl);
  const double invTau = fastRcp(cl.tau);
  w.gOverTau = G.g * invTau;
  const double half = 0.5 * G.g;
  if constexpr (L::VISC_ON) {
    const double rn = rho * cl.nuOverTau * cl.tau;
    const double sv = prm.highOrderVisc ? fastSqrt(fastDiv(rn * cl.tau, T)) : rn;
    const double a = w.gOverTau * sv * invDt, f = 3. * b0 * ib * ib;
    const double h = prm.highOrderVisc ? half * invDt * P[L::DP] : 0.;
#pragma unroll
    for (int mu = 0; mu < 4; mu++) w.wDP[mu] = a * (G.gcon0[mu] - f * bCon[mu]) - h * G.gcon0[mu];
    w.sDP = c.mask * (prm.highOrderVisc ? T * sv : cl.tau);
  }
  if constexpr (L::COND_ON) {
    const double rc = rho * cl.chiOverTau * cl.tau;
    const double sc = prm.highOrderCond ? fastSqrt(rc * cl.tau) : rc * T;
    const double a = w.gOverTau * sc * u0 * ib * invDt;
    const double h = prm.highOrderCond ? half * invDt * P[L::Q] : 0.;
#pragma unroll
    for (int nu = 0; nu < 4; nu++) w.wQ[nu] = a * bCon[nu] - h * G.gcon0[nu];
    w.wQT = w.gOverTau * fastDiv(sc, T) * b0 * ib * invDt;
    w.sQ = c.mask * (prm.highOrderCond ? T * sc : cl.tau);
  }
}

// The residual rows (residual<L> up to rounding).
template <class L>
__device__ __forceinline__ void residualFused(const double* P, const ZoneGeom& G, const ZoneConst<L>& c,
                                              const DevParams& prm, const ZoneScale& zs, const EmhdWeights& ew,
                                              double* R, FusedPrimal& f) {
#pragma clang fp contract(on)
  const double rho = smax(P[RHO], prm.rhoFloor);
  const double u = smax(P[UU], prm.uFloor);
  const double *ut = P + U1, *B = P + L::B1;
  const double p = (prm.gam - 1.) * u;
  double utLow[3], BLow[3];
  lower3(G, ut, utLow);
  lower3(G, B, BLow);
  const double lor = fastSqrt(1. + dot3(ut, utLow));
  const double u0 = lor * zs.invAlpha;
  const double invU0 = fastDiv(G.alpha, lor);
  const double uCov0 = G.cov(0, 1) * ut[0] + G.cov(0, 2) * ut[1] + G.cov(0, 3) * ut[2] - G.alpha * lor;
  const double b0 = dot3(B, utLow);
  const double bCov0 = (G.cov(0, 1) * B[0] + G.cov(0, 2) * B[1] + G.cov(0, 3) * B[2] + b0 * uCov0) * invU0;
  const double BB = dot3(B, BLow);
  const double bsq = (BB + b0 * b0) * invU0 * invU0 + prm.bSqrFloor;
  f.lor = lor;
  f.b0 = b0;
  f.BB = BB;
  double Au = (rho + u + p + bsq) * u0, Ab = -b0, E = p + 0.5 * bsq;
  double T = 0.;
  if constexpr (L::EMHD) {
    T = smax(p * fastRcp(rho), prm.tFloor);
    const double rcs2 = rho * (prm.gam * p * fastRcp(rho + prm.gam * u));
    f.ib = fastRsqrt(bsq);
    const double aC = (prm.closure == GRIM_CLOSURE_PER_ZONE) ? c.alphaC : prm.condAlpha;
    const double aV = (prm.closure == GRIM_CLOSURE_PER_ZONE) ? c.alphaV : prm.viscAlpha;
    if constexpr (L::COND_ON) {
      f.Kq = prm.highOrderCond ? T * fastSqrt(rcs2 * aC) : 1.;
      const double qb = P[L::Q] * f.Kq * f.ib;
      Au = Au + qb * b0;
      Ab = Ab + qb * u0;
    }
    if constexpr (L::VISC_ON) {
      f.Kd = prm.highOrderVisc ? fastSqrt(T * (rcs2 * aV)) : 1.;
      const double dP = P[L::DP] * f.Kd, third = dP * (1. / 3.);
      Au = Au + third * u0;
      Ab = Ab - dP * f.ib * f.ib * b0;
      E = E + third;
    }
  }
  const double Urho = G.g * (rho * u0);
  R[RHO] = (Urho - c.rhs[RHO]) * zs.scale;
  R[UU] = (G.g * (Au * uCov0 + Ab * bCov0 + E) + Urho - c.rhs[UU]) * zs.scale;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    const double bCovi = (BLow[i] + b0 * utLow[i]) * invU0;
    R[U1 + i] = (G.g * (Au * utLow[i] + Ab * bCovi) - c.rhs[U1 + i]) * zs.scale;
  }
  if constexpr (L::EMHD) {
    const double du[4] = {uCov0 - c.oldUCov[0], utLow[0] - c.oldUCov[1], utLow[1] - c.oldUCov[2],
                          utLow[2] - c.oldUCov[3]};
    const double gu0 = G.g * u0;
    if constexpr (L::COND_ON) {
      const double std = ew.wQT * (T - c.oldT) + ew.wQ[0] * du[0] + dot3(ew.wQ + 1, du + 1);
      R[L::Q] = ((gu0 * P[L::Q] - c.rhs[L::Q]) * zs.invDt + 0.5 * ew.gOverTau * P[L::Q] + std) * ew.sQ;
    }
    if constexpr (L::VISC_ON) {
      const double std = ew.wDP[0] * du[0] + dot3(ew.wDP + 1, du + 1);
      R[L::DP] = ((gu0 * P[L::DP] - c.rhs[L::DP]) * zs.invDt + 0.5 * ew.gOverTau * P[L::DP] + std) * ew.sDP;
    }
  }
}

// Solves the 3x3 system A x = b by elimination with partial pivoting
// (compare-and-swap, as luSolve).
__device__ __forceinline__ void solve3(double (&A)[3][3], double (&b)[3]) {
#pragma clang fp contract(on)
  auto order = [&](int k, int i) {
    const bool swap = fabs(A[i][k]) > fabs(A[k][k]);
#pragma unroll
    for (int j = k; j < 3; j++) {
      const double hi = A[k][j], lo = A[i][j];
      A[k][j] = swap ? lo : hi;
      A[i][j] = swap ? hi : lo;
    }
    const double hi = b[k], lo = b[i];
    b[k] = swap ? lo : hi;
    b[i] = swap ? hi : lo;
  };
  order(0, 1);
  order(0, 2);
  const double r0 = fastRcp(A[0][0]);
  const double m1 = A[1][0] * r0, m2 = A[2][0] * r0;
  A[1][1] = A[1][1] - m1 * A[0][1];
  A[1][2] = A[1][2] - m1 * A[0][2];
  b[1] = b[1] - m1 * b[0];
  A[2][1] = A[2][1] - m2 * A[0][1];
  A[2][2] = A[2][2] - m2 * A[0][2];
  b[2] = b[2] - m2 * b[0];
  order(1, 2);
  const double r1 = fastRcp(A[1][1]);
  const double m3 = A[2][1] * r1;
  A[2][2] = A[2][2] - m3 * A[1][2];
  b[2] = fastDiv(b[2] - m3 * b[1], A[2][2]);
  b[1] = (b[1] - A[1][2] * b[2]) * r1;
  b[0] = (b[0] - A[0][1] * b[1] - A[0][2] * b[2]) * r0;
}

// d = -J^-1 R at P, whose residual rows are R and whose primal is f.  P is at
// or above its floors (the iteration applies them first).
template <class L>
__device__ __forceinline__ void newtonStep(const double* P, const double* R, const ZoneGeom& G,
                                           const ZoneConst<L>& c, const DevParams& prm, const ZoneScale& zs,
                                           const EmhdWeights& ew, const FusedPrimal& f, double* d) {
#pragma clang fp contract(on)
  const double *ut = P + U1, *B = P + L::B1;
  const double gam = prm.gam, g1 = prm.gam - 1.;
  const double rho = P[RHO], u = P[UU], p = g1 * u;
  const double lor = f.lor, b0 = f.b0, BB = f.BB;
  // right-hand sides in units of U/g; rE is the t-component of T^0_nu
  const double rRho = -R[RHO] * zs.invGs;
  const double r[3] = {-R[U1] * zs.invGs, -R[U2] * zs.invGs, -R[U3] * zs.invGs};
  const double rU = dot3(ut, r), rB = dot3(B, r);
  // r^i = gamma^ij r_j, and beta^i r_i = g_0i r^i (the metric alone, so that
  // the step solves the residual's own system however the planes were rounded)
  double cf[6];
  cofactors3(G, cf);
  const double rc[3] = {(cf[0] * r[0] + cf[1] * r[1] + cf[2] * r[2]) * zs.invDet,
                        (cf[1] * r[0] + cf[3] * r[1] + cf[4] * r[2]) * zs.invDet,
                        (cf[2] * r[0] + cf[4] * r[1] + cf[5] * r[2]) * zs.invDet};
  const double rBeta = G.cov(0, 1) * rc[0] + G.cov(0, 2) * rc[1] + G.cov(0, 3) * rc[2];
  const double e = -R[UU] * zs.invGs - rRho - rBeta;
  const double u0 = lor * zs.invAlpha, invLor = fastRcp(lor), invU0 = G.alpha * invLor;
  const double bb = (BB + b0 * b0) * invU0 * invU0, bsq = bb + prm.bSqrFloor;
  const double hf = rho + u + p + prm.bSqrFloor, w = hf + bb;
  const double c2u0 = hf * u0 * u0 + BB;  // w (u^0)^2 - (b^0)^2
  const double u2 = lor * lor - 1.;
  const double dLor0 = invLor * zs.invAlpha;  // d(u^0) = X dLor0
  double su, sb, ic2, dRho, dU;               // sb multiplies b_i = (B_i + b0 u_i) / u0
  if constexpr (!L::EMHD) {
    ic2 = u0 * fastRcp(c2u0);
    const double ap = gam * p, ihf = fastRcp(hf), q = b0 * invU0;
    const double N = w + (hf - ap) * u2 - ap * ihf * q * q;
    const double K0 = -g1 * (rU + rRho) - gam * u0 * e;
    const double V = (G.alpha * G.alpha * (c2u0 * K0 - BB * rU + b0 * rB * (1. - ap * ihf)) - ap * lor * lor * rU) * fastRcp(N);
    su = V - rU;
    sb = (b0 * invLor * invLor * V - rB) * ihf * invU0;
    const double X = (rU - u2 * su - b0 * G.alpha * lor * sb) * ic2;
    const double Y = (rB - b0 * su - bb * u0 * sb) * ic2;
    const double du0 = X * dLor0;
    dRho = (rRho - rho * du0) * invU0;
    dU = (e + (V + bb * du0 - q * Y) * invU0) * fastRcp(g1);
  } else {
    const double ib = f.ib, ib2 = ib * ib, bn = bsq * ib, q0 = b0 * invU0;
    const double q = L::COND_ON ? P[L::Q] * f.Kq : 0., dP = L::VISC_ON ? P[L::DP] * f.Kd : 0.;
    const double qib = q * ib;
    ic2 = fastRcp(c2u0 * invU0 + 2. * qib * b0 - dP * (b0 * q0 * ib2 - u0 * (1. / 3.)));
    // affine in (1, S_u, S_b |b|): X, Y, Z = beta^i x_i, then d(u^0), d(u_0), d(b^2), d(rho)
    double utLow[3], BLow[3], bh[3];
    lower3(G, ut, utLow);
    lower3(G, B, BLow);
    const double k = invU0 * ib;
#pragma unroll
    for (int i = 0; i < 3; i++) bh[i] = (BLow[i] + b0 * utLow[i]) * k;
    const double uBeta = G.cov(0, 1) * ut[0] + G.cov(0, 2) * ut[1] + G.cov(0, 3) * ut[2];
    const double bBeta = (G.cov(0, 1) * B[0] + G.cov(0, 2) * B[1] + G.cov(0, 3) * B[2] + b0 * uBeta) * k;
    const double aLor = G.alpha * invLor;
    const double X[3] = {rU * ic2, -u2 * ic2, -b0 * G.alpha * lor * ib * ic2};
    const double Y[3] = {rB * ic2, -b0 * ic2, -bb * u0 * ib * ic2};
    const double Z[3] = {rBeta * ic2, -uBeta * ic2, -bBeta * ic2};
    double du0[3], du_0[3], db2[3], dr[3];
#pragma unroll
    for (int s = 0; s < 3; s++) {
      du0[s] = X[s] * dLor0;
      du_0[s] = Z[s] - aLor * X[s];
      db2[s] = 2. * invU0 * (q0 * Y[s] - bb * du0[s]);
      dr[s] = ((s == 0 ? rRho : 0.) - rho * du0[s]) * invU0;
    }
    const double iRho = fastRcp(rho), iU = fastRcp(u), iRG = fastRcp(rho + gam * u);
    const double rawT = p * iRho;
    const bool hot = rawT > prm.tFloor;
    const double sT = hot ? 1. : 0., T = hot ? rawT : prm.tFloor;
    const double idiag = fastRcp(G.g * u0 * zs.invDt + 0.5 * ew.gOverTau);
    // d(q/|b|) and d(dP), affine in (1, S_u, S_b |b|, d(u)); the rows' own
    // unknowns qt, pt likewise
    double dqb[4], dDP[4], qt[4], pt[4];
#pragma unroll
    for (int s = 0; s < 4; s++) dqb[s] = dDP[s] = qt[s] = pt[s] = 0.;
    if constexpr (L::COND_ON) {
      const double lr = prm.highOrderCond ? -sT * iRho + 0.5 * (iRho - iRG) : 0.;
      const double lu = prm.highOrderCond ? sT * iU + 0.5 * rho * iU * iRG : 0.;
      const double gq = G.g * zs.invDt * P[L::Q], wT = ew.wQT * sT * T;
      const double wx[3] = {dot3(ew.wQ + 1, r) * ic2, -dot3(ew.wQ + 1, utLow) * ic2, -dot3(ew.wQ + 1, bh) * ic2};
      const double rQ = -R[L::Q] * fastRcp(ew.sQ);
#pragma unroll
      for (int s = 0; s < 3; s++)
        qt[s] = ((s == 0 ? rQ : 0.) - gq * du0[s] + wT * iRho * dr[s] - ew.wQ[0] * du_0[s] - wx[s]) * idiag;
      qt[3] = -wT * iU * idiag;
#pragma unroll
      for (int s = 0; s < 3; s++) dqb[s] = ib * (f.Kq * qt[s] + q * (lr * dr[s])) - 0.5 * qib * ib2 * db2[s];
      dqb[3] = ib * (f.Kq * qt[3] + q * lu);
    }
    if constexpr (L::VISC_ON) {
      const double lr = prm.highOrderVisc ? 0.5 * (iRho - sT * iRho - iRG) : 0.;
      const double lu = prm.highOrderVisc ? 0.5 * (sT * iU + rho * iU * iRG) : 0.;
      const double gd = G.g * zs.invDt * P[L::DP];
      const double wx[3] = {dot3(ew.wDP + 1, r) * ic2, -dot3(ew.wDP + 1, utLow) * ic2, -dot3(ew.wDP + 1, bh) * ic2};
      const double rD = -R[L::DP] * fastRcp(ew.sDP);
#pragma unroll
      for (int s = 0; s < 3; s++) {
        pt[s] = ((s == 0 ? rD : 0.) - gd * du0[s] - ew.wDP[0] * du_0[s] - wx[s]) * idiag;
        dDP[s] = f.Kd * pt[s] + dP * (lr * dr[s]);
      }
      dDP[3] = dP * lu;
    }
    // the definitions of S_u and S_b |b| and the energy row; the affine
    // constant goes to the right-hand side
    double A[3][3], rhs[3];
    const double dPb = dP * ib2;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      const double x = s < 3 ? du0[s] : 0., y = s < 3 ? Y[s] : 0., b2 = s < 3 ? db2[s] : 0., m = s < 3 ? dr[s] : gam;
      const double e0 = u0 * (m + b2) + (w + dP * (1. / 3.)) * x + (2. * qib - q0 - dPb * q0) * y + b0 * dqb[s] +
                        u0 * (1. / 3.) * dDP[s];
      const double e1 = bn * ((q0 * x - y) * (1. + dPb) + u0 * dqb[s] - b0 * ib2 * (dDP[s] - dPb * b2));
      const double e2 = (s < 3 ? 0.5 * b2 : g1) + dDP[s] * (1. / 3.);
      if (s == 0) {
        rhs[0] = -e0;
        rhs[1] = -e1;
        rhs[2] = e + rU * invU0 - e2;
      } else {
        A[0][s - 1] = e0 - (s == 1 ? 1. : 0.);
        A[1][s - 1] = e1 - (s == 2 ? 1. : 0.);
        A[2][s - 1] = e2 - (s == 1 ? invU0 : 0.);
      }
    }
    solve3(A, rhs);
    su = rhs[0];
    sb = rhs[1] * ib;
    dU = rhs[2];
    dRho = dr[0] + dr[1] * rhs[0] + dr[2] * rhs[1];
    if constexpr (L::COND_ON) d[L::Q] = qt[0] + qt[1] * rhs[0] + qt[2] * rhs[1] + qt[3] * rhs[2];
    if constexpr (L::VISC_ON) d[L::DP] = pt[0] + pt[1] * rhs[0] + pt[2] * rhs[1];
  }
  d[RHO] = dRho;
  d[UU] = dU;
  // d(utilde^i) = gamma^ij x_j
  const double sB = sb * invU0, sU = su + b0 * sB;
#pragma unroll
  for (int i = 0; i < 3; i++) d[U1 + i] = (rc[i] - ut[i] * sU - B[i] * sB) * ic2;
}

}  // namespace grim
