// The fast explicit stage: the two heaviest kernels of grim's stage, the face
// fluxes (riemannSolver::solve with reconstruction, riemannsolver.cpp:
// 202-328) and the explicit sources (fluidElement::computeExplicitSources
// with computeEMHDGradients, physics.cpp:360-586), compiled with
// -ffp-contract=fast-honor-pragmas (fused multiply-adds).
//
// Same mathematics as the exact kernels of step.hip, reorganised for fewer
// instructions:
//  * WENO5 (weno5.cpp:111-257) forms each face value with one division: the
//    nonlinear weights c_k / beta_k^2 and their sum are scaled by
//    16 beta_1^2 beta_2^2 beta_3^2, which leaves products of the betas;
//  * each quotient family with a common divisor (1/u^0 in b^i, 1/|b| and
//    1/b^2 in the stress rows, 1/tau and 1/(rho + Gamma u) in the speeds,
//    1/(2A) for the two roots) takes one reciprocal;
//  * the characteristic speeds read the inverse metric entries the unit
//    covectors pick instead of contracting with zeros;
//  * the sources read the 40 symmetric connection planes once, in one pass
//    over the upper index that feeds both the geometric source and the
//    covariant derivative of u_mu;
//  * a*b + c contracts to a fused multiply-add.
// Rounding differs from grim's order at the 1e-16 relative level; the
// results are tested against the exact kernels and the oracle to 1e-12.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "fast_ops.hpp"
#include "fused.hpp"
#include "grim_hip.h"
#include "runtime.hpp"
#include "step_fast.hpp"
#include "step_physics.hpp"
#include "zone_physics.hpp"

namespace grim {
namespace {

// WENO5 face values of one zone from y[0..4] = in[i-2 .. i+2]: `right` at
// i + 1/2 (grim's primRight), `left` at i - 1/2 (primLeft); a side that is
// not used costs only its own candidates.
// grim's smoothness indicators (weno5.cpp:165-193) are the quadratic forms
// beta_k = 13/12 (second difference)^2 + 1/4 (first-difference combination)^2;
// they are formed here as 12 beta_k (eps2 scaled with them), a factor that
// cancels in the normalised weights.  The weights c_k / beta_k^2 and their
// sum are scaled by beta_1^2 beta_2^2 beta_3^2 and the linear weights folded
// into the candidate stencils, which leaves one quotient per side.
__device__ __forceinline__ void weno5Fast(const double* y, double& left, double& right) {
  const double eps = 12. * 1.0e-17;
  const double y0 = y[0], y1 = y[1], y2 = y[2], y3 = y[3], y4 = y[4];
  const double a12 = fabs(y1) + fabs(y2), a23 = fabs(y2) + fabs(y3);
  const double d1 = y0 - 2. * y1 + y2, e1 = y0 - 4. * y1 + 3. * y2;
  const double d2 = y1 - 2. * y2 + y3, e2 = y1 - y3;
  const double d3 = y2 - 2. * y3 + y4, e3 = 3. * y2 - 4. * y3 + y4;
  const double beta1 = 13. * d1 * d1 + 3. * e1 * e1 + eps * (1. + fabs(y0) + a12);
  const double beta2 = 13. * d2 * d2 + 3. * e2 * e2 + eps * (1. + a12 + fabs(y3));
  const double beta3 = 13. * d3 * d3 + 3. * e3 * e3 + eps * (1. + a23 + fabs(y4));
  const double b1 = beta1 * beta1, b2 = beta2 * beta2, b3 = beta3 * beta3;
  const double p1 = b2 * b3, p2 = b1 * b3, p3 = b1 * b2;
  // linear weights (1, 10, 5) / 16 of the candidates at i + 1/2
  right = fastDiv(p1 * (0.375 * y0 - 1.25 * y1 + 1.875 * y2) + p2 * (-1.25 * y1 + 7.5 * y2 + 3.75 * y3) +
                      p3 * (1.875 * y2 + 3.75 * y3 - 0.625 * y4),
                  p1 + 10. * p2 + 5. * p3);
  // (5, 10, 1) / 16 at i - 1/2
  left = fastDiv(p1 * (-0.625 * y0 + 3.75 * y1 + 1.875 * y2) + p2 * (3.75 * y1 + 7.5 * y2 - 1.25 * y3) +
                     p3 * (1.875 * y2 - 1.25 * y3 + 0.375 * y4),
                 5. * p1 + 10. * p2 + p3);
}

template <int RECON>
__device__ __forceinline__ void faceValues(const double* y, double theta, double& left, double& right) {
  if constexpr (RECON == GRIM_RECON_WENO5)
    weno5Fast(y, left, right);
  else
    reconstructZone<RECON>(y, theta, left, right);
}

// fluidElement::set's kinematics (physics.cpp:60-116) with one reciprocal of
// u^0 for the three b^i.
template <class L>
__device__ __forceinline__ void kinematicsFast(const double* P, const ZoneGeom& G, const DevParams& prm,
                                               Kinematics& k) {
  k.rho = smax(P[RHO], prm.rhoFloor);
  k.u = smax(P[UU], prm.uFloor);
  const double u1 = P[U1], u2 = P[U2], u3 = P[U3];
  const double B1 = P[L::B1], B2 = P[L::B2], B3 = P[L::B3];
  k.pressure = (prm.gam - 1.) * k.u;
  k.temperature = smax(fastDiv(k.pressure, k.rho), prm.tFloor);
  const double gamma = sqrt(1. + G.cov(1, 1) * u1 * u1 + G.cov(2, 2) * u2 * u2 + G.cov(3, 3) * u3 * u3 +
                            2. * (G.cov(1, 2) * u1 * u2 + G.cov(1, 3) * u1 * u3 + G.cov(2, 3) * u2 * u3));
  k.gammaLF = gamma;
  k.uCon[0] = fastDiv(gamma, G.alpha);
  const double invU0 = fastDiv(G.alpha, gamma);
  const double ga = gamma * G.alpha;
  k.uCon[1] = u1 - ga * G.gcon0[1];
  k.uCon[2] = u2 - ga * G.gcon0[2];
  k.uCon[3] = u3 - ga * G.gcon0[3];
#pragma unroll
  for (int mu = 0; mu < 4; mu++)
    k.uCov[mu] = G.cov(mu, 0) * k.uCon[0] + G.cov(mu, 1) * k.uCon[1] + G.cov(mu, 2) * k.uCon[2] +
                 G.cov(mu, 3) * k.uCon[3];
  k.bCon[0] = B1 * k.uCov[1] + B2 * k.uCov[2] + B3 * k.uCov[3];
  k.bCon[1] = (B1 + k.bCon[0] * k.uCon[1]) * invU0;
  k.bCon[2] = (B2 + k.bCon[0] * k.uCon[2]) * invU0;
  k.bCon[3] = (B3 + k.bCon[0] * k.uCon[3]) * invU0;
#pragma unroll
  for (int mu = 0; mu < 4; mu++)
    k.bCov[mu] = G.cov(mu, 0) * k.bCon[0] + G.cov(mu, 1) * k.bCon[1] + G.cov(mu, 2) * k.bCon[2] +
                 G.cov(mu, 3) * k.bCon[3];
  k.bSqr = k.bCon[0] * k.bCov[0] + k.bCon[1] * k.bCov[1] + k.bCon[2] * k.bCov[2] + k.bCon[3] * k.bCov[3] +
           prm.bSqrFloor;
}

// setFluidElementParameters and the rescaled q, deltaP of set() (physics.cpp:
// 118-151; torus closure torus/problem.cpp:7-55), the element's closure with
// unit alphas, as elementClosure.
template <class L>
__device__ __forceinline__ void closureFast(const double* P, const Kinematics& k, const DevParams& prm,
                                            double radius, Closure& c) {
  const double cs2 = fastDiv(prm.gam * k.pressure, k.rho + prm.gam * k.u);
  c.soundSpeed = sqrt(cs2);
  c.bNorm = sqrt(k.bSqr);
  c.q = 0.;
  c.deltaP = 0.;
  c.tau = c.chi = c.nu = 0.;
  if constexpr (L::EMHD) {
    const double aC = prm.condAlpha, aV = prm.viscAlpha;
    if constexpr (L::COND_ON)
      c.q = prm.highOrderCond ? P[L::Q] * k.temperature * sqrt(k.rho * aC * cs2) : P[L::Q];
    if constexpr (L::VISC_ON)
      c.deltaP = prm.highOrderVisc ? P[L::DP] * sqrt(k.temperature * k.rho * aV * cs2) : P[L::DP];
    if (prm.closure == GRIM_CLOSURE_LINEAR_MODES) {
      c.tau = 1.0;
      c.chi = cs2;
      c.nu = cs2;
    } else if (prm.closure == GRIM_CLOSURE_SHOCK_TESTS) {
      c.tau = 0.1;
      c.chi = prm.condAlpha * cs2 * c.tau;
      c.nu = prm.viscAlpha * cs2 * c.tau;
    } else if (prm.closure == GRIM_CLOSURE_BUOYANCY) {
      c.chi = sqrt(radius);
      c.tau = fastDiv(1.2 * c.chi, cs2);
    } else {
      const double dyn = radius * sqrt(radius);
      double tau = dyn;
      const double cs3 = cs2 * c.soundSpeed;
      if constexpr (L::COND_ON) {
        double y = fastDiv(fabs(c.q), prm.condClosureFactor * k.rho * cs3);
        y = exp((1. - y) * 100.);
        tau = smin(tau, dyn * (fastDiv(y, y + 1.) + 1.e-5));
      }
      if constexpr (L::VISC_ON) {
        const double p = k.pressure, dP = c.deltaP, bs = k.bSqr;
        const double dPmod = fastDiv(smax(p - (2. / 3.) * dP, prm.bSqrFloor), smax(p + (1. / 3.) * dP, prm.bSqrFloor));
        const double dPmaxPlus = smin(prm.viscClosureFactor * bs * 0.5 * dPmod, (1.49 / 1.07) * p);
        const double dPmaxMinus = smax(-prm.viscClosureFactor * bs, (-2.99 / 1.07) * p);
        const double dPmax = (dP > 0.) ? dPmaxPlus : dPmaxMinus;
        double y = fastDiv(fabs(dP), fabs(dPmax) + prm.bSqrFloor);
        y = exp((1. - y) * 100.);
        tau = smin(tau, dyn * (fastDiv(y, y + 1.) + 1.e-5));
      }
      c.tau = tau;
      const double maxAlpha = fastDiv(1. - cs2, 2. * cs2 + 1.e-12);
      c.chi = smin(maxAlpha, prm.condAlpha) * cs2 * c.tau;
      c.nu = smin(maxAlpha, prm.viscAlpha) * cs2 * c.tau;
    }
  }
}

// Reciprocals every stress row shares.
struct StressInv {
  double qOverB;   // q / |b|
  double dPOverB2; // deltaP / b^2
};

template <class L>
__device__ __forceinline__ StressInv stressInv(const Kinematics& k, const Closure& c) {
  StressInv s{0., 0.};
  if constexpr (L::COND_ON) s.qOverB = fastDiv(c.q, c.bNorm);
  if constexpr (L::VISC_ON) s.dPOverB2 = fastDiv(c.deltaP, k.bSqr);
  return s;
}

// Row MU of T^mu_nu (physics.cpp:153-178).
template <class L, int MU>
__device__ __forceinline__ void stressRowFast(const Kinematics& k, const Closure& c, const StressInv& si,
                                              double* T) {
  const double w = k.rho + k.u + k.pressure + k.bSqr;
  const double wu = w * k.uCon[MU];
#pragma unroll
  for (int nu = 0; nu < 4; nu++) {
    double t = wu * k.uCov[nu] - k.bCon[MU] * k.bCov[nu];
    if (MU == nu) t += k.pressure + 0.5 * k.bSqr;
    if constexpr (L::COND_ON) t += si.qOverB * (k.uCon[MU] * k.bCov[nu] + k.bCon[MU] * k.uCov[nu]);
    if constexpr (L::VISC_ON)
      t += -si.dPOverB2 * (k.bCon[MU] * k.bCov[nu]) +
           (c.deltaP * (1. / 3.)) * ((MU == nu ? 1. : 0.) + k.uCon[MU] * k.uCov[nu]);
    T[nu] = t;
  }
}

// fluidElement::computeFluxes(DIR) (physics.cpp:185-217); DIR = 0 gives U.
template <class L, int DIR>
__device__ __forceinline__ void fluxesFast(const double* P, const Kinematics& k, const Closure& c,
                                           const StressInv& si, double g, double* F) {
  double T[4];
  stressRowFast<L, DIR>(k, c, si, T);
  const double gu = g * k.uCon[DIR];
  F[RHO] = gu * k.rho;
  F[UU] = g * T[0] + F[RHO];
  F[U1] = g * T[1];
  F[U2] = g * T[2];
  F[U3] = g * T[3];
  // the component along DIR is b^d u^d - b^d u^d = 0 exactly, as grim
  // computes it (a contracted b^d u^d - b^d u^d would leave the product's
  // rounding error)
#pragma unroll
  for (int c = 1; c <= 3; c++)
    F[L::B1 + c - 1] = (c == DIR) ? 0. : g * (k.bCon[c] * k.uCon[DIR] - k.bCon[DIR] * k.uCon[c]);
  if constexpr (L::COND_ON) F[L::Q] = gu * P[L::Q];
  if constexpr (L::VISC_ON) F[L::DP] = gu * P[L::DP];
}

// The geometry one side of a face needs: the zone geometry, the inverse
// metric entry g^{ss} of the face direction and r (the torus closure).
struct FaceGeom {
  ZoneGeom zg;
  double gconSS, r;
};

template <int DIR>
__device__ __forceinline__ void loadFaceGeom(const double* geom, int64_t n, uint32_t zb, FaceGeom& G) {
#pragma unroll
  for (int k = 0; k < 10; k++) G.zg.gcov[k] = ldOff(geom + k * n, zb);
#pragma unroll
  for (int k = 0; k < 4; k++) G.zg.gcon0[k] = ldOff(geom + (GEOM_GCON0 + k) * n, zb);
  G.zg.alpha = ldOff(geom + GEOM_ALPHA * n, zb);
  G.zg.g = ldOff(geom + GEOM_G * n, zb);
  // planes 16..21 hold g^{11} g^{12} g^{13} g^{22} g^{23} g^{33}
  constexpr int ss = DIR == 0 ? 0 : (DIR == 1 ? 3 : 5);
  G.gconSS = ldOff(geom + (16 + ss) * n, zb);
  G.r = ldOff(geom + LOC_R * n, zb);
}

// The element of one face value (fluidElement::set, physics.cpp:53-183), its
// computeFluxes(DIR + 1) and computeFluxes(0) (:185-217) and its speeds along
// DIR (computeMinMaxCharSpeeds, riemannsolver.cpp:54-200).
//
// In the identity form of the solve's residual (fused.hpp): lowered spatial
// vectors from gamma_ij, b_mu = (B_mu + b^0 u_mu)/u^0, and the two rows of
// T^mu_nu as A^mu u_nu + C^mu b_nu + d^mu_nu E, so no other contravariant
// component is formed.  The conserved field is g (b^i u^0 - b^0 u^i) = g B^i,
// its flux g (B^c u^d - B^d u^c)/u^0.  The speeds read chi/tau and nu/tau,
// in which tau cancels: the torus closure's two exponentials do not enter
// the fluxes.  The unit covectors of the speeds pick single entries of the
// inverse metric.  (Against the reference's order of operations this took
// the two states of a face from 2,750 to about 1,600 VALU instructions.)
//
// The results go to `out` one by one, first the speeds, out.speeds(mn, mx),
// then out.row(v, F_v, U_v) without the common factor g: a consumer that
// combines each row at once never holds all of them.
template <class L, int DIR, class Out>
__device__ __forceinline__ void faceElement(const double* P, const FaceGeom& fg, const DevParams& prm, Out&& out) {
  constexpr int D = DIR + 1;
  const ZoneGeom& G = fg.zg;
  const double rho = smax(P[RHO], prm.rhoFloor), u = smax(P[UU], prm.uFloor);
  const double *ut = P + U1, *B = P + L::B1;
  const double p = (prm.gam - 1.) * u;
  double utLow[3], BLow[3];
  lower3(G, ut, utLow);
  lower3(G, B, BLow);
  const double lor = fastSqrt(1. + dot3(ut, utLow));
  const double u0 = fastDiv(lor, G.alpha), invU0 = fastDiv(G.alpha, lor), ga = lor * G.alpha;
  double uc[3];  // u^1..u^3
#pragma unroll
  for (int i = 0; i < 3; i++) uc[i] = ut[i] - ga * G.gcon0[i + 1];
  const double ud = uc[DIR];
  double uCov[4], bCov[4];
  uCov[0] = G.cov(0, 1) * ut[0] + G.cov(0, 2) * ut[1] + G.cov(0, 3) * ut[2] - G.alpha * lor;
  const double b0 = dot3(B, utLow), bd = (B[DIR] + b0 * ud) * invU0;
  bCov[0] = (G.cov(0, 1) * B[0] + G.cov(0, 2) * B[1] + G.cov(0, 3) * B[2] + b0 * uCov[0]) * invU0;
#pragma unroll
  for (int i = 0; i < 3; i++) {
    uCov[i + 1] = utLow[i];
    bCov[i + 1] = (BLow[i] + b0 * utLow[i]) * invU0;
  }
  const double bsq = (dot3(B, BLow) + b0 * b0) * invU0 * invU0 + prm.bSqrFloor;
  const double rhoGu = rho + prm.gam * u, invRhoGu = fastRcp(rhoGu);
  const double cs2 = prm.gam * p * invRhoGu;
  const double w = rho + u + p + bsq;
  double Ad = w * ud, A0 = w * u0, Cd = -bd, C0 = -b0, E = p + 0.5 * bsq;
  double conSqr = 0., visSqr = 0.;
  if constexpr (L::EMHD) {
    const double T = smax(p * fastRcp(rho), prm.tFloor), ib = fastRsqrt(bsq);
    FastClosure cl;
    fastClosure<L>(rho, u, p, T, bsq, 0., 0., prm, 1., 1., fg.r, cl);
    if constexpr (L::COND_ON) {
      const double qb = (prm.highOrderCond ? P[L::Q] * T * fastSqrt(rho * prm.condAlpha * cs2) : P[L::Q]) * ib;
      Ad = Ad + qb * bd;
      A0 = A0 + qb * b0;
      Cd = Cd + qb * ud;
      C0 = C0 + qb * u0;
      conSqr = (prm.gam - 1.) * cl.chiOverTau;
    }
    if constexpr (L::VISC_ON) {
      const double dP = prm.highOrderVisc ? P[L::DP] * fastSqrt(T * rho * prm.viscAlpha * cs2) : P[L::DP];
      const double third = dP * (1. / 3.), dPb = dP * ib * ib;
      Ad = Ad + third * ud;
      A0 = A0 + third * u0;
      Cd = Cd - dPb * bd;
      C0 = C0 - dPb * b0;
      E = E + third;
      visSqr = (4. / 3.) * rho * cl.nuOverTau * invRhoGu;
    }
  }
  {
    const double alfSqr = bsq * fastRcp(rhoGu + bsq);
    double cSqr = 0.5 * (cs2 + conSqr + fastSqrt(cs2 * cs2 + conSqr * conSqr)) + visSqr;
    cSqr = cSqr + alfSqr - cSqr * alfSqr;
    cSqr = cSqr > 1. ? 1. : cSqr;
    const double A = u0 * u0 - (G.gcon0[0] + u0 * u0) * cSqr;
    const double Bq = 2. * (ud * u0 - (G.gcon0[D] + ud * u0) * cSqr);
    const double C = ud * ud - (fg.gconSS + ud * ud) * cSqr;
    const double discr = fastSqrt(smax(Bq * Bq - 4. * A * C, 1.e-16));
    const double inv2A = 0.5 * fastRcp(A);
    const double mn = (Bq - discr) * inv2A, mx = (Bq + discr) * inv2A;
    out.speeds(mn > -1.e-15 ? -1.e-15 : mn, mx < 1.e-15 ? 1.e-15 : mx);
  }
  const double Frho = rho * ud, Urho = rho * u0;
  out.row(RHO, Frho, Urho);
  out.row(UU, Ad * uCov[0] + Cd * bCov[0] + Frho, A0 * uCov[0] + C0 * bCov[0] + E + Urho);
#pragma unroll
  for (int nu = 1; nu < 4; nu++)
    out.row(UU + nu, Ad * uCov[nu] + Cd * bCov[nu] + (nu == D ? E : 0.), A0 * uCov[nu] + C0 * bCov[nu]);
  if constexpr (L::COND_ON) out.row(L::Q, ud * P[L::Q], u0 * P[L::Q]);
  if constexpr (L::VISC_ON) out.row(L::DP, ud * P[L::DP], u0 * P[L::DP]);
#pragma unroll
  for (int c = 0; c < 3; c++)
    out.row(L::B1 + c, c == DIR ? 0. : (B[c] * ud - B[DIR] * uc[c]) * invU0, B[c]);
}

// A face's left state in LDS, each entry a row over the workgroup's lanes:
// the conserved variables, the two speeds and the fluxes but that of the
// field along DIR, which is zero.
template <class L, int LANES>
using FaceSlots = double[2 * L::DOF + 1][LANES];

// Row of flux v, and whether it has one.
template <class L, int DIR>
__device__ __forceinline__ int fluxSlot(int v) {
  return L::DOF + 2 + (v > L::B1 + DIR ? v - 1 : v);
}
template <class L, int DIR>
__device__ __forceinline__ bool noFlux(int v) {
  return v == L::B1 + DIR;
}

template <class L, int DIR, int LANES>
struct StoreSide {
  FaceSlots<L, LANES>& sh;
  int slot;
  __device__ __forceinline__ void speeds(double mn, double mx) {
    sh[L::DOF][slot] = mn;
    sh[L::DOF + 1][slot] = mx;
  }
  __device__ __forceinline__ void row(int v, double F, double U) {
    sh[v][slot] = U;
    if (!noFlux<L, DIR>(v)) sh[fluxSlot<L, DIR>(v)][slot] = F;
  }
};

// The right state of a face on its way out of faceElement: the HLL or LLF
// flux of each row against the left state in LDS (riemannsolver.cpp:270-328),
// stored at byte offset zb of its flux plane.
template <class L, int DIR, int LANES>
struct SolveFace {
  const StepArgs& a;
  FaceSlots<L, LANES>& sh;
  int slot;
  double metric;
  double* flux;
  uint32_t zb;
  double mn, mx, k, b;  // speeds; HLL: g/(mx - mn) and mn mx, LLF: g/2 and the largest speed
  __device__ __forceinline__ void speeds(double mnR, double mxR) {
    mn = stdmin(sh[L::DOF][slot], mnR);
    mx = stdmax(sh[L::DOF + 1][slot], mxR);
    const bool hll = a.riemann == GRIM_RIEMANN_HLL;
    k = hll ? metric * fastRcp(mx - mn) : 0.5 * metric;
    b = hll ? mn * mx : stdmax(mx, -mn);
  }
  __device__ __forceinline__ void row(int v, double FR, double UR) {
    const double FL = noFlux<L, DIR>(v) ? 0. : sh[fluxSlot<L, DIR>(v)][slot], UL = sh[v][slot];
    const double f = a.riemann == GRIM_RIEMANN_HLL ? mx * FL - mn * FR + b * (UR - UL) : FL + FR - b * (UR - UL);
    stOff(flux + v * a.D.n, zb, f * k);
  }
};

// A state held in registers until its partner is in LDS.
template <class L>
struct HoldSide {
  double F[L::DOF], U[L::DOF], mn, mx;
  __device__ __forceinline__ void speeds(double a, double b) {
    mn = a;
    mx = b;
  }
  __device__ __forceinline__ void row(int v, double f, double u) {
    F[v] = f;
    U[v] = u;
  }
  template <class Out>
  __device__ __forceinline__ void to(Out&& out) const {
    out.speeds(mn, mx);
#pragma unroll
    for (int v = 0; v < L::DOF; v++) out.row(v, F[v], U[v]);
  }
};

// The face values of every variable of the zone at byte offset zb.
template <class L, int DIR, int RECON>
__device__ __forceinline__ void reconstructBoth(const StepArgs& a, const double* __restrict__ prim, uint32_t zb,
                                                double* left, double* right) {
  const int64_t n = a.D.n;
  uint32_t off[5];
#pragma unroll
  for (int q = 0; q < 5; q++) off[q] = zb + (uint32_t)((q - 2) * a.D.s[DIR] * 8);
  // Two variables' stencils are in flight while the two before them are
  // reconstructed; pinning each result keeps the compiler from issuing every
  // variable's loads first, which would hold 50 values in registers.
  constexpr int GROUP = 2, GROUPS = (L::DOF + GROUP - 1) / GROUP;
  double y[2][GROUP][5];
  auto load = [&](int g) {
#pragma unroll
    for (int e = 0; e < GROUP; e++)
#pragma unroll
      for (int q = 0; q < 5; q++)
        if (g * GROUP + e < L::DOF) y[g & 1][e][q] = ldOff(prim + (g * GROUP + e) * n, off[q]);
  };
  load(0);
#pragma unroll
  for (int g = 0; g < GROUPS; g++) {
    if (g + 1 < GROUPS) load(g + 1);
#pragma unroll
    for (int e = 0; e < GROUP; e++) {
      const int v = g * GROUP + e;
      if (v >= L::DOF) continue;
      faceValues<RECON>(y[g & 1][e], a.theta, left[v], right[v]);
      asm volatile("" : "+v"(left[v]), "+v"(right[v]));
    }
  }
}

// X1 faces of large grids.  A lane takes one zone: both its face values from
// one set of smoothness indicators, then the elements of both.  The state it
// leaves right of itself is the next lane's left state, read from LDS within
// the wavefront (no barrier), so no state is built twice.  The zones of all
// rows (one more than the faces of a row) are numbered through; a wavefront
// takes 63 of them and the one before.  Bound by FP64 issue (1,660
// instructions per zone, about 210 us of 350 at 192x192x128 zones, EMHD; 510
// with two threads per face) and by the 780 MB it moves; a fourth wavefront
// per SIMD (blocks of 64) adds nothing.
constexpr int kRowBlock = 128;
template <class L, int RECON>
__global__ __launch_bounds__(kRowBlock) __attribute__((amdgpu_waves_per_eu(3))) void faceFluxRowKernel(
    StepArgs a, Box box, const double* __restrict__ prim, const double* __restrict__ geomFace,
    double* __restrict__ flux) {
  __shared__ FaceSlots<L, kRowBlock> sh;
  const int lane = threadIdx.x & 63;
  const unsigned wave = blockIdx.x * (kRowBlock / 64) + (threadIdx.x >> 6);
  const unsigned rowZones = (unsigned)(box.hi[0] - box.lo[0]) + 1u, rows1 = (unsigned)(box.hi[1] - box.lo[1]);
  const unsigned total = rowZones * rows1 * (unsigned)(box.hi[2] - box.lo[2]);
  const unsigned t = wave * 63u + (unsigned)lane;
  if (t >= total) return;
  const unsigned row = t / rowZones, iz = t % rowZones;
  const uint32_t i = (uint32_t)box.lo[0] - 1u + iz;
  const uint32_t zgb = (i + (uint32_t)(box.lo[1] + (int)(row % rows1)) * (uint32_t)a.D.s[1]) * 8u;
  const uint32_t zb = zgb + (uint32_t)(box.lo[2] + (int)(row / rows1)) * (uint32_t)a.D.s[2] * 8u;
  double left[L::DOF], right[L::DOF];
  reconstructBoth<L, 0, RECON>(a, prim, zb, left, right);
  FaceGeom G;
  loadFaceGeom<0>(geomFace, a.D.ng, zgb + 8u, G);  // the face right of the zone
  faceElement<L, 0>(right, G, a.prm, StoreSide<L, 0, kRowBlock>{sh, (int)threadIdx.x});
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (lane == 0 || iz == 0) return;
  loadFaceGeom<0>(geomFace, a.D.ng, zgb, G);
  faceElement<L, 0>(left, G, a.prm, SolveFace<L, 0, kRowBlock>{a, sh, (int)threadIdx.x - 1, G.zg.g, flux, zb});
}

// X2 and X3 faces of large grids.  A lane walks `steps` faces along DIR in
// one (X1, other) column with the five stencil values of every variable in
// registers, so each primitive is loaded once per walk (and four more at its
// start), one zone ahead of its use; it keeps the state right of the zone it
// has just left (in its own LDS slots) for the next face, so each zone's
// indicators and elements are formed once.  That takes 224 registers, two
// wavefronts per SIMD; loading the stencils again for every zone leaves room
// for three but reads each value five times, mostly past the L2 (a lane's
// column is its own): 482 and 553 us for X2 and X3 of 192x192x128 EMHD zones
// against 377 and 382 (510 and 525 with two threads per face).  Bound by FP64
// issue as the X1 kernel.
template <class L, int DIR, int RECON>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2))) void faceFluxMarchKernel(
    StepArgs a, Box box, int steps, const double* __restrict__ prim, const double* __restrict__ geomFace,
    double* __restrict__ flux) {
  __shared__ FaceSlots<L, kBlock> sh;
  constexpr int OTHER = 3 - DIR;
  const int64_t n = a.D.n;
  const unsigned ni = (unsigned)(box.hi[0] - box.lo[0]);
  const unsigned cols = ni * (unsigned)(box.hi[OTHER] - box.lo[OTHER]);
  const unsigned perSeg = (cols + kBlock - 1) / kBlock;
  const unsigned seg = blockIdx.x / perSeg;
  const unsigned c = (blockIdx.x % perSeg) * kBlock + threadIdx.x;
  if (c >= cols) return;
  const int slot = (int)threadIdx.x;
  const int first = box.lo[DIR] + (int)seg * steps;
  const int last = min(first + steps, box.hi[DIR]);  // faces [first, last)
  const uint32_t sB = (uint32_t)a.D.s[DIR] * 8u;
  // bytes from one face to the next in a geometry plane (X3: the same column)
  const uint32_t gB = DIR == 1 ? sB : 0u;
  const uint32_t other = (uint32_t)(box.lo[OTHER] + (int)(c / ni));
  uint32_t zgb = ((uint32_t)box.lo[0] + c % ni) * 8u + (DIR == 1 ? (uint32_t)first * sB : other * (uint32_t)a.D.s[1] * 8u);
  uint32_t zb = ((uint32_t)box.lo[0] + c % ni) * 8u + other * (uint32_t)a.D.s[OTHER] * 8u + (uint32_t)first * sB;
  // the zone before the first face, then each zone of the walk: its left
  // state closes a face, its right state opens the next
  double y[L::DOF][5];
  zb -= sB;
#pragma unroll
  for (int v = 0; v < L::DOF; v++)
#pragma unroll
    for (int q = 0; q < 5; q++) y[v][q] = ldOff(prim + v * n, zb + (uint32_t)((q - 2) * a.D.s[DIR] * 8));
  for (int f = first - 1; f < last; f++) {
    const bool more = f + 1 < last;
    double next[L::DOF], left[L::DOF], right[L::DOF];
    if (more) {
#pragma unroll
      for (int v = 0; v < L::DOF; v++) next[v] = ldOff(prim + v * n, zb + 3 * sB);
    }
    FaceGeom G;
    if (f >= first) loadFaceGeom<DIR>(geomFace, a.D.ng, zgb, G);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int v = 0; v < L::DOF; v++) {
      faceValues<RECON>(y[v], a.theta, left[v], right[v]);
      asm volatile("" : "+v"(left[v]), "+v"(right[v]));
    }
    if (f >= first) {
      faceElement<L, DIR>(left, G, a.prm, SolveFace<L, DIR, kBlock>{a, sh, slot, G.zg.g, flux, zb});
      zgb += gB;
    }
    if (more) {
      loadFaceGeom<DIR>(geomFace, a.D.ng, zgb, G);
      faceElement<L, DIR>(right, G, a.prm, StoreSide<L, DIR, kBlock>{sh, slot});
#pragma unroll
      for (int v = 0; v < L::DOF; v++) {
#pragma unroll
        for (int q = 0; q < 4; q++) y[v][q] = y[v][q + 1];
        y[v][4] = next[v];
      }
    }
    zb += sB;
  }
}

// Small grids: two threads per face, wavefronts 0-1 of a workgroup the left
// states, 2-3 the right states, which meet in LDS (as the split face kernel of
// step.hip): twice the wavefronts, each half as long.
template <class L, int DIR, int RECON>
__global__ __launch_bounds__(kBlock) void faceFluxFastKernel(StepArgs a, Box box, const double* __restrict__ prim,
                                                             const double* __restrict__ geomFace,
                                                             double* __restrict__ flux) {
  __shared__ FaceSlots<L, kFacesPerBlock> sh;
  const int side = threadIdx.x / kFacesPerBlock;
  const int lf = threadIdx.x % kFacesPerBlock;
  const int64_t f = (int64_t)blockIdx.x * kFacesPerBlock + lf;
  const bool active = f < box.count();
  uint32_t zb = 0;
  double P[L::DOF], unused[L::DOF];
  FaceGeom G;
  if (active) {
    int i, j, k;
    box.at(f, i, j, k);
    const uint32_t zgb = ((uint32_t)i + (uint32_t)j * (uint32_t)a.D.s[1]) * 8u;
    zb = zgb + (uint32_t)k * (uint32_t)a.D.s[2] * 8u;
    if (side == 0)
      reconstructBoth<L, DIR, RECON>(a, prim, zb - (uint32_t)a.D.s[DIR] * 8u, unused, P);
    else
      reconstructBoth<L, DIR, RECON>(a, prim, zb, P, unused);
    loadFaceGeom<DIR>(geomFace, a.D.ng, zgb, G);
  }
  HoldSide<L> s;
  if (active) {
    faceElement<L, DIR>(P, G, a.prm, s);
    if (side == 0) s.to(StoreSide<L, DIR, kFacesPerBlock>{sh, lf});
  }
  __syncthreads();
  if (active && side == 1) s.to(SolveFace<L, DIR, kFacesPerBlock>{a, sh, lf, G.zg.g, flux, zb});
}

__host__ __device__ constexpr int sym4(int k, int m) {
  return (k < m ? k : m) * 4 - ((k < m ? k : m) * ((k < m ? k : m) + 1)) / 2 + (k < m ? m : k);
}

// computeExplicitSources (physics.cpp:360-586) for the bulk zones of box:
// one pass over the connection's upper index l, whose 10 symmetric planes
// feed the geometric source -g T^k_l Gamma^l_{k n} and the covariant
// derivative u_{mu;nu} = d_nu u_mu - Gamma^l_{nu mu} u_l; the old implicit
// sources with the stage element's tau; on the half stage consOld.
template <class L, int RECON>
__global__ __launch_bounds__(kBlock) void sourcesFastKernel(StepArgs a, Box box, const double* __restrict__ prim,
                                                            const double* __restrict__ primOld,
                                                            const double* __restrict__ geomC,
                                                            const double* __restrict__ gamma40,
                                                            const double* __restrict__ uT, double* __restrict__ sExp,
                                                            double* __restrict__ sImp, double* __restrict__ consOld) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= box.count()) return;
  int i, j, k;
  box.at(t, i, j, k);
  const Dims& D = a.D;
  const int64_t n = D.n, z = flatIndex(D, i, j, k);
  const int64_t ng = D.ng, zg = geomIndex(D, i, j);
  double P[L::DOF];
#pragma unroll
  for (int v = 0; v < L::DOF; v++) P[v] = prim[v * n + z];
  GeomFull G;
  loadGeomFull(geomC, ng, zg, G);
  Kinematics kk;
  Closure cc;
  kinematicsFast<L>(P, G.zg, a.prm, kk);
  closureFast<L>(P, kk, a.prm, G.r, cc);
  const StressInv si = stressInv<L>(kk, cc);
  const double g = G.zg.g;
  if (consOld) {
    double U[L::DOF];
    fluxesFast<L, 0>(P, kk, cc, si, g, U);
#pragma unroll
    for (int v = 0; v < L::DOF; v++) consOld[v * n + z] = U[v];
  }
  double src[L::NF];
#pragma unroll
  for (int v = 0; v < L::NF; v++) src[v] = 0.;
  const bool curved = a.metric != GRIM_METRIC_MINKOWSKI;
  // T^k_l, k-major
  double T[4][4];
  if (curved) {
    stressRowFast<L, 0>(kk, cc, si, T[0]);
    stressRowFast<L, 1>(kk, cc, si, T[1]);
    stressRowFast<L, 2>(kk, cc, si, T[2]);
    stressRowFast<L, 3>(kk, cc, si, T[3]);
  }
  double graduCov[4][4];
  if constexpr (L::EMHD) {
    auto slopeOf = [&](const double* arr, int d) {
      double y[5];
#pragma unroll
      for (int q = 0; q < 5; q++) y[q] = arr[z + (q - 2) * D.s[d]];
      return slopeZone<RECON>(y, a.theta, a.dX[d]);
    };
#pragma unroll
    for (int mu = 0; mu < 4; mu++) {
      const double* um = uT + mu * n;
      graduCov[0][mu] = 0.;
      graduCov[1][mu] = slopeOf(um, 0);
      graduCov[2][mu] = D.dim > 1 ? slopeOf(um, 1) : 0.;
      graduCov[3][mu] = D.dim > 2 ? slopeOf(um, 2) : 0.;
    }
  }
  if (curved || L::EMHD) {
#pragma unroll
    for (int l = 0; l < 4; l++) {
      double gam[10];
#pragma unroll
      for (int q = 0; q < 10; q++) gam[q] = gamma40[(l * 10 + q) * ng + zg];
      if (curved) {
#pragma unroll
        for (int nu = 0; nu < 4; nu++) {
          double s = 0.;
#pragma unroll
          for (int kap = 0; kap < 4; kap++) s += T[kap][l] * gam[sym4(kap, nu)];
          src[UU + nu] -= g * s;
        }
      }
      if constexpr (L::EMHD) {
        const double ul = kk.uCov[l];
#pragma unroll
        for (int nu = 0; nu < 4; nu++)
#pragma unroll
          for (int mu = 0; mu < 4; mu++) graduCov[nu][mu] -= gam[sym4(nu, mu)] * ul;
      }
    }
  }
  if constexpr (L::EMHD) {
    double divuCov = 0.;
#pragma unroll
    for (int mu = 0; mu < 4; mu++)
#pragma unroll
      for (int nu = 0; nu < 4; nu++) divuCov += G.con(mu, nu) * graduCov[mu][nu];
    const double invTau = 1. / cc.tau;
    if constexpr (L::VISC_ON) {
      const double rn = kk.rho * cc.nu;
      const double c3 = 3. * rn / kk.bSqr;
      double bb = 0.;
#pragma unroll
      for (int mu = 0; mu < 4; mu++)
#pragma unroll
        for (int nu = 0; nu < 4; nu++) bb += kk.bCon[mu] * kk.bCon[nu] * graduCov[mu][nu];
      double deltaP0 = -divuCov * rn + c3 * bb;
      if (a.prm.highOrderVisc == 1) deltaP0 = deltaP0 * sqrt(cc.tau / (rn * kk.temperature));
      double sd = -g * deltaP0 * invTau;
      if (a.prm.highOrderVisc == 1) sd -= 0.5 * g * divuCov * P[L::DP];
      src[L::DP] = sd;
    }
    if constexpr (L::COND_ON) {
      const double* Tp = uT + 4 * n;
      double gradT[4];
      gradT[0] = 0.;
      {
        double y[5];
#pragma unroll
        for (int q = 0; q < 5; q++) y[q] = Tp[z + (q - 2) * D.s[0]];
        gradT[1] = slopeZone<RECON>(y, a.theta, a.dX[0]);
      }
      gradT[2] = 0.;
      gradT[3] = 0.;
      if (D.dim > 1) {
        double y[5];
#pragma unroll
        for (int q = 0; q < 5; q++) y[q] = Tp[z + (q - 2) * D.s[1]];
        gradT[2] = slopeZone<RECON>(y, a.theta, a.dX[1]);
      }
      if (D.dim > 2) {
        double y[5];
#pragma unroll
        for (int q = 0; q < 5; q++) y[q] = Tp[z + (q - 2) * D.s[2]];
        gradT[3] = slopeZone<RECON>(y, a.theta, a.dX[2]);
      }
      // q0 = -rho chi / |b| (b^mu d_mu T + T b^nu u^mu u_{nu;mu})
      const double rcb = kk.rho * cc.chi / cc.bNorm;
      double bgT = 0., buu = 0.;
#pragma unroll
      for (int mu = 0; mu < 4; mu++) {
        bgT += kk.bCon[mu] * gradT[mu];
#pragma unroll
        for (int nu = 0; nu < 4; nu++) buu += kk.bCon[nu] * kk.uCon[mu] * graduCov[mu][nu];
      }
      double q0 = -rcb * (bgT + kk.temperature * buu);
      if (a.prm.highOrderCond == 1) q0 = q0 * sqrt(cc.tau / (kk.rho * cc.chi)) / kk.temperature;
      double sq = -g * q0 * invTau;
      if (a.prm.highOrderCond == 1) sq -= 0.5 * g * divuCov * P[L::Q];
      src[L::Q] = sq;
    }
    if (sImp) {
#pragma unroll
      for (int v = 0; v < L::NF; v++) sImp[v * n + z] = 0.;
      const double gt = g * invTau;
      if constexpr (L::VISC_ON) sImp[L::DP * n + z] = gt * primOld[L::DP * n + z];
      if constexpr (L::COND_ON) sImp[L::Q * n + z] = gt * primOld[L::Q * n + z];
    }
  }
#pragma unroll
  for (int v = 0; v < L::NF; v++) sExp[v * n + z] = src[v];
}

__global__ __launch_bounds__(kBlock) void gamma40Kernel(int64_t n, const double* __restrict__ g64,
                                                        double* __restrict__ g40) {
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (z >= n) return;
#pragma unroll
  for (int l = 0; l < 4; l++)
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int m = k; m < 4; m++) g40[(l * 10 + sym4(k, m)) * n + z] = g64[(l * 16 + k * 4 + m) * n + z];
}

inline unsigned blocks(int64_t count, int per) { return (unsigned)((count + per - 1) / per); }

}  // namespace

// Faces from which X1's fluxes go by rows of zones, and X2's and X3's by walks,
// instead of two threads per face.  EMHD, WENO5, both kernels, us per call:
//   faces           32,768  110,592  262,144  512,000  884,736  1.6 M  4.7 M
//   X1 split          13.3     24.8     43.5     74.4      117    225    612
//   X1 rows           13.9     21.5     36.2     57.9       88    166    482
//   X2 split          13.4     24.9     47.4     82.3      126    218    643
//   X2 walks          28.2     32.8     53.8     80.1      110    181    461
// (X3 as X2; with 110 us of other work in the last column).  A walk is a serial
// chain of its faces: below half a million faces too few are in flight.
constexpr int64_t kRowFaces = 1 << 16;
constexpr int64_t kMarchFaces = 1 << 19;
// Wavefronts that a launch of walks should keep: two fit a SIMD at a time, so
// this is four rounds of the chip; fewer and longer walks (6144) are no faster.
constexpr int64_t kMarchWaves = 8192;

int launchFaceFast(const grim_params& p, const StepArgs& a, int dir, int recon, const Box& b, const double* prim,
                   const double* geomFace, double* flux, hipStream_t s) {
  GRIM_REQUIRE(planeOffsetsFit(a.D.n), "fast explicit stage: planes must hold fewer than 2^29 zones");
  const int64_t faces = b.count();
  // zones one face before the box belong to the grid (the stencil reaches two
  // further), so a walk may start from them
  const bool large = faces >= (dir == 0 ? kRowFaces : kMarchFaces);
  return dispatchLayout(p, [&]<class L>() -> int {
    auto go = [&]<int DIR, int RECON>() {
      if (!large) {
        faceFluxFastKernel<L, DIR, RECON><<<blocks(faces, kFacesPerBlock), kBlock, 0, s>>>(a, b, prim, geomFace, flux);
      } else if constexpr (DIR == 0) {
        const int64_t rows = (int64_t)(b.hi[1] - b.lo[1]) * (b.hi[2] - b.lo[2]);
        const int64_t waves = (rows * (b.hi[0] - b.lo[0] + 1) + 62) / 63;
        faceFluxRowKernel<L, RECON><<<blocks(waves, kRowBlock / 64), kRowBlock, 0, s>>>(a, b, prim, geomFace, flux);
      } else {
        const int len = b.hi[DIR] - b.lo[DIR];
        const int64_t cols = faces / len;
        int64_t steps = cols * len / (kMarchWaves * 64);
        steps = std::max<int64_t>(4, std::min<int64_t>(16, steps));
        const int segs = (int)((len + steps - 1) / steps);
        const int even = (len + segs - 1) / segs;  // the walks of a column of like length
        const unsigned nb = blocks(cols, kBlock) * (unsigned)((len + even - 1) / even);
        faceFluxMarchKernel<L, DIR, RECON><<<nb, kBlock, 0, s>>>(a, b, even, prim, geomFace, flux);
      }
    };
    auto byRecon = [&]<int DIR>() {
      if (recon == GRIM_RECON_WENO5) go.template operator()<DIR, GRIM_RECON_WENO5>();
      else if (recon == GRIM_RECON_PPM) go.template operator()<DIR, GRIM_RECON_PPM>();
      else go.template operator()<DIR, GRIM_RECON_MINMOD>();
    };
    if (dir == 0) byRecon.template operator()<0>();
    else if (dir == 1) byRecon.template operator()<1>();
    else byRecon.template operator()<2>();
    return checkLaunch("face fluxes (fast)");
  });
}

int launchSourcesFast(const grim_params& p, const StepArgs& a, int recon, const Box& b, const double* prim,
                      const double* primOld, const double* geomC, const double* gamma40, const double* uT,
                      double* sExp, double* sImp, double* consOld, hipStream_t s) {
  GRIM_REQUIRE(planeOffsetsFit(a.D.n), "fast explicit stage: planes must hold fewer than 2^29 zones");
  const unsigned nb = blocks(b.count(), kBlock);
  return dispatchLayout(p, [&]<class L>() -> int {
    switch (recon) {
      case GRIM_RECON_WENO5:
        sourcesFastKernel<L, GRIM_RECON_WENO5><<<nb, kBlock, 0, s>>>(a, b, prim, primOld, geomC, gamma40, uT, sExp,
                                                                     sImp, consOld);
        break;
      case GRIM_RECON_PPM:
        sourcesFastKernel<L, GRIM_RECON_PPM><<<nb, kBlock, 0, s>>>(a, b, prim, primOld, geomC, gamma40, uT, sExp,
                                                                   sImp, consOld);
        break;
      default:
        sourcesFastKernel<L, GRIM_RECON_MINMOD><<<nb, kBlock, 0, s>>>(a, b, prim, primOld, geomC, gamma40, uT,
                                                                      sExp, sImp, consOld);
    }
    return checkLaunch("sources (fast)");
  });
}

void launchGamma40(int64_t n, const double* gamma64, double* gamma40, hipStream_t s) {
  gamma40Kernel<<<blocks(n, kBlock), kBlock, 0, s>>>(n, gamma64, gamma40);
}

}  // namespace grim
