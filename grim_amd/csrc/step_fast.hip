// The fast explicit stage: the two heaviest kernels of grim's stage, the face
// fluxes (riemannSolver::solve with reconstruction, riemannsolver.cpp:
// 202-328) and the explicit sources (fluidElement::computeExplicitSources
// with computeEMHDGradients, physics.cpp:360-586), compiled with
// -ffp-contract=fast-honor-pragmas (fused multiply-adds).
//
// Same mathematics as the exact kernels of step.hip, reorganised for fewer
// instructions:
//  * WENO5 (weno5.cpp:111-257) forms both face values of a zone from one set
//    of smoothness indicators, each with one division: the nonlinear weights
//    c_k / beta_k^2 and their sum are scaled by beta_1^2 beta_2^2 beta_3^2,
//    which leaves products of the betas;
//  * T^mu_nu is A^mu u_nu + C^mu b_nu + delta^mu_nu E, of which only the rows
//    and components that enter a result are formed, with shared reciprocals
//    (1/u^0, 1/|b|, 1/(rho + Gamma u), 1/(2A) for the two speeds);
//  * the closure enters fluxes and sources through chi/tau and nu/tau, in
//    which tau cancels;
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
// with two threads per face) and by the 1.2 GB it moves (250 us at copy rate);
// a fourth wavefront per SIMD (blocks of 64) adds nothing.
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

// The zone of this thread when the planes of a box are dealt to the 8 XCDs in
// bands of X2 rows (workgroups go round the XCDs in turn): the X2 and X3
// neighbours of a zone and its geometry column, which every X3 plane reads
// again, then stay in one XCD's L2 (sourcesFastKernel on 192x192x128 EMHD
// zones: 500 us, 1.8 GB fetched from beyond the L2; 529 us with the workgroups
// in memory order, which fetched 2.8 GB).
__device__ __forceinline__ bool bandZone(const Box& box, int& i, int& j, int& k) {
  const unsigned ni = (unsigned)(box.hi[0] - box.lo[0]), nk = (unsigned)(box.hi[2] - box.lo[2]);
  const unsigned plane = ni * (unsigned)(box.hi[1] - box.lo[1]);
  const unsigned x = blockIdx.x & 7u, t = (blockIdx.x >> 3) * (unsigned)kBlock + threadIdx.x;
  const unsigned lo = plane / 8u * x + min(x, plane % 8u), size = plane / 8u + (x < plane % 8u ? 1u : 0u);
  if (size == 0 || t >= size * nk) return false;
  const unsigned r = lo + t % size;
  i = box.lo[0] + (int)(r % ni);
  j = box.lo[1] + (int)(r / ni);
  k = box.lo[2] + (int)(t / size);
  return true;
}

unsigned bandBlocks(const Box& b) {
  const int64_t plane = (int64_t)(b.hi[0] - b.lo[0]) * (b.hi[1] - b.lo[1]);
  return 8u * (unsigned)(((plane + 7) / 8 * (b.hi[2] - b.lo[2]) + kBlock - 1) / kBlock);
}

// computeExplicitSources (physics.cpp:360-586) for the bulk zones of box, the
// old implicit sources with the stage element's tau and, on the half stage,
// consOld, from the element in the form of faceElement.
//
// Nothing is held that is only contracted: each derivative d_nu u_mu and each
// connection entry goes at once into the three scalars the EMHD sources read
// (g^{mu nu}, b^mu b^nu and u^mu b^nu times u_{nu;mu}), and T^k_l is formed
// for one l at a time from A^k u_l + C^k b_l + delta^k_l E.  tau cancels from
// the sources of q and deltaP.
//
// 1,080 instructions instead of 1,670 and three wavefronts per SIMD instead of
// two: 670 to 500 us on 192x192x128 EMHD zones (550 when two stencil fields
// are loaded ahead instead of three directions, which spills).  Bound by the
// 2.4 GB it moves, 480 us at the rate of a large copy.
//
// sparseImp: only the q and deltaP rows of the old implicit sources are
// written (the others are zero from the start).
struct PerDir {
  double v[3];
};

template <class L, int RECON>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3))) void sourcesFastKernel(
    StepArgs a, PerDir inv12dX, Box box, const double* __restrict__ prim, const double* __restrict__ primOld,
    const double* __restrict__ geomC, const double* __restrict__ gamma40, const double* __restrict__ uT,
    double* __restrict__ sExp, double* __restrict__ sImp, double* __restrict__ consOld, int sparseImp) {
  int i, j, k;
  if (!bandZone(box, i, j, k)) return;
  const Dims& D = a.D;
  const int64_t n = D.n, ng = D.ng;
  const uint32_t zb = (uint32_t)flatIndex(D, i, j, k) * 8u, zg = (uint32_t)geomIndex(D, i, j) * 8u;
  const DevParams& prm = a.prm;
  double P[L::DOF];
#pragma unroll
  for (int v = 0; v < L::DOF; v++) P[v] = ldOff(prim + v * n, zb);
  ZoneGeom G;
#pragma unroll
  for (int q = 0; q < 10; q++) G.gcov[q] = ldOff(geomC + q * ng, zg);
#pragma unroll
  for (int q = 0; q < 4; q++) G.gcon0[q] = ldOff(geomC + (GEOM_GCON0 + q) * ng, zg);
  G.alpha = ldOff(geomC + GEOM_ALPHA * ng, zg);
  G.g = ldOff(geomC + GEOM_G * ng, zg);
  // The stencils of u_0..u_3 and T along each direction, three ahead of their
  // use.
  constexpr int STENCILS = L::EMHD ? (L::COND_ON ? 15 : 12) : 0, RING = 4;
  double y[RING][5];
  int sB[3];  // no neighbours along a missing dimension: the zone itself
#pragma unroll
  for (int d = 0; d < 3; d++) sB[d] = d < D.dim ? (int)D.s[d] * 8 : 0;
  auto loadStencil = [&](int e) {
    if (e >= STENCILS) return;
#pragma unroll
    for (int q = 0; q < 5; q++)
      if (q != 2 || RECON != GRIM_RECON_WENO5)
        y[e % RING][q] = ldOff(uT + e / 3 * n, zb + (uint32_t)((q - 2) * sB[e % 3]));
  };
  double gam[2][10];
  auto loadGamma = [&](int l) {
#pragma unroll
    for (int q = 0; q < 10; q++) gam[l & 1][q] = ldOff(gamma40 + (l * 10 + q) * ng, zg);
  };
#pragma unroll
  for (int e = 0; e < RING - 1; e++) loadStencil(e);

  const double rho = smax(P[RHO], prm.rhoFloor), u = smax(P[UU], prm.uFloor);
  const double *ut = P + U1, *B = P + L::B1;
  const double p = (prm.gam - 1.) * u, g = G.g;
  double uc[4], uCov[4], bc[4], bCov[4];
  lower3(G, ut, uCov + 1);
  lower3(G, B, bCov + 1);
  const double lor = fastSqrt(1. + dot3(ut, uCov + 1));
  const double invU0 = fastDiv(G.alpha, lor), ga = lor * G.alpha;
  uc[0] = fastDiv(lor, G.alpha);
  uCov[0] = G.cov(0, 1) * ut[0] + G.cov(0, 2) * ut[1] + G.cov(0, 3) * ut[2] - ga;
  const double b0 = dot3(B, uCov + 1);
  const double bsq = (dot3(B, bCov + 1) + b0 * b0) * invU0 * invU0 + prm.bSqrFloor;
  bc[0] = b0;
  bCov[0] = (G.cov(0, 1) * B[0] + G.cov(0, 2) * B[1] + G.cov(0, 3) * B[2] + b0 * uCov[0]) * invU0;
#pragma unroll
  for (int q = 1; q < 4; q++) {
    uc[q] = ut[q - 1] - ga * G.gcon0[q];
    bc[q] = (B[q - 1] + b0 * uc[q]) * invU0;
    bCov[q] = (bCov[q] + b0 * uCov[q]) * invU0;
  }
  const double w = rho + u + p + bsq;
  double A[4], C[4], E = p + 0.5 * bsq, T = 0., ib = 0.;
  FastClosure cl{1., 0., 0.};
  double qb = 0., third = 0., dPb = 0.;
  if constexpr (L::EMHD) {
    T = smax(p * fastRcp(rho), prm.tFloor);
    ib = fastRsqrt(bsq);
    const double r = ldOff(geomC + LOC_R * ng, zg);
    fastClosure<L>(rho, u, p, T, bsq, L::COND_ON ? P[L::Q] : 0., L::VISC_ON ? P[L::DP] : 0., prm, 1., 1., r, cl);
    const double cs2 = prm.gam * p * fastRcp(rho + prm.gam * u);
    if constexpr (L::COND_ON)
      qb = (prm.highOrderCond ? P[L::Q] * T * fastSqrt(rho * prm.condAlpha * cs2) : P[L::Q]) * ib;
    if constexpr (L::VISC_ON) {
      const double dP = prm.highOrderVisc ? P[L::DP] * fastSqrt(T * rho * prm.viscAlpha * cs2) : P[L::DP];
      third = dP * (1. / 3.);
      dPb = dP * ib * ib;
    }
    E = E + third;
  }
#pragma unroll
  for (int q = 0; q < 4; q++) {
    A[q] = w * uc[q] + qb * bc[q] + third * uc[q];
    C[q] = qb * uc[q] - bc[q] - dPb * bc[q];
  }
  if (consOld) {
    stOff(consOld, zb, g * (rho * uc[0]));
    stOff(consOld + UU * n, zb, g * (A[0] * uCov[0] + C[0] * bCov[0] + E + rho * uc[0]));
#pragma unroll
    for (int q = 1; q < 4; q++) stOff(consOld + (UU + q) * n, zb, g * (A[0] * uCov[q] + C[0] * bCov[q]));
    if constexpr (L::COND_ON) stOff(consOld + L::Q * n, zb, g * (uc[0] * P[L::Q]));
    if constexpr (L::VISC_ON) stOff(consOld + L::DP * n, zb, g * (uc[0] * P[L::DP]));
#pragma unroll
    for (int q = 0; q < 3; q++) stOff(consOld + (L::B1 + q) * n, zb, g * B[q]);
  }
  if constexpr (L::EMHD) {
    if (sImp) {
      const double gt = g * fastRcp(cl.tau);
#pragma unroll
      for (int v = 0; v < L::NF; v++) {
        const bool row = (L::VISC_ON && v == L::DP) || (L::COND_ON && v == L::Q);
        if (row)
          stOff(sImp + v * n, zb, gt * ldOff(primOld + v * n, zb));
        else if (!sparseImp)
          stOff(sImp + v * n, zb, 0.);
      }
    }
  }

  // g^{mu nu}, b^mu b^nu and u^mu b^nu times u_{nu;mu}; b^mu d_mu T
  double div = 0., bb = 0., ub = 0., bT = 0.;
  double gcon[10];  // g^{mu nu}, packed as sym4
  if constexpr (L::EMHD) {
#pragma unroll
    for (int q = 0; q < 4; q++) gcon[q] = G.gcon0[q];
#pragma unroll
    for (int q = 0; q < 6; q++) gcon[4 + q] = ldOff(geomC + (16 + q) * ng, zg);
#pragma unroll
    for (int e = 0; e < STENCILS; e++) {
      loadStencil(e + RING - 1);
      const int m = e / 3, d = e % 3;
      const double* f = y[e % RING];
      double s;
      if constexpr (RECON == GRIM_RECON_WENO5)  // central differences (weno5.cpp:52-65)
        s = ((f[0] - f[4]) + 8. * (f[3] - f[1])) * inv12dX.v[d];
      else
        s = slopeZone<RECON>(f, a.theta, a.dX[d]);
      if (d >= D.dim) s = 0.;
      if (m < 4) {
        div = div + gcon[sym4(d + 1, m & 3)] * s;
        bb = bb + bc[d + 1] * bc[m & 3] * s;
        ub = ub + uc[d + 1] * bc[m & 3] * s;
      } else {
        bT = bT + bc[d + 1] * s;
      }
      asm volatile("" : "+v"(div), "+v"(bb), "+v"(ub), "+v"(bT));
    }
  }
  double src[4] = {0., 0., 0., 0.};
  const bool curved = a.metric != GRIM_METRIC_MINKOWSKI;
  if (curved || L::EMHD) {
    loadGamma(0);
#pragma unroll
    for (int l = 0; l < 4; l++) {
      if (l < 3) loadGamma(l + 1);
      const double* ga4 = gam[l & 1];
      if (curved) {
        double t[4];
#pragma unroll
        for (int q = 0; q < 4; q++) t[q] = A[q] * uCov[l] + C[q] * bCov[l] + (q == l ? E : 0.);
#pragma unroll
        for (int nu = 0; nu < 4; nu++)
#pragma unroll
          for (int q = 0; q < 4; q++) src[nu] = src[nu] + t[q] * ga4[sym4(q, nu)];
      }
      if constexpr (L::EMHD) {
        double cd = 0., cb = 0., cu = 0.;
#pragma unroll
        for (int mu = 0; mu < 4; mu++) {
          double vb = 0.;  // Gamma^l_{mu nu} b^nu
#pragma unroll
          for (int nu = 0; nu < 4; nu++) {
            vb = vb + ga4[sym4(mu, nu)] * bc[nu];
            if (nu >= mu) cd = cd + (nu > mu ? 2. : 1.) * gcon[sym4(mu, nu)] * ga4[sym4(mu, nu)];
          }
          cb = cb + bc[mu] * vb;
          cu = cu + uc[mu] * vb;
        }
        div = div - cd * uCov[l];
        bb = bb - cb * uCov[l];
        ub = ub - cu * uCov[l];
      }
      asm volatile("" : "+v"(src[0]), "+v"(src[1]), "+v"(src[2]), "+v"(src[3]), "+v"(div), "+v"(bb), "+v"(ub));
    }
  }
  stOff(sExp, zb, 0.);
#pragma unroll
  for (int nu = 0; nu < 4; nu++) stOff(sExp + (UU + nu) * n, zb, curved ? -g * src[nu] : 0.);
  // q0 = -rho chi/|b| (b^mu d_mu T + T b^nu u^mu u_{nu;mu}) and deltaP0 =
  // rho nu (3/b^2 b^mu b^nu u_{nu;mu} - u^mu_{;mu}), over tau; the high-order
  // closure scales them by sqrt(tau/(rho chi))/T and sqrt(tau/(rho nu T))
  if constexpr (L::COND_ON) {
    const double rc = rho * cl.chiOverTau;
    double s = g * ib * (bT + T * ub);
    s = prm.highOrderCond == 1 ? s * fastSqrt(rc) * fastRcp(T) - 0.5 * g * div * P[L::Q] : s * rc;
    stOff(sExp + L::Q * n, zb, s);
  }
  if constexpr (L::VISC_ON) {
    const double rn = rho * cl.nuOverTau;
    double s = g * (div - 3. * ib * ib * bb);
    s = prm.highOrderVisc == 1 ? s * fastSqrt(fastDiv(rn, T)) - 0.5 * g * div * P[L::DP] : s * rn;
    stOff(sExp + L::DP * n, zb, s);
  }
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
                      double* sExp, double* sImp, double* consOld, bool sparseImp, hipStream_t s) {
  GRIM_REQUIRE(planeOffsetsFit(a.D.n), "fast explicit stage: planes must hold fewer than 2^29 zones");
  const unsigned nb = bandBlocks(b);
  PerDir c;
  for (int d = 0; d < 3; d++) c.v[d] = 1. / (12. * a.dX[d]);
  return dispatchLayout(p, [&]<class L>() -> int {
    switch (recon) {
      case GRIM_RECON_WENO5:
        sourcesFastKernel<L, GRIM_RECON_WENO5><<<nb, kBlock, 0, s>>>(a, c, b, prim, primOld, geomC, gamma40, uT, sExp,
                                                                     sImp, consOld, sparseImp);
        break;
      case GRIM_RECON_PPM:
        sourcesFastKernel<L, GRIM_RECON_PPM><<<nb, kBlock, 0, s>>>(a, c, b, prim, primOld, geomC, gamma40, uT, sExp,
                                                                   sImp, consOld, sparseImp);
        break;
      default:
        sourcesFastKernel<L, GRIM_RECON_MINMOD><<<nb, kBlock, 0, s>>>(a, c, b, prim, primOld, geomC, gamma40, uT,
                                                                      sExp, sImp, consOld, sparseImp);
    }
    return checkLaunch("sources (fast)");
  });
}

void launchGamma40(int64_t n, const double* gamma64, double* gamma40, hipStream_t s) {
  gamma40Kernel<<<blocks(n, kBlock), kBlock, 0, s>>>(n, gamma64, gamma40);
}

}  // namespace grim
