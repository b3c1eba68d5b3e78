// Per-zone Newton kernels shared by the exact and the fast translation units.
//
// newton.hip includes this header and compiles with -ffp-contract=off (the
// reference FD path and the analytic FP64 path round every operation as
// written, bit-identical to the oracle); newton_fast.hip compiles the same
// templates with -ffp-contract=fast-honor-pragmas (fused multiply-adds) for the mixed
// precision path and the fast FD variant.  Each translation unit
// instantiates different modes, so no kernel is compiled twice.
//
// Design: one thread per zone, the whole Newton iteration in registers.  The
// zone's Jacobian is 5x5 (ideal MHD) to 7x7 (EMHD): far too small for MFMA
// tiles and small enough to stay in VGPRs, so LU with partial pivoting runs
// fully unrolled on register arrays with selects in place of row swaps.  All
// planes are zone-major structure of arrays: lane i of a wavefront touches
// zone base+i of every plane, so every load and store is a coalesced 512-byte
// wavefront access.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "analytic.hpp"
#include "fold.hpp"
#include "fused.hpp"
#include "grim_hip.h"
#include "zone_physics.hpp"

namespace grim {

constexpr int kDefaultBlock = 256;
constexpr int kMaxGroup = 8;  // largest grim_newton_opts.phase2_group taken

// dt' of the batch: from device memory when the caller computed it there.
__device__ __forceinline__ double batchDt(const grim_zone_batch& b) {
  return b.dt_prime_device ? *b.dt_prime_device : b.dt_prime;
}

// Jacobian / precision modes of the per-zone Newton kernel.
//  MODE_FD:          grim's residual and FD Jacobian, FP64 LU (reference path)
//  MODE_ANALYTIC64:  grim's residual, analytic Jacobian and LU in FP64
//  MODE_MIXED:       fused FP64 residual; the analytic Newton step by
//                    elimination (newtonStep, fused.hpp), in FP64
//  MODE_FD_FAST:     grim's FD Jacobian rule on the reciprocal-form FP64
//                    residual, one reciprocal per FD column, FP64 LU (the
//                    fastest FD-FP64 variant, for a like-for-like comparison)
enum { MODE_FD = 0, MODE_ANALYTIC64 = 1, MODE_MIXED = 2, MODE_FD_FAST = 3 };

template <int MODE>
struct ModeTraits {
  static constexpr bool fused = (MODE == MODE_MIXED || MODE == MODE_FD_FAST);
};

// The EMHD mixed solve keeps each zone's metric (16 doubles) and EMHD
// weights (12) in LDS slots instead of VGPRs: held in registers across the
// Newton loop they pushed it past 256 VGPRs into scratch (224 bytes per
// lane).  Slots are 17 and 13 doubles apart, so that the 64 lanes of a b64
// read cover every bank.  Every residual evaluation and Jacobian assembly
// starts behind a compiler fence, so the slots are read where they are used
// instead of being hoisted back into registers for the whole loop.
template <class L, int MODE>
constexpr bool kLdsState = L::EMHD && MODE == MODE_MIXED;
constexpr int kGeomSlot = 17, kWeightSlot = 13;
constexpr size_t kLdsStateBytes = (size_t)(kGeomSlot + kWeightSlot) * sizeof(double);  // per lane

template <class L, int MODE>
__device__ __forceinline__ void slotFence() {
  if constexpr (kLdsState<L, MODE>) asm volatile("" ::: "memory");
}

template <class L, int MODE>
__device__ __forceinline__ void evalResidual(const double* P, const ZoneGeom& G,
                                             const ZoneConst<L>& c, const DevParams& prm,
                                             double dt, const ZoneScale& zs, const EmhdWeights& ew,
                                             double* R, FusedPrimal& f) {
  slotFence<L, MODE>();
  if constexpr (ModeTraits<MODE>::fused)
    residualFused<L>(P, G, c, prm, zs, ew, R, f);
  else
    residual<L>(P, G, c, prm, dt, R);
}

// grim's forward-difference Jacobian (solve.cpp:82-109): A[i][j] = dR_i/dP_j
// with P_j perturbed by eps*P_j, or by eps when |P_j| < eps/2.
template <class L>
__device__ __forceinline__ void fdJacobian(const double* P, const double* R, const ZoneGeom& G,
                                           const ZoneConst<L>& c, const DevParams& prm,
                                           double dt, double (&A)[L::NF][L::NF]) {
  double Pp[L::DOF];
#pragma unroll
  for (int v = 0; v < L::DOF; v++) Pp[v] = P[v];
#pragma unroll
  for (int row = 0; row < L::NF; row++) {
    const double eps = prm.jacEps;
    const bool small = fabs(P[row]) < .5 * eps;
    Pp[row] = small ? P[row] + eps : P[row] + eps * P[row];
    double Rp[L::NF];
    residual<L>(Pp, G, c, prm, dt, Rp);
    const double dP = Pp[row] - P[row];
#pragma unroll
    for (int col = 0; col < L::NF; col++) A[col][row] = (Rp[col] - R[col]) / dP;
    Pp[row] = P[row];
  }
}

// grim's FD rule with the residual of MODE and one reciprocal per column.
template <class L, int MODE>
__device__ __forceinline__ void fdJacobianFast(const double* P, const double* R, const ZoneGeom& G,
                                               const ZoneConst<L>& c, const DevParams& prm,
                                               double dt, const ZoneScale& zs, const EmhdWeights& ew,
                                               double (&A)[L::NF][L::NF]);

// Small batches: grim's FD solve with one zone per kWide lanes of a
// wavefront.  Lane r + 1 of a zone's group evaluates the residual with P_r
// perturbed (grim's rule), so the NF columns of the FD Jacobian come from
// one residual evaluation's latency instead of NF; every other step runs on
// all lanes of the group with identical operands.  The result is the
// one-lane solve's bit for bit.
constexpr int kWide = 8;
constexpr int64_t kWideMaxZones = 16384;  // below this a one-lane grid leaves most CUs idle

template <class L>
__device__ __forceinline__ void fdJacobianWide(const double* P, const double* R, const ZoneGeom& G,
                                               const ZoneConst<L>& c, const DevParams& prm,
                                               double dt, double (&A)[L::NF][L::NF]) {
  static_assert(L::NF < kWide, "one lane per FD column");
  const int lane = threadIdx.x & 63;
  const int sub = lane % kWide;
  const int first = lane - sub;
  // lanes 1..NF take columns 0..NF-1; the others repeat column 0 (unused)
  const int row = (sub >= 1 && sub <= L::NF) ? sub - 1 : 0;
  const double eps = prm.jacEps;
  double Pp[L::DOF];
#pragma unroll
  for (int v = 0; v < L::DOF; v++) Pp[v] = P[v];
  double dP = 0.;
#pragma unroll
  for (int v = 0; v < L::NF; v++) {
    const bool small = fabs(P[v]) < .5 * eps;
    const double pv = small ? P[v] + eps : P[v] + eps * P[v];
    Pp[v] = (v == row) ? pv : P[v];
    dP = (v == row) ? pv - P[v] : dP;
  }
  double Rp[L::NF];
  residual<L>(Pp, G, c, prm, dt, Rp);
  double colv[L::NF];
#pragma unroll
  for (int k = 0; k < L::NF; k++) colv[k] = (Rp[k] - R[k]) / dP;
#pragma unroll
  for (int r = 0; r < L::NF; r++)
#pragma unroll
    for (int k = 0; k < L::NF; k++) A[k][r] = __shfl(colv[k], first + 1 + r, 64);
}

// One Newton update after the convergence test (solve.cpp:80-198): Jacobian,
// LU solve of J d = -R, quadratic backtracking line search, P += lambda d.
// Returns true when the last evaluated trial was accepted; Rt (and f, the
// primal of the fused modes) then holds the residual at the new P
// (bit-identical to a fresh evaluation, since the new P is computed by the
// same expression as the trial).
template <class L, int MODE, bool WIDE = false>
__device__ __forceinline__ bool newtonUpdate(double* P, const double* R, double l2,
                                             const ZoneGeom& G, const ZoneConst<L>& c,
                                             const DevParams& prm, double dt, const ZoneScale& zs,
                                             const EmhdWeights& ew, FusedPrimal& f, double* Rt, int& evals) {
  double d[L::NF];
  if constexpr (MODE == MODE_FD) {
    double A[L::NF][L::NF];
    if constexpr (WIDE)
      fdJacobianWide<L>(P, R, G, c, prm, dt, A);
    else
      fdJacobian<L>(P, R, G, c, prm, dt, A);
    evals += L::NF;
#pragma unroll
    for (int v = 0; v < L::NF; v++) d[v] = -R[v];
    luSolve<double, L::NF>(A, d);
  } else if constexpr (MODE == MODE_FD_FAST) {
    double A[L::NF][L::NF];
    fdJacobianFast<L, MODE>(P, R, G, c, prm, dt, zs, ew, A);
    evals += L::NF;
#pragma unroll
    for (int v = 0; v < L::NF; v++) d[v] = -R[v];
    luSolve<double, L::NF>(A, d);
  } else if constexpr (MODE == MODE_ANALYTIC64) {
    double A[L::NF][L::NF];
    analyticJacobian<double, L>(P, G, prm, c.mask / dt, c, ew, dt, A);
#pragma unroll
    for (int v = 0; v < L::NF; v++) d[v] = -R[v];
    luSolve<double, L::NF>(A, d);
  } else {
    slotFence<L, MODE>();
    newtonStep<L>(P, R, G, c, prm, zs, ew, f, d);
  }

  const double f0 = 0.5 * l2;
  const double fPrime0 = -2. * f0;
  double lambda = 1.;
  double Pt[L::DOF];
#pragma unroll
  for (int v = 0; v < L::DOF; v++) Pt[v] = P[v];
  bool accepted = false;
  bool finiteTrial = true;
  for (int ls = 0; ls < prm.maxLS; ls++) {
#pragma unroll
    for (int v = 0; v < L::NF; v++) Pt[v] = P[v] + lambda * d[v];
    evalResidual<L, MODE>(Pt, G, c, prm, dt, zs, ew, Rt, f);
    evals += 1;
    const double f1 = 0.5 * sumSq<L::NF>(Rt);
    if constexpr (MODE == MODE_FD) {
      // grim's test: a non-finite trial compares false and is accepted
      const bool condition = f1 > f0 * (1. - 1e-4 * lambda) + prm.lsFloor;
      if (!condition) {
        accepted = true;
        break;
      }
    } else {
      // this build's solvers reject a non-finite trial and halve the step (a
      // near-singular zone can overshoot into states where the residual
      // overflows)
      finiteTrial = isfinite(f1);
      if (f1 <= f0 * (1. - 1e-4 * lambda) + prm.lsFloor) {
        accepted = true;
        break;
      }
      if (!finiteTrial) {
        lambda = 0.5 * lambda;
        continue;
      }
    }
    const double denom = f1 - f0 - fPrime0 * lambda;
    lambda = -fPrime0 * lambda * lambda / denom / 2.;
  }
  // grim applies the last step length even when no trial passed; after a
  // non-finite last trial this build's solvers keep the zone where it is
  if (MODE != MODE_FD && !accepted && !finiteTrial) return false;
#pragma unroll
  for (int v = 0; v < L::NF; v++) P[v] = P[v] + lambda * d[v];
  return accepted;
}

// Newton iterations of one zone, from the primitives P, for at most
// `limit` updates (solve.cpp:10-200 read per zone: the zone stops when its
// own sum R^2 <= atol).  Writes the primitives back; stats are stored, or
// added to the earlier phase's when `accumulate`.  Once `budget` updates are
// done, a wavefront left with fewer than `keep` unconverged zones stops too:
// returns true then, with the updates done in `done` (the same for every
// lane that returns true), and a later phase continues the zone -- every
// iteration is a function of P alone, so stopping and resuming changes no
// result.  WIDE: the zone's kWide lanes run it together; only the first
// writes.
template <class L, int MODE, bool WIDE>
__device__ __forceinline__ bool solveZoneCore(const DevParams& prm, const grim_zone_batch& b,
                                              const grim_newton_stats& st, int64_t z, int budget, int limit,
                                              int keep, bool accumulate, double dt, const ZoneGeom& G,
                                              const ZoneConst<L>& c, const ZoneScale& zs, const EmhdWeights& ew,
                                              double (&P)[L::DOF], int& done);

// FOLDED: the zone's right-hand side, field rows and residual mask come from
// the caller's registers (foldRhs, foldB, foldMask: the stage fold computed
// in the same kernel) instead of the batch's planes.
template <class L, int MODE, bool WIDE = false, bool FOLDED = false>
__device__ __forceinline__ bool solveZone(const DevParams& prm, const grim_zone_batch& b,
                                          const grim_newton_stats& st, int64_t z, int budget, int limit,
                                          int keep, bool accumulate, int& done, const double* foldRhs = nullptr,
                                          const double* foldB = nullptr, double foldMask = 0.) {
  const int64_t n = b.n;
  const bool lead = !WIDE || (threadIdx.x % kWide) == 0;
  // the starting fluid rows: the caller's guess planes on a first pass,
  // else prim (a later phase resumes from what the earlier one wrote)
  const double* start = (b.guess && !accumulate) ? b.guess : b.prim;
  const double maskZ = FOLDED ? foldMask : (b.residual_mask ? b.residual_mask[z] : 1.);
  if ((FOLDED || b.residual_mask) && maskZ == 0.) {
    // outside the residual mask (ghost zones of a grid) R = 0: the zone
    // takes its floors and stops at the first test, as in the full path
    if (!lead) return false;
    if (start != b.prim)
#pragma unroll
      for (int v = U1; v < L::NF; v++) b.prim[v * n + z] = start[v * n + z];
    b.prim[RHO * n + z] = smax(start[RHO * n + z], prm.rhoFloor);
    b.prim[UU * n + z] = smax(start[UU * n + z], prm.uFloor);
    if (st.iterations) st.iterations[z] = accumulate ? st.iterations[z] : 0;
    if (st.residual_evals) st.residual_evals[z] = (accumulate ? st.residual_evals[z] : 0) + 1;
    if (st.final_l2) st.final_l2[z] = 0.;
    return false;
  }
  const double dt = batchDt(b);
  ZoneGeom G;
  loadBatchGeom(b, z, G);
  double P[L::DOF];
  auto loadStart = [&] {
#pragma unroll
    for (int v = 0; v < L::DOF; v++)
      P[v] = v < L::NF ? start[v * n + z] : (FOLDED ? foldB[v - L::NF] : b.prim[v * n + z]);
  };
  ZoneConst<L> c;
  ZoneScale zs;
  EmhdWeights ew;
  if constexpr (!ModeTraits<MODE>::fused) loadZoneConst<L, !FOLDED>(b, prm, G, z, c);
  if constexpr (ModeTraits<MODE>::fused || FOLDED) {
#pragma unroll
    for (int v = 0; v < L::NF; v++) c.rhs[v] = FOLDED ? foldRhs[v] : b.rhs[v * n + z];
    c.mask = maskZ;
  }
  if constexpr (ModeTraits<MODE>::fused) {
    EmhdPlanes<L> planes;
    if constexpr (L::EMHD) {
      // every load of the zone is in flight before the constants of the first
      // are formed
      loadEmhdPlanes<L>(b, z, planes);
      loadStart();
      __builtin_amdgcn_sched_barrier(0);
    }
    zoneScale(G, maskZ, dt, zs);
    if constexpr (L::EMHD) fusedEmhdConstants<L>(b, prm, G, planes, zs.invDt, c, ew);
  } else if constexpr (MODE == MODE_ANALYTIC64 && L::EMHD) {
    emhdWeights<L>(G, c, prm, dt, ew);
  }
  if constexpr (!(ModeTraits<MODE>::fused && L::EMHD)) loadStart();
  if constexpr (kLdsState<L, MODE>) {
    static_assert(sizeof(ZoneGeom) <= kGeomSlot * sizeof(double) &&
                  sizeof(EmhdWeights) <= kWeightSlot * sizeof(double), "LDS slot sizes");
    // the launch gives kLdsStateBytes of dynamic LDS per lane
    extern __shared__ double zoneSlots[];
    ZoneGeom* gs = reinterpret_cast<ZoneGeom*>(zoneSlots + (size_t)kGeomSlot * threadIdx.x);
    EmhdWeights* ws =
        reinterpret_cast<EmhdWeights*>(zoneSlots + (size_t)kGeomSlot * blockDim.x + (size_t)kWeightSlot * threadIdx.x);
    *gs = G;
    *ws = ew;
    return solveZoneCore<L, MODE, WIDE>(prm, b, st, z, budget, limit, keep, accumulate, dt, *gs, c, zs, *ws, P,
                                        done);
  } else {
    return solveZoneCore<L, MODE, WIDE>(prm, b, st, z, budget, limit, keep, accumulate, dt, G, c, zs, ew, P, done);
  }
}

template <class L, int MODE, bool WIDE>
__device__ __forceinline__ bool solveZoneCore(const DevParams& prm, const grim_zone_batch& b,
                                              const grim_newton_stats& st, int64_t z, int budget, int limit,
                                              int keep, bool accumulate, double dt, const ZoneGeom& G,
                                              const ZoneConst<L>& c, const ZoneScale& zs, const EmhdWeights& ew,
                                              double (&P)[L::DOF], int& done) {
  const int64_t n = b.n;
  const bool lead = !WIDE || (threadIdx.x % kWide) == 0;

  double R[L::NF];
  FusedPrimal f;
  bool haveR = false;
  bool converged = false, handOver = false;
  int iters = 0, evals = 0;
  double l2 = 0.;
  while (iters < limit) {
    // floors at the top of every iteration (solve.cpp:17-18)
    const double p0 = smax(P[RHO], prm.rhoFloor);
    const double p1 = smax(P[UU], prm.uFloor);
    if (!(p0 == P[RHO] && p1 == P[UU])) haveR = false;
    P[RHO] = p0;
    P[UU] = p1;
    if (!haveR) {
      evalResidual<L, MODE>(P, G, c, prm, dt, zs, ew, R, f);
      evals++;
    }
    l2 = sumSq<L::NF>(R);
    if (!(l2 > prm.atol)) {
      converged = true;
      break;
    }
    if (iters >= budget && __popcll(__ballot(1)) < keep) {
      handOver = true;
      break;
    }
    double Rt[L::NF];
    haveR = newtonUpdate<L, MODE, WIDE>(P, R, l2, G, c, prm, dt, zs, ew, f, Rt, evals);
    iters++;
    if (haveR) {
#pragma unroll
      for (int v = 0; v < L::NF; v++) R[v] = Rt[v];
    }
  }
  if (!converged && !handOver) {
    // out of updates: the statistics take the residual where the zone ended
    if (!haveR) evalResidual<L, MODE>(P, G, c, prm, dt, zs, ew, R, f);
    l2 = sumSq<L::NF>(R);
  }
  done = iters;
  if (!lead) return handOver;
#pragma unroll
  for (int v = 0; v < L::NF; v++) b.prim[v * n + z] = P[v];
  if (st.iterations) st.iterations[z] = (accumulate ? st.iterations[z] : 0) + iters;
  if (st.residual_evals) st.residual_evals[z] = (accumulate ? st.residual_evals[z] : 0) + evals;
  if (st.final_l2) st.final_l2[z] = l2;
  return handOver;
}

// Per-zone semantics, one pass: each thread iterates its own zone until
// sum R^2 <= atol or maxNonLinearIter updates.
//
// The EMHD solves need more than 256 registers per lane; asking for two
// wavefronts per SIMD (instead of one with AGPR spills) measured 8-10 %
// faster on the 3D torus, for the one-pass and the phase-1 kernel alike.
template <class L, int MODE>
__global__ __launch_bounds__(kDefaultBlock) __attribute__((amdgpu_waves_per_eu(2))) void newtonPerZone(
    DevParams prm, grim_zone_batch b, grim_newton_stats st) {
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (z >= b.n) return;
  int done;
  solveZone<L, MODE>(prm, b, st, z, prm.maxIter, prm.maxIter, 0, false, done);
}

// One-pass per-zone solve with the stragglers gathered inside the workgroup:
// every zone first gets budget1 updates; the zones still unconverged are then
// packed, by index, onto the workgroup's first lanes, which continue them for
// the remaining updates.  A zone's iterations are a function of its own
// primitives, so the results are the one-pass kernel's bit for bit, but the
// wavefronts left without a straggler end instead of idling through the last
// updates of a few lanes (about a quarter of the zones of a Kerr-Schild batch
// need a third update).  The zones the continuing lanes take are the
// workgroup's own, so their inputs come back from the caches.  It pays where
// updates are costly and a tail of zones needs many (grim's FD solve of the
// EMHD batch: 20.7 -> 15.0 ms); where the extra updates are few and cheap
// the two barriers and the restart cost more than they save (the mixed
// solve; the FD solve on the torus, 4.55 -> 5.05 ms per stage), so it is an
// option (grim_newton_opts.compaction = 2) the autotuner weighs.
template <class L, int MODE>
__global__ __launch_bounds__(kDefaultBlock) __attribute__((amdgpu_waves_per_eu(2))) void newtonPerZoneSplit(
    DevParams prm, grim_zone_batch b, grim_newton_stats st, int budget1) {
  __shared__ int list[kDefaultBlock];
  __shared__ int waveCount[kDefaultBlock / 64];
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool more = false;
  int done;
  if (z < b.n) more = solveZone<L, MODE>(prm, b, st, z, budget1, prm.maxIter, 65, false, done);
  const unsigned long long ballot = __ballot(more);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) waveCount[wave] = __popcll(ballot);
  __syncthreads();
  int base = 0, total = 0;
  for (int w = 0; w < (int)(blockDim.x >> 6); w++) {
    base += w < wave ? waveCount[w] : 0;
    total += waveCount[w];
  }
  if (more) list[base + __popcll(ballot & ((1ull << lane) - 1ull))] = (int)z;
  __syncthreads();
  if ((int)threadIdx.x < total)
    solveZone<L, MODE>(prm, b, st, (int64_t)list[threadIdx.x], prm.maxIter, prm.maxIter - budget1, 0, true, done);
}

// The one-pass FD solve of a small batch, kWide lanes per zone (every lane
// of a group shares z, so groups leave together).
template <class L>
__global__ __launch_bounds__(kDefaultBlock) void newtonPerZoneWide(DevParams prm, grim_zone_batch b,
                                                                  grim_newton_stats st) {
  const int64_t z = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / kWide;
  if (z >= b.n) return;
  int done;
  solveZone<L, MODE_FD, true>(prm, b, st, z, prm.maxIter, prm.maxIter, 0, false, done);
}

// The compacting solve.  Phase 1 gives every zone `budget1` updates, and goes
// on while a wavefront holds at least kKeepLanes unconverged zones; what is
// left it hands over as one 64-bit mask of lanes and one update count per
// wavefront.  Phase 2's wavefronts gather those zones, 64 at a time.
//
// Handing a zone over costs its planes again, 64-byte sectors of which it
// uses one entry (about 45 planes of an EMHD zone: 2.9 KB, the share of
// 1,300 cycles of a SIMD at the memory's rate), so it pays only where the
// update a wavefront would repeat for the zone's sake is dearer: about 2,800
// cycles for the fused step (three lanes), 10,000 for the dense analytic one
// and 20,000 and more for finite differences.  With every straggler handed
// over after two updates, a fifth of the 700,001-zone EMHD batch, phase 2
// took 75 us and the list 15 us beside phase 1's 83; now 100 and 5 us.
template <int MODE>
constexpr int kKeepLanes = MODE == MODE_MIXED ? 3 : (MODE == MODE_ANALYTIC64 ? 6 : 12);

// Lane 0 of a wavefront holding at least one zone stores what it hands over;
// wavefronts wholly past the end of the batch own no entry.
__device__ __forceinline__ void storeHandOver(bool more, int done, int64_t z, int64_t n,
                                              unsigned long long* __restrict__ masks, int* __restrict__ updates) {
  const unsigned long long ballot = __ballot(more);
  const int first = ballot ? __ffsll((long long)ballot) - 1 : 0;
  const int count = __shfl(done, first, 64);
  if ((threadIdx.x & 63) == 0 && z < n) {
    masks[z >> 6] = ballot;
    updates[z >> 6] = count;
  }
}

template <class L, int MODE>
__global__ __launch_bounds__(kDefaultBlock) __attribute__((amdgpu_waves_per_eu(2))) void newtonPhase1(
    DevParams prm, grim_zone_batch b, grim_newton_stats st, int budget1, unsigned long long* __restrict__ masks,
    int* __restrict__ updates) {
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool more = false;
  int done = 0;
  if (z < b.n) more = solveZone<L, MODE>(prm, b, st, z, budget1, prm.maxIter, kKeepLanes<MODE>, false, done);
  storeHandOver(more, done, z, b.n, masks, updates);
}

// The stage fold in front of a zone's Newton iterations: a bulk zone forms
// its right-hand side, its new field rows and its residual scale from the
// face fluxes, EMFs, consOld and sources (foldZone, the fold kernel's
// arithmetic bit for bit), writes the field rows and the mask plane, and
// keeps the right-hand side in registers.  The fold's memory traffic overlaps
// the solves' arithmetic, and no fold kernel and no copy of the field rows
// precede the solve.  `lead`: this lane writes for its zone.
template <class L, int DIM>
__device__ __forceinline__ bool foldForSolve(const grim_zone_batch& b, const FoldArgs& f, int64_t z, bool lead,
                                             double (&rhs)[L::NF], double (&B)[3], double& mask) {
  const int64_t n = b.n;
  int i, j, k;
  zoneIndex(f.D, z, i, j, k);
  const bool bulk = i >= f.bulk.lo[0] && i < f.bulk.hi[0] && j >= f.bulk.lo[1] && j < f.bulk.hi[1] &&
                    k >= f.bulk.lo[2] && k < f.bulk.hi[2];
  mask = 0.;
#pragma unroll
  for (int v = 0; v < L::NF; v++) rhs[v] = 0.;
  B[0] = B[1] = B[2] = 0.;
  if (bulk) {
    double rmax;
    foldZone<L, DIM, true>(f.D, f.dX, f.F, f.emf, f.geomC, f.consOld, f.sExp, f.sImp, batchDt(b), z, i, j,
                     f.fluxFilter, rhs, B, rmax);
    mask = f.scaling ? 1. / rmax : f.mask[z];
    if (lead) {
#pragma unroll
      for (int c = 0; c < 3; c++) b.prim[(L::NF + c) * n + z] = B[c];
      if (f.scaling) f.mask[z] = mask;
    }
  } else if (lead) {
#pragma unroll
    for (int c = 0; c < 3; c++) b.prim[(L::NF + c) * n + z] = f.fieldIn[c * n + z];
  }
  return bulk;
}

// Phase 1 of a grid stage's compacting solve with the stage fold; only the
// zones left unconverged store their right-hand side, for phase 2.
template <class L, int MODE, int DIM>
__global__ __launch_bounds__(kDefaultBlock) __attribute__((amdgpu_waves_per_eu(2))) void newtonPhase1Fold(
    DevParams prm, grim_zone_batch b, grim_newton_stats st, int budget1, unsigned long long* __restrict__ masks,
    int* __restrict__ updates, FoldArgs f) {
  const int64_t z = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  bool more = false;
  int done = 0;
  if (z < b.n) {
    double rhs[L::NF], B[3], mask;
    foldForSolve<L, DIM>(b, f, z, true, rhs, B, mask);
    more = solveZone<L, MODE, false, true>(prm, b, st, z, budget1, prm.maxIter, kKeepLanes<MODE>, false, done, rhs, B,
                                           mask);
    if (more)
#pragma unroll
      for (int v = 0; v < L::NF; v++) f.rhs[v * b.n + z] = rhs[v];
  }
  storeHandOver(more, done, z, b.n, masks, updates);
}

// A grid stage's one-pass solve with the stage fold (WIDE: kWide lanes per
// zone); the right-hand side of every bulk zone is stored, as the fold kernel
// leaves it.
template <class L, int MODE, int DIM, bool WIDE>
__global__ __launch_bounds__(kDefaultBlock) __attribute__((amdgpu_waves_per_eu(WIDE ? 1 : 2))) void newtonPerZoneFold(
    DevParams prm, grim_zone_batch b, grim_newton_stats st, FoldArgs f) {
  const int64_t z = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / (WIDE ? kWide : 1);
  if (z >= b.n) return;
  const bool lead = !WIDE || (threadIdx.x % kWide) == 0;
  double rhs[L::NF], B[3], mask;
  if (foldForSolve<L, DIM>(b, f, z, lead, rhs, B, mask) && lead)
#pragma unroll
    for (int v = 0; v < L::NF; v++) f.rhs[v * b.n + z] = rhs[v];
  int done;
  solveZone<L, MODE, WIDE, true>(prm, b, st, z, prm.maxIter, prm.maxIter, 0, false, done, rhs, B, mask);
}

// Compacting solve, phase 2.  Wavefront w of W takes the hand-over masks w,
// w + W, w + 2W, ... (stragglers cluster in space, so neighbouring masks go
// to different wavefronts), gathers their zones in a small list in LDS and
// solves them 64 at a time; what is left at the end runs on fewer lanes.  It
// needs no list in memory, no prefix sums between the phases (three launches
// of 5 us) and no shared counter, and every wavefront ends after nMasks / W
// masks.
template <class L, int MODE>
__global__ __launch_bounds__(kDefaultBlock) void newtonPhase2(DevParams prm, grim_zone_batch b,
                                                              grim_newton_stats st, int64_t nMasks,
                                                              const unsigned long long* __restrict__ masks,
                                                              const int* __restrict__ updates) {
  __shared__ int zones[kDefaultBlock / 64][128], left[kDefaultBlock / 64][128];
  const int lane = threadIdx.x & 63;
  int* zone = zones[threadIdx.x >> 6];
  int* rest = left[threadIdx.x >> 6];
  const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
  const int64_t wave = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  auto ordered = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); };
  auto run = [&](int count) {
    ordered();
    int done;
    if (lane < count)
      solveZone<L, MODE>(prm, b, st, (int64_t)zone[lane], prm.maxIter, rest[lane], 0, true, done);
    ordered();
  };
  int held = 0;  // zones in the list, below 64 between masks
  for (int64_t base = 0; base < nMasks; base += waves * 64) {
    // 64 of the wavefront's masks, one per lane
    const int64_t m = base + lane * waves + wave;
    unsigned long long mine = m < nMasks ? masks[m] : 0ull;
    int mineRest = mine ? prm.maxIter - updates[m] : 0;
    for (unsigned long long todo = __ballot(mine != 0ull); todo; todo &= todo - 1ull) {
      const int src = __ffsll((long long)todo) - 1;
      const unsigned long long mask = __shfl(mine, src, 64);
      const int r = __shfl(mineRest, src, 64);
      if ((mask >> lane) & 1ull) {
        const int at = held + __popcll(mask & ((1ull << lane) - 1ull));
        zone[at] = (int)((base + src * waves + wave) * 64 + lane);
        rest[at] = r;
      }
      held += __popcll(mask);
      if (held >= 64) {
        run(64);
        held -= 64;
        if (lane < held) {
          zone[lane] = zone[64 + lane];
          rest[lane] = rest[64 + lane];
        }
        ordered();
      }
    }
  }
  run(held);
}

template <class L, int MODE>
__device__ __forceinline__ void fdJacobianFast(const double* P, const double* R, const ZoneGeom& G,
                                               const ZoneConst<L>& c, const DevParams& prm,
                                               double dt, const ZoneScale& zs, const EmhdWeights& ew,
                                               double (&A)[L::NF][L::NF]) {
  double Pp[L::DOF];
#pragma unroll
  for (int v = 0; v < L::DOF; v++) Pp[v] = P[v];
#pragma unroll
  for (int row = 0; row < L::NF; row++) {
    const double eps = prm.jacEps;
    const bool small = fabs(P[row]) < .5 * eps;
    Pp[row] = small ? P[row] + eps : P[row] + eps * P[row];
    double Rp[L::NF];
    FusedPrimal f;
    evalResidual<L, MODE>(Pp, G, c, prm, dt, zs, ew, Rp, f);
    const double inv = 1. / (Pp[row] - P[row]);
#pragma unroll
    for (int col = 0; col < L::NF; col++) A[col][row] = (Rp[col] - R[col]) * inv;
    Pp[row] = P[row];
  }
}

// Carve-up of the caller's (or the library's) compaction workspace: per
// phase-1 wavefront the zones it hands over and the updates they have had.
struct CompactionWorkspace {
  unsigned long long* masks;
  int* updates;
};

constexpr int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// Bytes of the workspace for n zones, and the carve-up of a buffer of that size.
constexpr int64_t compactionBytes(int64_t n) {
  const int64_t nMasks = (n + 63) / 64;
  return align256(nMasks * 8) + align256(nMasks * 4) + 256;
}

inline CompactionWorkspace carveCompaction(void* base, int64_t n) {
  const int64_t nMasks = (n + 63) / 64;
  return {(unsigned long long*)base, (int*)((char*)base + align256(nMasks * 8))};
}

// Launch configuration of the per-zone solve (chosen by the autotuner or the
// caller).
struct LaunchCfg {
  int block;                 // threads per workgroup: 64, 128 or 256
  bool compaction;           // two-phase compacting solve
  bool workgroupSplit;       // one pass, stragglers gathered inside each workgroup (newtonPerZoneSplit)
  int budget1;               // phase-1 update budget
  int persistentWaves;       // phase-2 grid, in wavefronts
  CompactionWorkspace ws;    // what phase 1 hands over
};

// Dynamic LDS of a per-zone solve workgroup of `block` lanes.
template <class L, int MODE>
constexpr size_t ldsBytes(int block) {
  return kLdsState<L, MODE> ? kLdsStateBytes * (size_t)block : 0;
}

// Enqueue the per-zone solve of mode MODE on stream s.
// fold: a grid stage's fold runs inside the solve (the caller has checked
// foldFusable).
template <class L, int MODE>
void launchSolve(const DevParams& prm, const grim_zone_batch& b, const grim_newton_stats& st,
                 const LaunchCfg& cfg, hipStream_t s, const FoldArgs* fold = nullptr) {
  const unsigned grid = (unsigned)((b.n + cfg.block - 1) / cfg.block);
  constexpr bool canFold = MODE == MODE_FD || MODE == MODE_MIXED;
  // f.operator()<DIM>() for the grid's dimension
  auto byDim = [&](auto&& f) {
    if (fold->D.dim == 1) f.template operator()<1>();
    else if (fold->D.dim == 2) f.template operator()<2>();
    else f.template operator()<3>();
  };
  if (!cfg.compaction || cfg.budget1 >= prm.maxIter) {
    if constexpr (canFold) {
      if (fold) {
        byDim([&]<int DIM>() {
          if constexpr (MODE == MODE_FD) {
            if (b.n <= kWideMaxZones) {
              const unsigned wideGrid = (unsigned)((b.n * kWide + kDefaultBlock - 1) / kDefaultBlock);
              newtonPerZoneFold<L, MODE, DIM, true><<<wideGrid, kDefaultBlock, 0, s>>>(prm, b, st, *fold);
              return;
            }
          }
          newtonPerZoneFold<L, MODE, DIM, false><<<grid, cfg.block, ldsBytes<L, MODE>(cfg.block), s>>>(prm, b, st,
                                                                                                      *fold);
        });
        return;
      }
    }
    if constexpr (MODE == MODE_FD) {
      if (b.n <= kWideMaxZones) {
        const unsigned wideGrid = (unsigned)((b.n * kWide + kDefaultBlock - 1) / kDefaultBlock);
        newtonPerZoneWide<L><<<wideGrid, kDefaultBlock, 0, s>>>(prm, b, st);
        return;
      }
    }
    if (cfg.workgroupSplit && cfg.budget1 < prm.maxIter)
      newtonPerZoneSplit<L, MODE><<<grid, cfg.block, ldsBytes<L, MODE>(cfg.block), s>>>(prm, b, st, cfg.budget1);
    else
      newtonPerZone<L, MODE><<<grid, cfg.block, ldsBytes<L, MODE>(cfg.block), s>>>(prm, b, st);
    return;
  }
  const CompactionWorkspace& w = cfg.ws;
  const size_t lds = ldsBytes<L, MODE>(cfg.block);
  if constexpr (MODE == MODE_MIXED) {
    if (fold)
      byDim([&]<int DIM>() {
        newtonPhase1Fold<L, MODE, DIM><<<grid, cfg.block, lds, s>>>(prm, b, st, cfg.budget1, w.masks, w.updates, *fold);
      });
    else
      newtonPhase1<L, MODE><<<grid, cfg.block, lds, s>>>(prm, b, st, cfg.budget1, w.masks, w.updates);
  } else {
    newtonPhase1<L, MODE><<<grid, cfg.block, lds, s>>>(prm, b, st, cfg.budget1, w.masks, w.updates);
  }
  const int64_t nMasks = (b.n + 63) / 64;
  const int64_t waves = std::min<int64_t>(cfg.persistentWaves, nMasks);
  const unsigned grid2 = (unsigned)((waves * 64 + cfg.block - 1) / cfg.block);
  newtonPhase2<L, MODE><<<grid2, cfg.block, lds, s>>>(prm, b, st, nMasks, w.masks, w.updates);
}

// Host launcher of the fast translation unit (newton_fast.hip).
int launchNewtonFast(int mode, const grim_params& p, const grim_zone_batch& b,
                     const grim_newton_stats& st, const LaunchCfg& cfg, hipStream_t s,
                     const FoldArgs* fold = nullptr);

}  // namespace grim
