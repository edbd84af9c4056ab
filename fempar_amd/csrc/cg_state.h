// cg_state.h -- scalar state of the CG solvers and the decisions taken on it
// (device code shared by cg.hip and batch.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "femhip_internal.h"

namespace femhip {
namespace {

struct CgState {
  double rz, rnrm_m, alpha, beta;
  double rhs_test, rhs_extra, est, pap, pp;
  double bnorm, r0norm, rnorm;
  double rtol, atol;
  double rmax, delta;          // reliable updates
  double ru_rz, ru_rmax, ru_rnorm, ru_beta;
  double rscale, ru_rscale;    // ||S r|| / ||r|| at the last update (scaled inner residual)
  int iter, done, converged, maxit, crit, ru, updates, ru_conv, ru_done, first;
  int set, pad;                // lattice FP32 passes: which of the two vector sets holds r, p, s
};

struct CgResult {
  double est, rhs_test, rnorm, bnorm;
  int iter, done, converged, updates;
  double prog;                 // latest quantity the stopping test compares with rhs_test ...
  int prog_it, pad;            // ... and its iteration (for the host's chunk planning)
};

__device__ __forceinline__ bool is_delta(int c) {
  return c == FEMHIP_DELTA_RHS || c == FEMHIP_DELTA_DELTA || c >= FEMHIP_DELTA_RHS_AND_RES_RES;
}
__device__ __forceinline__ bool is_delta_delta(int c) {
  return c == FEMHIP_DELTA_DELTA || c == FEMHIP_DELTA_DELTA_AND_RES_RES || c == FEMHIP_DELTA_DELTA_AND_RES_RHS;
}

// The next FP32 CG direction p' = beta p + z, rounded once (fused multiply-add).
__device__ __forceinline__ float dir_value(float beta, float p, float z) { return __builtin_fmaf(beta, p, z); }

// FP64 solution plus FP32 increment (scaled by sc when set): the solution a
// reliable update makes.
__device__ __forceinline__ double new_x(double x, float d, const double *sc, int64_t i) {
  return sc ? __builtin_fma(sc[i], (double)d, x) : x + (double)d;
}

// Stopping test (cg.f90:323-407) of iteration `it`, whose <r,z>, ||r||^2 are
// red[0], red[1] and whose alpha and ||p||^2 are in cur: its estimate and
// threshold; returns whether it converged.
__device__ __forceinline__ bool cg_test(const CgState &cur, int it, const double (&red)[2], double rnorm, double &est,
                                        double &rhs_test) {
  const int c = cur.crit;
  est = cur.est;
  rhs_test = cur.rhs_test;
  if (it == 1 && is_delta(c)) {
    est = cur.alpha * sqrt(cur.pp);
    if (is_delta_delta(c)) rhs_test = cur.rtol * est + cur.atol;
  }
  if (c == FEMHIP_RES_RES || c == FEMHIP_RES_RHS) est = rnorm;
  else if (is_delta(c)) {
    if (it != 1) est = cur.alpha * sqrt(cur.pp);
  } else est = cur.rnrm_m;
  bool conv = est <= rhs_test;
  if (c >= FEMHIP_DELTA_RHS_AND_RES_RES && conv) conv = rnorm <= cur.rhs_extra;
  return conv;
}

// The test after an iteration; `lead` (one thread of the launch) writes the
// next state, the history and the result blocks.  Returns done, beta for the
// next direction.
__device__ __forceinline__ bool cg_decide(const CgState &cur, const double (&red)[2], bool lead, CgState &next,
                                          double *hist, CgResult *R, CgResult *Rh, double &beta_out) {
  const int it = cur.iter + 1;
  const double rnorm = sqrt(red[1]);
  double est, rhs_test;
  const int conv = cg_test(cur, it, red, rnorm, est, rhs_test);
  const bool done = conv || it >= cur.maxit;
  double beta = 1.0 / cur.rz;
  beta = beta * red[0];
  if (lead) {
    CgState nx = cur;
    nx.first = 0;
    nx.iter = it;
    nx.est = est;
    nx.rhs_test = rhs_test;
    nx.rnorm = rnorm;
    nx.converged = conv;
    nx.done = done;
    nx.beta = beta;
    nx.rz = red[0];
    nx.rnrm_m = sqrt(red[0]);
    next = nx;
    if (hist) hist[it - 1] = est;
    R->iter = it;
    R->est = est;
    R->rhs_test = rhs_test;
    R->rnorm = rnorm;
    R->converged = conv;
    R->done = done;
    R->prog = est;
    R->prog_it = it;
    if (Rh) *Rh = *R;
  }
  beta_out = beta;
  return done;
}

// What a slot A does: the decision after the previous slot B, whose <r,r> (and
// after a fold the FP64 ||b - A x||^2) are red; `lead` writes the next state.
struct RfStep {
  int fold, upd_d, done;
  double beta;
};
__device__ __forceinline__ RfStep rf_decide(const CgState &cur, const double (&red)[2], bool lead, CgState &next,
                                            CgResult *R) {
  if (lead) {
    next = cur;
    next.first = 0;
  }
  int fold = 0, upd_d = 0, done = 0;
  double beta = 0.0;
  if (cur.first) {           // p = r, q = A r
  } else if (!cur.ru) {      // an iteration's r update has been made
    const int it = cur.iter + 1;
    const double rnorm = sqrt(red[0]);   // of the scaled FP32 residual
    // residual fell by delta since the last update, looks converged (threshold
    // carried into the scaled norm by the last update's ratio), or budget spent
    fold = rnorm < cur.delta * cur.rmax || rnorm <= cur.rhs_test * cur.rscale || it >= cur.maxit;
    if (!fold) {
      beta = 1.0 / cur.rz;
      beta = beta * red[0];
      upd_d = 1;
    }
    if (lead) {
      CgState &w = next;
      w.iter = it;
      w.rnorm = rnorm;
      w.ru = fold;
      if (!fold) {
        w.beta = beta;
        w.rz = red[0];
        w.rmax = fmax(cur.rmax, rnorm);
      }
      R->iter = it;
      R->prog = cur.rscale > 0.0 ? rnorm / cur.rscale : rnorm;   // estimate in the stopping test's norm
      R->prog_it = it;
    }
  } else {                   // slot B replaced r by the FP64 residual of the folded x
    const double rn64 = sqrt(red[1]);
    const int conv = rn64 <= cur.rhs_test;
    beta = 1.0 / cur.rz;
    beta = beta * red[0];
    done = conv || cur.iter >= cur.maxit;
    if (lead) {
      CgState &w = next;
      w.ru = 0;
      w.rz = red[0];
      w.beta = beta;
      w.rmax = sqrt(red[0]);
      w.rscale = rn64 > 0.0 ? sqrt(red[0]) / rn64 : cur.rscale;
      w.updates = cur.updates + 1;
      w.est = rn64;
      w.rnorm = rn64;
      w.converged = conv;
      w.done = done;
      R->iter = cur.iter;
      R->est = rn64;
      R->rnorm = rn64;
      R->converged = conv;
      R->done = done;
      R->updates = cur.updates + 1;
      R->prog = rn64;
      R->prog_it = cur.iter;
    }
  }
  return {fold, upd_d, done, beta};
}

}  // namespace
}  // namespace femhip
