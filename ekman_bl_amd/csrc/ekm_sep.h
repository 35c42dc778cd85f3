// ekm_sep.h -- the separable solver of the consistent projection on grids
// without cross terms (ekm_sep.hip).
#pragma once
#include <vector>

#include "ekm_host.h"
#include "ekm_internal.h"

// Finest operator and problem of a projection, on the host.
struct SepProblem {
  const HostMgLevel* fine;      // rows with the consistent cells and identity rows at specified points
  const unsigned char* spec;    // specified points of the finest level
  bool per;                     // periodic z ends
  int pin;                      // singular kx = 0 problem: the pinned point, else -1
  const double* kx2;            // kx^2 of the live modes
  int nmode;
};

// Per-solve device state and operands of a solve, owned by the TightPlan.
struct SepBuffers {
  const double* cf64;           // finest c1..c8, [8][n]
  const unsigned char* spec;
  const double* wnull;          // left null vector of the singular problem, or null
  double tol;
  int maxit;
  const double* rhs;            // RHS_TMP planes [nsolve][n]
  double* phi;                  // solution planes [nsolve][n]
  int* cycles;
  double* r;                    // scratch: residual planes, [nsolve][n] doubles
  float* t;                     // scratch: 2 * nsolve * n floats
};

// Builds the plan; sp.on stays 0 where the operator is not close enough to a
// separable one (the caller then iterates with the multigrid cycle).
int sep_plan_build(SepPlan& sp, const SepProblem& q, int nsolve_max);
void sep_plan_free(SepPlan& sp);
// Runs up to kSepIter residual iterations on every solve: phi, cycles and, in
// sp.rmax + sep_iters(maxit) * nsolve_max, each solve's last max|residual|.
// guess: as in tight_solve_ex.
int sep_solve(const SepPlan& sp, const SepBuffers& b, int nsolve, const double* guess, hipStream_t st);
constexpr int kSepIter = 5;
inline int sep_iters(int maxit) { return maxit < kSepIter ? maxit : kSepIter; }
