// Device state of one CG solve, shared by the CG kernels (cg.hip) and the
// operator kernels that form the search direction themselves.
#pragma once
#include <hip/hip_runtime.h>

#include "reduce.hpp"

namespace ngsamd {

struct CGScalars {
  double wdn[2];     // <w,d> of the current iteration, by iteration parity
  double alpha, beta;
  double final_res;  // stopping threshold
  double tol, atol;  // tol < 0: not given; atol < 0: not given
  int it;            // CheckResidual calls so far
  int done;          // 0 running, 1 converged / maxiter, 2 breakdown
  int maxiter;
  int pad;
};

constexpr int kCgBlock = 256;

// The steps of one entry, spelled out so that every kernel that takes them
// rounds alike: the solvers with and without the direction in the product give
// the same iterates bit for bit.
__device__ __forceinline__ double CgFma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float CgFma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }

__device__ __forceinline__ void CheckResidual(CGScalars* S, double* residuals, double res) {
  S->it += 1;
  if (S->it <= S->maxiter) residuals[S->it - 1] = res;
  if (S->it == 1) {
    if (S->tol < 0) S->final_res = S->atol;
    else {
      S->final_res = res * S->tol;
      if (S->atol >= 0 && S->atol > S->final_res) S->final_res = S->atol;
    }
  }
  if (S->it >= S->maxiter || res <= S->final_res) S->done = 1;
}

// The direction step s = beta s + z as part of the operator kernel: the
// operator reads {s, z} pairs (one 16-byte load per entry), uses and stores the
// new s, so the iteration needs no kernel of its own for it.  The pairs are
// double-buffered by iteration parity: every workgroup reads the old ones
// (pair), the owner of a dof writes the new s (next).
struct CgDirection {
  const double* pair = nullptr;  // [n][2]
  double* next = nullptr;        // [n][2]
  CGScalars* S = nullptr;
  const double* pw = nullptr;    // partials of <w, d> of the update kernel
  int nw = 0;
  int P = 0;                     // iteration parity
  double* residuals = nullptr;
};

// beta = <w,d> / previous <w,d> (0 in the first iteration), the same bits in
// every workgroup; workgroup 0 also keeps <w,d> for the update kernel and does
// the stopping test (the others may go on: their results are not used once
// the loop has stopped).  stopped: the loop had stopped before this kernel, or
// workgroup 0 has seen it stop.  lds: kCgBlock / 64 + 2 doubles.
__device__ __forceinline__ double DirectionBeta(const CgDirection& D, bool& stopped, double* lds) {
  const double wdn = SumPartialsUnless<kCgBlock>(&D.S->done, stopped, D.pw, D.nw, lds);
  if (stopped) return 0.0;
  const double wd = D.S->wdn[D.P];
  const double beta = wd == 0.0 ? 0.0 : wdn / wd;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    D.S->wdn[D.P ^ 1] = wdn;
    D.S->beta = beta;
    CheckResidual(D.S, D.residuals, sqrt(fabs(wdn)));
  }
  return beta;
}

}  // namespace ngsamd
