// hoc_status.hpp - device side of an iteration's end: the convergence test on the summed norms and
// the publication of the solve's state in pinned host memory.  Shared by the finalize kernel
// (hoc_la.hip) and by the fine-level kernel that carries the test in a block of its own
// (hoc_poisson.hip).
#pragma once

#include "hoc_la.hpp"

namespace hoc {

// The solve's results, then, after a system-scope fence, the status word: the host follows
// the iterations and takes the results without a copy.
__device__ __forceinline__ void publish(MirrorState* __restrict__ mirror, int seq, bool near,
                                        const double* __restrict__ S, const int* __restrict__ F) {
  mirror->bb = S[S_BB];
  mirror->rr = S[S_RR];
  mirror->iter = F[F_ITER];
  mirror->zero = F[F_ZERO];
  __threadfence_system();
  __hip_atomic_store(&mirror->status, status_word(seq, near, F[F_ACTIVE] != 0), __ATOMIC_RELAXED,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}

// The number that a status goes out with: seq, or the next of the device's counter for seq < 0.
__device__ __forceinline__ int take_seq(int seq, int* __restrict__ F) {
  return seq >= 0 ? seq : (F[F_SEQ] = seq_add(F[F_SEQ], 1));
}

// Whether the next iteration is likely the last, if it reduces the residual as the one before did
// (within 2x of the tolerance: a needless wait costs the host's answer, 8 us; an iteration queued for
// nothing 25 us).
__device__ __forceinline__ bool likely_last(const double* __restrict__ S) {
  return S[S_PRED] <= 4. * S[S_TOL2] * S[S_BB];
}

// Start of a solve, from its first residual: a = r.r, b = ||r||^2 (unscaled), above: over the tolerance.
__device__ __forceinline__ void init_phase(double a, double b, bool above, double* __restrict__ S,
                                           int* __restrict__ F, int maxiter) {
  S[S_RR] = S[S_RRL] = S[S_PRED] = b;
  const double tiny = 2. * 2.220446049250313e-16;
  const bool zero = S[S_BB] < tiny * tiny;
  F[F_ZERO] = zero;
  F[F_ITER] = 0;
  F[F_HALF] = 0;
  F[F_BREAK] = 0;
  F[F_ACTIVE] = (!zero && above && maxiter > 0) ? 1 : 0;
  S[S_RZ] = 0.; S[S_RHO] = S[S_RHON] = a; S[S_ALPHA] = 1.; S[S_OMEGA] = 1.; S[S_BETA] = 0.;
}

// Whether a test has a solve to test.  After a breakdown that the update in front of it has seen (F_BREAK) it
// has none: x and r are those of the iteration before, and the norms are not this one's.
__device__ __forceinline__ bool solve_live(const int* __restrict__ F) {
  const int a = F[F_ACTIVE], b = F[F_BREAK];  // (both loads under way before either is looked at)
  return (a != 0) & (b == 0);
}

// b = ||r||^2 (unscaled) against the tolerance.  PH_UPD: end of a PCG iteration.  PH_BHALF: BiCGSTAB
// at its half step (x already holds alpha ph).  PH_BNEXT: end of a BiCGSTAB iteration, a = rh . r of
// the next; rho = 0 or not finite is a breakdown.
__device__ __forceinline__ void check_phase(int phase, double a, double b, double* __restrict__ S,
                                            int* __restrict__ F, int maxiter) {
  const double tol2bb = S[S_TOL2] * S[S_BB];
  S[S_RR] = b;
  if (phase == PH_BHALF) {
    if (b <= tol2bb) { F[F_ITER] += 1; F[F_ACTIVE] = 0; }
    return;
  }
  S[S_PRED] = b * (b / S[S_RRL]);
  S[S_RRL] = b;
  F[F_ITER] += 1;
  bool go = b > tol2bb && F[F_ITER] < maxiter && isfinite(b);
  if (phase == PH_BNEXT) go = go && S[S_OMEGA] != 0. && a != 0. && isfinite(a);
  F[F_ACTIVE] = go ? 1 : 0;
}

}  // namespace hoc
