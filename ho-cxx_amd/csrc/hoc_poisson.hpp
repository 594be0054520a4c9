// hoc_poisson.hpp - launchers of the fine-level Poisson kernels (hoc_poisson.hip).
#pragma once

#include "hoc_kernels.hpp"
#include "hoc_la.hpp"

namespace hoc {

// What a fine-operator kernel does with As u (As = -W A, W = w_i w_j):
//   EPI_STORE     y = As u; partial sums of u.y
//   EPI_RESID     y = b - As u; partial sums of y.y and (y/W).(y/W)
//   EPI_SMOOTH    y = u + omega B (b - As u); optional partial sums of b.y
//   EPI_RESTRICT  ec[el][a] = sum_ij q1w(a,ij) (b - As u)_ij      (Pc^T residual, per element)
//   EPI_PLAIN     y = A u (the operator itself, unscaled)
//   EPI_DOTS      y = As u; partial sums of b.y and y.y
enum { EPI_STORE = 0, EPI_RESID = 1, EPI_SMOOTH = 2, EPI_RESTRICT = 3, EPI_PLAIN = 4, EPI_DOTS = 5 };
// The field u it is applied to:
//   IN_X     u = x
//   IN_PROL  u = x + Pc xc (bilinear from the corner vertices)
//   IN_PUPD  u = z + beta p, written to pn (PCG's direction update)
enum { IN_X = 0, IN_PROL = 1, IN_PUPD = 2 };
// The geometry the kernels are instantiated for: elements with constant orthogonal metrics,
// constant metrics, metrics per point.
enum { GEO_ORTHO = 0, GEO_AFFINE = 1, GEO_POINT = 2 };

constexpr int kFineThreads = 256;
// Elements per wavefront: K lanes each.  A block's four wavefronts hold a multiple of 4, so that its
// elements start on a 16-byte boundary in every field.
constexpr int fine_epw(int K) { return K == 2 ? 32 : K == 3 ? 20 : K == 4 ? 16 : K == 5 ? 12 : 10; }
// Up to this many partials every block of the next kernel sums them itself, which saves a launch
// (4.4 us in a chain of dependent kernels) for about 1 us; above, a finalize kernel does.
constexpr int kInlineParts = 1024;
inline int fine_blocks(int K, int N) {
  const int e = fine_epw(K) * (kFineThreads / 64);
  return (N + e - 1) / e;
}

// Static data of the fine level in precision R.
template <class R>
struct FineGeo {
  int N;
  const R* ac;           // [N][2] mean metrics (g22/J, g11/J) over the element: B's scales, and the
                         // metrics themselves where they are constant and orthogonal
  const R* fdm;          // [9] per pair of end kinds: eigenvalues [K], eigenvectors [K][K]
  const R* lane;         // [K][4] weight, point and interior eigenvalue of a lane
  const uint16_t* ftype; // [N] kinds of the west/east and south/north ends: 9-way codes tx + 16 ty
  const R* gel;          // [N][3]    Ga, Gb, Gc of affine elements
  const R* gface;        // [N][4][2] fa, fb of affine elements
  const R *Ga, *Gb, *Gc; // [N][K2]
  const R *fa, *fb;      // [N][4][K]
  const R* qn;           // [E][K][K] Neumann common values from value + inward derivative / g'
  const int32_t* nb;     // [N][4] neighbour or -1-edge
  const int32_t* nbf;    // [N] the four neighbours' faces, one per byte
  const int8_t* sw;      // [E] 0 Dirichlet / 1 Neumann
  const int32_t* ev;     // [N][4] corner vertices
  const int32_t* inst;   // [N] ensemble instance, or null
  const int* iact;       // [instances] live flags (null: all): blocks of one stopped instance return
};

// 1-D tables of the fine-level kernels (kernel argument).  The Gauss points are symmetric, so the
// line operators are applied to a line's even and odd parts, e_i = u_i + u_{K-1-i} (the middle value
// itself) and o_i = u_i - u_{K-1-i}: about half the products and half the constants, which then
// stay in scalar registers.
// Aligned to the scalar cache's lines, so that the arguments behind it keep their places in them.
template <class R>
struct alignas(64) FineTab {
  R lv[6], ld[6];  // l_m(-1), l_m'(-1) (the upper end by reflection)
  R lvE[3], lvO[3], ldE[3], ldO[3];      // the same on the even and odd parts
  R DDE[3][3], DDO[3][3];                // second derivative: [in][out] (V-cycle)
  R gdE[3], gdO[3], DgE[3], DgO[3];      // lower Radau correction's derivative, and its derivative
  R m0, m1;        // that correction's derivative extrapolated to -1 and +1
  R g0, ig0;       // -g'(-1), the interface coefficient, and its inverse
  R w[6], x[6];    // Gauss weights and points
  R SE[3][3], SO[3][3], lam[6];  // eigenpairs of an interior element's line operator, even ones first
  R D[6][6], gd[6];  // l_m'(xi_k), the correction's derivative (elements with tangential metrics)
  R DE[3][3], DO[3][3];  // derivative: the odd part of an even line's, and vice versa (behind what the
                         // V-cycle's kernels load: in front, 0.3 us more for each of them, FP32, 121 x 121, K = 3)
};

template <class R>
struct FineArgs {
  const R* x = nullptr;      // IN_X, IN_PROL: the field; IN_PUPD: p
  const void* z = nullptr;   // IN_PUPD: z (R, or float for the mixed-precision direction update)
  R* pn = nullptr;           // IN_PUPD: the new direction
  const R* xc = nullptr;     // IN_PROL: vertex values
  const R* b = nullptr;
  R* y = nullptr;
  double omega = 0.;
  double* scal = nullptr;  // IN_PUPD: beta = scal[scal_idx], scal_idx < 0: scal[inst[el]]
  int scal_idx = 0;
  // IN_PUPD, small meshes: r.z as np partials, summed by every block; block 0 leaves the new r.z and
  // beta in scal (S_RZN, S_BETA).  On a breakdown (r.z not positive) nothing else is written
  const double* rz = nullptr;
  int np = 0;
  double* part = nullptr;    // [fine_blocks] sums, then [fine_blocks] second sums
  double* elpart = nullptr;  // instead: the first sum's share of every element [N]
  const double* b64 = nullptr;  // EPI_SMOOTH in FP32: b in FP64 for the sums of b.y
  int* active = nullptr;     // the Krylov flags F (may be null)
  int* ran = nullptr;        // set to 1 when the launch worked, 0 when active made it return at once
  // EPI_SMOOTH of IN_X: a block more, which tests np pairs of partial norms that an earlier kernel
  // left (phase: check_phase, or PH_INIT) on the flags chk_F and publishes the state; the other blocks
  // do not wait for it.  chk_bb: chk_nbb partials of ||b||^2 for scal[S_BB] (PH_INIT; may be null)
  int* chk_F = nullptr;
  const double* chk_bb = nullptr;
  int chk_nbb = 0;
  const double* chk_part = nullptr;
  int chk_np = 0, chk_phase = 0, chk_maxit = 0, chk_seq = 0;
  MirrorState* chk_mirror = nullptr;  // null: tested, not published
};

hipError_t launch_fine(int K, int geo, int in, int epi, const FineTab<double>& T, const FineGeo<double>& G,
                       const FineArgs<double>& A, hipStream_t s);
hipError_t launch_fine(int K, int geo, int in, int epi, const FineTab<float>& T, const FineGeo<float>& G,
                       const FineArgs<float>& A, hipStream_t s);
// IN_PUPD + EPI_STORE with z in FP32
hipError_t launch_fine_pupd_f32z(int K, int geo, const FineTab<double>& T, const FineGeo<double>& G,
                                 const FineArgs<double>& A, hipStream_t s);

// First smoothing step from zero, z = omega B r, with a Krylov update in front of it (up):
//   PRE_NONE
//   PRE_XR      x += alpha p, r -= alpha q; alpha = scal[scal_idx], or scal[inst[el]] with scal_idx < 0,
//               where elements of alpha = 0 keep x and r; partial sums of r.r and (r/W).(r/W)
//   PRE_BICGP   p = r + beta (p - omega_k q), z = omega B p, with BiCGSTAB's beta and omega_k from scal
//   PRE_BICG0   the same before the first iteration: p = r, and rh = r
// FP32 V-cycle: r32 receives the residual that the cycle is for in FP32.
enum { PRE_NONE = 0, PRE_XR = 1, PRE_BICGP = 2, PRE_BICG0 = 3 };
template <class R>
struct PreArgs {
  double *r = nullptr, *x = nullptr;
  const double *p = nullptr, *q = nullptr;
  R* z = nullptr;
  R* r32 = nullptr;
  double omega = 0.;
  double* scal = nullptr;
  int scal_idx = 0;
  int up = PRE_NONE;
  double *pw = nullptr, *rh = nullptr;  // PRE_BICGP, PRE_BICG0: the direction, the shadow residual
  // small meshes: a dot product as np partials, summed by every block.  PRE_XR: the denominator of
  // alpha (numerator scal[num]); block 0 leaves alpha and the numerator (in scal[keep]) behind.  On a
  // breakdown (spd: also where either is not positive) no block writes x or r, and block 0 sets F_BREAK
  // for the test of the iteration.  PRE_BICGP: rh.r, from which
  // block 0 leaves beta and scal[S_RHON]; a breakdown is left to the test of the iteration.
  const double* pq = nullptr;
  int np = 0, num = 0, keep = 0;
  bool spd = true;
  double* part = nullptr;
  double* elpart = nullptr;  // instead: every element's share of (r/W).(r/W) [N]
  int* active = nullptr;     // the Krylov flags F (may be null)
  double iw[6] = {0., 0., 0., 0., 0., 0.};  // 1 / w_k
  const double* iwl = nullptr;              // the same on the device, for the lane's own
};
hipError_t launch_pre(int K, const FineTab<double>& T, const FineGeo<double>& G, const PreArgs<double>& A,
                      hipStream_t s);
hipError_t launch_pre(int K, const FineTab<float>& T, const FineGeo<float>& G, const PreArgs<float>& A, hipStream_t s);

// End of a BiCGSTAB iteration: x += omega sh, r -= omega t; partial sums of rh.r and (r/W).(r/W).
// omega = scal[S_OMEGA]; with ts set, from np pairs of partials of (t.s, t.t), summed by every block,
// and left in scal by block 0.
struct BicgArgs {
  double *x = nullptr, *r = nullptr;
  const double *sh = nullptr, *t = nullptr, *rh = nullptr;
  double* scal = nullptr;
  const double* ts = nullptr;
  int np = 0;
  double* part = nullptr;
  const int* active = nullptr;
  double iw[6] = {0., 0., 0., 0., 0., 0.};
  const double* iwl = nullptr;
};
hipError_t launch_bicg_x(int K, int N, const BicgArgs& A, hipStream_t s);

}  // namespace hoc
