// hoc_kernels.hpp - gfx950 kernels of the HO-CXX time-step hot path.
//
// Fields are element-major ([el][j][i], K*K values per element); the kernels' mapping is in
// hoc_rowlane.hpp.
// Face numbering ijp: 0 west (xi=-1), 1 east, 2 south (eta=-1), 3 north.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>

namespace hoc {

constexpr int kMaxKd = 8;

// 1-D FR tables, passed by value (kernel argument space).
struct Tab {
  double bb[kMaxKd][2];      // l_m(-1), l_m(+1)
  double bgb[kMaxKd][2];     // l_m'(-1), l_m'(+1)
  double D[kMaxKd][kMaxKd];  // D[m][k] = l_m'(xi_k)
  double rad[kMaxKd][2];     // g_L, g_R at xi_k
  double grad[kMaxKd][2];    // g_L', g_R' at xi_k
  double gp[2];              // g'(-1), g'(+1)
  double w[kMaxKd];          // Gauss weights
  double x[kMaxKd];          // Gauss points (bilinear coarse-space weights)
};

// Bilinear (Q1) weight of element corner a (0 SW, 1 SE, 2 NE, 3 NW of the element's
// reference square) at solution point (i along xi, j along eta).
__device__ __forceinline__ double q1w(const Tab& T, int a, int j, int i) {
  const double xi = T.x[i], et = T.x[j];
  const double sx = (a == 1 || a == 2) ? 1. + xi : 1. - xi;
  const double sy = (a >= 2) ? 1. + et : 1. - et;
  return 0.25 * sx * sy;
}

// Static per-mesh device arrays of the stage kernels.
struct Geo {
  int N, E;
  const double *jac, *xxi, *xeta, *yxi, *yeta;  // [N][K2]
  const double *Ga, *Gb, *Gc;                   // g22/J, g12/J, g11/J at sps
  const double *fa, *fb;                        // [N][4][K]  A/fjac, B/fjac
  const double *fA, *fjac, *fAn;                // [N][4][K]  raw face metrics
  const double* gel;                            // [N][3]     Ga, Gb, Gc of affine elements
  const double* gface;                          // [N][4][2]  fa, fb of affine elements
  const double* gjm;                            // [N][5]     xxi, xeta, yxi, yeta, jac of affine elements
  const int32_t* nb;                            // [N][4] neighbour or -1-edge
  const int8_t* nbf;                            // [N][4] neighbour's face
  const int8_t *sw_psi, *sw_diff;               // [E] 0 Dirichlet / 1 Neumann
  const int8_t* no_slip;                        // [E]
  const double* esign;                          // [E] 2*(ijp%2)-1 of the owner face
  const int32_t* inst;                          // [N] ensemble instance of each element, or null
  const double* dcol;                           // [K][K]     l_d'(xi_k), k first
  const double* wrow;                           // [K]        weights
  const double* qn;                             // [E][K][K]  see FineGeo
};

// Hybrid operation (problem_type 11): per-edge kind and the open-boundary values at the
// start and end of the outer step, blended per stage (src/HO_2D.cpp:2104-2191).
struct HybridDev {
  const uint8_t* kind;       // [E] 0 wall, 1 open, 2 inlet, 3 outlet
  const double* inlet_nvel;  // [E]
  const double* esign;       // [E]
  const int8_t* sw_diff;     // [E]
  const double *vn0, *vn1, *vp0, *vp1, *vw0, *vw1;  // [E][K] normal/tangential velocity, vorticity
  const double *w0, *w1, *wgt;                      // [N][K2] solution vorticity targets and weights
};

// Per-instance parameters of an ensemble (null pointers: one instance, scalar arguments).
struct InstDev {
  const double* re_inv;      // [n_inst] 1/Re
  const double* dt;          // [n_inst] time step
  const double* inv_dt_re;   // [n_inst] 1/(dt Re^-1), wall-vorticity flux scale
  const double* ramp;        // [n_inst] time factor of the boundary values at the stage time
  const int32_t* edge_inst;  // [E] instance of each boundary edge
};

// Time-dependent boundary values [E][K] (edge flux-point order).
struct BCDev {
  double *psi, *diff, *nvel, *pvel, *vjump, *vort, *adv;
  const double *psi0, *psi_r, *diff0, *diff_r, *nvel0, *nvel_r, *pvel0, *pvel_r;
};

}  // namespace hoc
