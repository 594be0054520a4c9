// hoc_fr.hpp - launchers of the FR stage kernels (hoc_fr.hip).
#pragma once

#include "hoc_kernels.hpp"

namespace hoc {

// Outputs of the stage kernel.
struct StageOut {
  double* k = nullptr;       // k_s = dt (adv + diff), or nullptr
  double* next = nullptr;    // base + c k_s (next stage input), or nullptr
  double c = 0.;
  double* base = nullptr;    // omega_n (read for next; updated for final_mode)
  int final_mode = 0;        // 0 none, 1 Euler, 2 RK2 (needs k1), 4 RK4 (needs k1..k3)
  const double *k1 = nullptr, *k2 = nullptr, *k3 = nullptr;
  // linearised stage (launch_stage mode 1 records, mode 2 reads the upwind switches)
  int8_t* sig = nullptr;               // [N][4][K] upwind switch of each interior flux point
  const double* omega_adv = nullptr;   // mode 2: advected vorticity and its traces
  const double* trw_adv = nullptr;
  // mode 2 batches: nbatch independent products in one launch, probe b reading/writing its
  // arrays at b * (stride in values); stride 0 shares an array between the probes
  int nbatch = 1;
  int adv_only = 0;  // mode 2: the diffusion inputs are zero (skip the diffusion term)
  size_t bs_w = 0, bs_trw = 0, bs_U = 0, bs_tru = 0, bs_wa = 0, bs_trwa = 0, bs_k = 0, bs_diff = 0;
};

// Batch strides (in values) of the batched velocity launch.
struct VelBatch {
  size_t psi = 0, trpsi = 0, omega = 0, vel = 0, U = 0, trw = 0, tru = 0, vjump = 0, diff = 0, pvel = 0;
};

// Face traces of x (face-major, see hoc_fr.hip).
hipError_t launch_trace(int K, int N, const Tab& T, const double* x, double* tr, hipStream_t s);
hipError_t launch_rhs(int K, int N, const Tab& T, const Geo& G, const double* omega, const double* bcpsi, double* bs,
                      double* part, hipStream_t s);
hipError_t launch_velocity(int K, int N, const Tab& T, const Geo& G, const BCDev& B, const double* psi,
                           const double* trpsi, const double* omega, double* vel, double* U, double* trw,
                           double* tru, double inv_dt_re, const InstDev& I, hipStream_t s);
// nbatch velocity evaluations in one launch (probe b offset by b * the strides of vb)
hipError_t launch_velocity_batch(int K, int N, const Tab& T, const Geo& G, const BCDev& B, const double* psi,
                                 const double* trpsi, const double* omega, double* vel, double* U, double* trw,
                                 double* tru, double inv_dt_re, const InstDev& I, int nbatch, const VelBatch& vb,
                                 hipStream_t s);
hipError_t launch_stage(int K, int adv, int N, const Tab& T, const Geo& G, const BCDev& B, const double* omega,
                        const double* U, const double* trw, const double* tru, double re_inv, double dt,
                        const InstDev& I, const StageOut& so, hipStream_t s, int mode = 0);
// n = E*K boundary values; tc = time factor (per instance through I.ramp when set)
hipError_t launch_update_bcs(int n, int K, const BCDev& B, double tc, const InstDev& I, hipStream_t s);
// problem_type 11: boundary values at fraction fac1 (fac2 = 1 - fac1) of the outer step,
// and the blend w = (1 - wgt) w + wgt (fac1 w0 + fac2 w1)
hipError_t launch_update_bcs_hybrid(int n, int K, const BCDev& B, const HybridDev& H, double fac1, double fac2,
                                    hipStream_t s);
hipError_t launch_hybrid_blend(size_t n, double* w, const HybridDev& H, double fac1, double fac2, hipStream_t s);
int lap_blocks(int N);

}  // namespace hoc
