// hoc_fr.hpp - launchers of the stage kernels (hoc_stage.hip) and of the boundary values (hoc_fr.hip).
#pragma once

#include "hoc_kernels.hpp"

namespace hoc {

// Outputs of the stage kernel.
struct StageOut {
  double* k = nullptr;       // k_s = dt (adv + diff), or nullptr
  double* next = nullptr;    // base + c k_s (next stage input), or nullptr
  double c = 0.;
  double* base = nullptr;    // omega_n (read for next; updated for final_mode)
  int final_mode = 0;        // 0 none, 2 RK2 (needs k1), 4 RK4 (needs k1..k3)
  const double *k1 = nullptr, *k2 = nullptr, *k3 = nullptr;
  // linearised stage (launch_stage mode 1 records, mode 2 reads the upwind switches)
  int8_t* sig = nullptr;               // [N][4][K] upwind switch of each interior flux point
  // mode 2 batches: nbatch independent products in one launch, probe b reading/writing its
  // arrays at b * (stride in values); stride 0 shares an array between the probes
  int nbatch = 1;
  int adv_only = 0;  // mode 2: the diffusion inputs are zero (skip the diffusion term)
  size_t bs_w = 0, bs_U = 0, bs_tru = 0, bs_k = 0, bs_diff = 0;
  bool inner = false;  // an intermediate stage: the Cartesian velocity is not an output
};

// Batch strides (in values) of the batched velocity launch.
struct VelBatch {
  size_t psi = 0, U = 0, tru = 0, vjump = 0, diff = 0, pvel = 0;
};

// geo: GEO_ORTHO, GEO_AFFINE or GEO_POINT (hoc_poisson.hpp).  part: fine_blocks(K, N) sums.
hipError_t launch_rhs(int K, int geo, int N, const Tab& T, const Geo& G, const double* omega, const double* bcpsi,
                      double* bs, double* part, hipStream_t s);
// vel may be null; tru: the normal traces of U, face-major [4][N][K].  nbatch velocity evaluations in one
// launch: probe b offset by b * the strides of vb, vel null.
hipError_t launch_velocity(int K, int geo, int N, const Tab& T, const Geo& G, const BCDev& B, const double* psi,
                           double* vel, double* U, double* tru, double inv_dt_re, const InstDev& I, hipStream_t s,
                           int nbatch = 1, const VelBatch& vb = VelBatch{});
// omega may be none of the arrays that the launch writes.
hipError_t launch_stage(int K, int geo, int adv, int N, const Tab& T, const Geo& G, const BCDev& B,
                        const double* omega, const double* U, const double* tru, double re_inv, double dt,
                        const InstDev& I, const StageOut& so, hipStream_t s, int mode = 0);
// n = E*K boundary values; tc = time factor (per instance through I.ramp when set)
hipError_t launch_update_bcs(int n, int K, const BCDev& B, double tc, const InstDev& I, hipStream_t s);
// problem_type 11: boundary values at fraction fac1 (fac2 = 1 - fac1) of the outer step,
// and the blend w = (1 - wgt) w + wgt (fac1 w0 + fac2 w1)
hipError_t launch_update_bcs_hybrid(int n, int K, const BCDev& B, const HybridDev& H, double fac1, double fac2,
                                    hipStream_t s);
hipError_t launch_hybrid_blend(size_t n, double* w, const HybridDev& H, double fac1, double fac2, hipStream_t s);

}  // namespace hoc
