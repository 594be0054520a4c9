// hoc_stage.hip - the Poisson right-hand side, the velocity and the stage kernel for gfx950.
//
// Velocity from the stream function (src/HO_2D.cpp:3174-3366), diffusion (src/HO_2D.cpp:2666-2831),
// advection (src/HO_2D.cpp:2245-2645) and the RK stage update (src/HO_2D.cpp:1465-1531, 1833-1836).
//
// K lanes per element as in hoc_rowlane.hpp.  What a face needs from the neighbour is one line of its
// field, read where it lies, so no kernel leaves face traces behind; only the contravariant normal
// velocity on the faces is stored (one value against a line of K).  An element a thread, with the
// element's values in registers and traces stored between the kernels, left 4 wavefronts a CU at 512 x
// 512 elements and a serial chain at 32 x 32.  Before and now, us: 512 x 512, K = 5, velocity 152 + 34
// for the traces, now 107; stage 185, now 132; right-hand side 65, now 30 (its HBM time is 26); 32 x 32,
// K = 4, velocity 18 + 3.5, now 6.5; stage 21.7, now 7.1; 96 x 96 curved, K = 6, velocity 45 + 7, now 19,
// stage 110, now 26.  Registers bound velocity and stage (2 wavefronts a SIMD; held to 3, velocity spills
// and takes 131 us).
#include "hoc_fr.hpp"
#include "hoc_rowlane.hpp"

namespace hoc {

namespace {

__device__ __forceinline__ int face_sign(int f, int fn) { return ((f + fn) & 1) ? 1 : -1; }
// element-local flux point k of face f -> boundary-edge flux point (src/HO_2D.cpp:2229)
template <int K>
__device__ __forceinline__ int edge_fp(int f, int k) { return (f == 0 || f == 3) ? K - 1 - k : k; }

// Where a lane stands.
template <int K>
struct Lane {
  static constexpr int EPW = Lay<K>::EPW, EPB = EPW * (kFineThreads / 64);
  int blk, wv, le, k, el;
  bool live;
  __device__ __forceinline__ explicit Lane(int N) {
    blk = xcd_block(blockIdx.x, gridDim.x);
    wv = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    // lanes past the mesh follow its last element, lanes past the last slot its last row; neither
    // writes to memory
    le = lane < EPW * K ? lane / K : EPW - 1;
    k = lane < EPW * K ? lane - le * K : K - 1;
    const int e0 = blk * EPB + wv * EPW + le;
    live = lane < EPW * K && e0 < N;
    el = min(e0, N - 1);
  }
};

// The neighbours across an element's faces, seen from a lane's face points.
template <int K>
struct Nbrs {
  int nb[4], fn[4], kk[4];
  bool opp[4];
  __device__ __forceinline__ Nbrs(const Geo& G, int el, int k) {
    const int4 n4 = *reinterpret_cast<const int4*>(G.nb + (size_t)el * 4);
    const int nf = reinterpret_cast<const int32_t*>(G.nbf)[el];
    const int n[4] = {n4.x, n4.y, n4.z, n4.w};
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      nb[f] = n[f];
      const int g = n[f] >= 0 ? (nf >> (8 * f)) & 3 : f ^ 1;
      opp[f] = __all(g == (f ^ 1));
      fn[f] = opp[f] ? (f ^ 1) : g;
      kk[f] = opp[f] ? k : face_point<K>(f, g, k);
    }
  }
  // value and inward derivative of x at the lane's face points on the neighbours' sides (a boundary
  // face reads the element's own line, and nothing uses it)
  __device__ __forceinline__ void traces(const Tab& T, const double* __restrict__ x, int el, int k, double (&v)[4],
                                         double (&g)[4]) const {
    double l[4][K];
#pragma unroll
    for (int f = 0; f < 4; ++f) nbr_line<K>(x, nb[f] >= 0 ? nb[f] : el, f, fn[f], kk[f], k, opp[f], l[f]);
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      v[f] = 0.;
      g[f] = 0.;
#pragma unroll
      for (int m = 0; m < K; ++m) {
        v[f] += l[f][m] * T.bb[m][0];
        g[f] += l[f][m] * T.bgb[m][0];
      }
    }
  }
};

// Own value and coordinate derivative at the lane's face points, from its row and column.
template <int K>
__device__ __forceinline__ void own_traces(const Tab& T, const double (&u)[K], const double (&uc)[K], double (&bv)[4],
                                           double (&bg)[4]) {
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    bv[f] = 0.;
    bg[f] = 0.;
#pragma unroll
    for (int m = 0; m < K; ++m) {
      const double x = f < 2 ? u[m] : uc[m];
      bv[f] += x * T.bb[m][f & 1];
      bg[f] += x * T.bgb[m][f & 1];
    }
  }
}

// Common value and common normal flux of the second-order operator at the lane's face points: inside,
// the average of both sides (src/HO_2D.cpp:2742-2768, 2833-2870); on the boundary, by the switch sw,
// the value bc or the flux bc |g| with the value from it (src/HO_2D.cpp:2872-2927; the K x K system of
// a face with tangential metrics is inverted at setup, G.qn).  bcv: edge values (null: zero).
// Tangential derivatives along a face go through tf, 4 K values of LDS per element; dcv (NVEL) receives
// those of the common values where a face of the wavefront is a Neumann one.
template <int K, int GEO, bool NVEL>
__device__ __forceinline__ void common_faces(const Tab& T, const Geo& G, const Nbrs<K>& Nb, int el, int k, double* tf,
                                             const int8_t* __restrict__ sw, const double* __restrict__ bcv,
                                             bool signed_neumann, const double (&bv)[4], const double (&bg)[4],
                                             const double (&vn)[4], const double (&gn)[4], double (&cv)[4],
                                             double (&cg)[4], double (&dcv)[NVEL ? 4 : 1]) {
  constexpr bool TAN = GEO != GEO_ORTHO;
  bool neu[4];
  double fa[4], fb[TAN ? 4 : 1];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const int nb = Nb.nb[f];
    if constexpr (GEO == GEO_POINT) {
      const size_t q = ((size_t)el * 4 + f) * K + k;
      fa[f] = G.fa[q];
      fb[f] = G.fb[q];
    } else {
      fa[f] = G.gface[((size_t)el * 4 + f) * 2];
      if constexpr (TAN) fb[f] = G.gface[((size_t)el * 4 + f) * 2 + 1];
    }
    neu[f] = false;
    cg[f] = 0.;
    if (nb >= 0) {
      cv[f] = 0.5 * (bv[f] + vn[f]);
    } else {
      const int e = -1 - nb;
      const double b = bcv ? bcv[(size_t)e * K + edge_fp<K>(f, k)] : 0.;
      neu[f] = sw[e] != 0;
      cv[f] = b;
      if (neu[f]) {
        const size_t q = ((size_t)el * 4 + f) * K + k;
        const double A = G.fA[q];
        cg[f] = (signed_neumann ? G.esign[e] * b : b) * G.fAn[q];
        cv[f] = (G.fjac[q] * cg[f] - A * bg[f]) / (A * T.gp[f & 1]) + bv[f];
      }
    }
  }
  double cr[TAN ? 4 : 1];
  // without tangential metrics only Neumann faces (of any lane) need a derivative, for their velocity
  if (TAN || (NVEL && __any(neu[0] || neu[1] || neu[2] || neu[3]))) {
    const double* D = G.dcol + k * K;  // l_d'(xi_k)
    if constexpr (TAN) {
      wave_fence();
#pragma unroll
      for (int f = 0; f < 4; ++f) tf[f * K + k] = cv[f];
      wave_fence();
#pragma unroll
      for (int f = 0; f < 4; ++f)
        if (neu[f]) {
          const double* q = G.qn + ((size_t)(-1 - Nb.nb[f]) * K + k) * K;
          double s = 0.;
#pragma unroll
          for (int i = 0; i < K; ++i) s += q[i] * tf[f * K + i];
          cv[f] = s;
        }
    }
    wave_fence();
#pragma unroll
    for (int f = 0; f < 4; ++f) tf[f * K + k] = cv[f];
    wave_fence();
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      double s = 0.;
#pragma unroll
      for (int d = 0; d < K; ++d) s += tf[f * K + d] * D[d];
      if constexpr (TAN) cr[f] = s;
      if constexpr (NVEL) dcv[f] = s;
    }
  }
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    if (neu[f]) continue;
    const double dv = bg[f] + (cv[f] - bv[f]) * T.gp[f & 1];
    double F = dv * fa[f];
    if constexpr (TAN) F -= cr[f] * fb[f];
    const int nb = Nb.nb[f];
    if (nb < 0) {
      cg[f] = F;
      continue;
    }
    // the neighbour's derivative along its own coordinate: inward at its lower faces
    const int fn = Nb.fn[f];
    const double gc = (fn & 1) ? -gn[f] : gn[f], gp = (fn & 1) ? T.gp[1] : T.gp[0];
    const double dvn = gc + (cv[f] - vn[f]) * gp;
    double Fn;
    if constexpr (GEO == GEO_POINT) {
      const size_t q = ((size_t)nb * 4 + fn) * K + Nb.kk[f];
      Fn = dvn * G.fa[q] - (((f + fn - f / 2 - fn / 2 + 1) & 1) ? -cr[f] : cr[f]) * G.fb[q];
    } else {
      const size_t q = ((size_t)nb * 4 + fn) * 2;
      Fn = dvn * G.gface[q];
      if constexpr (TAN) Fn -= (((f + fn - f / 2 - fn / 2 + 1) & 1) ? -cr[f] : cr[f]) * G.gface[q + 1];
    }
    cg[f] = 0.5 * (F + (face_sign(f, fn) > 0 ? Fn : -Fn));
  }
}

// The corrected gradient's contravariant components (src/HO_2D.cpp:2771-2816): the xi one on the lane's
// row (ft, with the Radau amplitudes fB of its two ends), the eta one on its column (gt, gB).
template <int K, int GEO>
__device__ __forceinline__ void gradient(const Tab& T, const Geo& G, int el, int k, double* t, const double (&u)[K],
                                         const double (&uc)[K], const double (&bv)[4], const double (&cv)[4],
                                         const double (&cg)[4], double (&ft)[K], double (&gt)[K], double (&fB)[2],
                                         double (&gB)[2]) {
  double dx[K], de[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    double a = 0., b = 0.;
#pragma unroll
    for (int d = 0; d < K; ++d) { a += u[d] * T.D[d][i]; b += uc[d] * T.D[d][i]; }
    dx[i] = a + (cv[0] - bv[0]) * T.grad[i][0] + (cv[1] - bv[1]) * T.grad[i][1];
    de[i] = b + (cv[2] - bv[2]) * T.grad[i][0] + (cv[3] - bv[3]) * T.grad[i][1];
  }
  if constexpr (GEO == GEO_ORTHO) {
    const double a = G.gel[(size_t)el * 3], c = G.gel[(size_t)el * 3 + 2];
#pragma unroll
    for (int i = 0; i < K; ++i) { ft[i] = dx[i] * a; gt[i] = de[i] * c; }
  } else {
    double der[K], dxc[K];
    cols_to_rows<K>(t, k, de, der);
    rows_to_cols<K>(t, k, dx, dxc);
    if constexpr (GEO == GEO_AFFINE) {
      const double a = G.gel[(size_t)el * 3], b = G.gel[(size_t)el * 3 + 1], c = G.gel[(size_t)el * 3 + 2];
#pragma unroll
      for (int i = 0; i < K; ++i) {
        ft[i] = dx[i] * a - der[i] * b;
        gt[i] = de[i] * c - dxc[i] * b;
      }
    } else {
      const size_t o = (size_t)el * K * K;
      double ga[K], gb[K];
      load_row<K>(G.Ga + o + k * K, ga);
      load_row<K>(G.Gb + o + k * K, gb);
#pragma unroll
      for (int i = 0; i < K; ++i) {
        ft[i] = dx[i] * ga[i] - der[i] * gb[i];
        gt[i] = de[i] * G.Gc[o + i * K + k] - dxc[i] * G.Gb[o + i * K + k];
      }
    }
  }
#pragma unroll
  for (int ib = 0; ib < 2; ++ib) {
    double a = cg[ib], b = cg[2 + ib];
#pragma unroll
    for (int d = 0; d < K; ++d) { a -= ft[d] * T.bb[d][ib]; b -= gt[d] * T.bb[d][ib]; }
    fB[ib] = a;
    gB[ib] = b;
  }
}

// Corrected derivative along a line: out = D v + end amplitudes.
template <int K>
__device__ __forceinline__ void line_div(const Tab& T, const double (&v)[K], const double (&B)[2], double (&out)[K]) {
#pragma unroll
  for (int i = 0; i < K; ++i) {
    double r = 0.;
#pragma unroll
    for (int d = 0; d < K; ++d) r += v[d] * T.D[d][i];
    out[i] = r + B[0] * T.grad[i][0] + B[1] * T.grad[i][1];
  }
}

// LDS of a wavefront: its tile, and 4 K face values per element.
template <int K>
struct Lds {
  static constexpr int W = Lay<K>::TILE + Lay<K>::EPW * 4 * K;
  static constexpr int N = (kFineThreads / 64) * W;
  static __device__ __forceinline__ double* tile(double* lds, const Lane<K>& L) {
    return lds + L.wv * W + L.le * Lay<K>::ES;
  }
  static __device__ __forceinline__ double* faces(double* lds, const Lane<K>& L) {
    return lds + L.wv * W + Lay<K>::TILE + L.le * 4 * K;
  }
};

// ==========================================================================================
// Poisson right-hand side (src/HO_2D.cpp:1881-1900) in the scaled form
//   bs = W (omega J + L(0; BC_psi)),   with partial sums of (bs/W)^2 = ||b||^2.
// Neumann values enter with the owner face's outward sign: boundary_source . BC_Poisson
// (src/HO_2D.cpp:1660-1714, sign (2t-1) of :1685) equals L(0; sign * BC) on such faces.  Bound by HBM:
// omega and bs (and J where it varies); wavefronts without a boundary element skip L.
// ==========================================================================================
template <int K, int GEO>
__global__ __launch_bounds__(kFineThreads) void k_rhs(int N, Tab T, Geo G, const double* __restrict__ omega,
                                                      const double* __restrict__ bcpsi, double* __restrict__ bs,
                                                      double* __restrict__ part) {
  __shared__ double lds[Lds<K>::N];
  __shared__ double sp[kFineThreads / 64];
  const Lane<K> L(N);
  const int el = L.el, k = L.k;
  double *t = Lds<K>::tile(lds, L), *tf = Lds<K>::faces(lds, L);
  const size_t row = ((size_t)el * K + k) * K;
  double w[K], jac[K], out[K];
  load_row<K>(omega + row, w);
  if constexpr (GEO == GEO_POINT) {
    load_row<K>(G.jac + row, jac);
  } else {
    const double j = G.gjm[(size_t)el * 5 + 4];
#pragma unroll
    for (int i = 0; i < K; ++i) jac[i] = j;
  }
  const Nbrs<K> Nb(G, el, k);
  const bool bnd = Nb.nb[0] < 0 || Nb.nb[1] < 0 || Nb.nb[2] < 0 || Nb.nb[3] < 0;
#pragma unroll
  for (int i = 0; i < K; ++i) out[i] = 0.;
  if (__any(bnd)) {
    const double z[K] = {}, z4[4] = {};
    double cv[4], cg[4], ft[K], gt[K], fB[2], gB[2], oc[K], oc_r[K], none[1];
    common_faces<K, GEO, false>(T, G, Nb, el, k, tf, G.sw_psi, bcpsi, true, z4, z4, z4, z4, cv, cg, none);
    gradient<K, GEO>(T, G, el, k, t, z, z, z4, cv, cg, ft, gt, fB, gB);
    line_div<K>(T, ft, fB, out);
    line_div<K>(T, gt, gB, oc);
    cols_to_rows<K>(t, k, oc, oc_r);
#pragma unroll
    for (int i = 0; i < K; ++i) out[i] += oc_r[i];
  }
  double p0 = 0.;
  const double wk = G.wrow[k];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    const double b = -w[i] * jac[i] - out[i];  // unscaled reference RHS
    p0 += b * b;
    out[i] = -(wk * T.w[i]) * b;
  }
  if (L.live) store_row<K>(bs + row, out);
  else p0 = 0.;
  p0 = wave_sum(p0);
  if ((threadIdx.x & 63) == 0) sp[threadIdx.x >> 6] = p0;
  __syncthreads();
  if (threadIdx.x == 0) part[L.blk] = sp[0] + sp[1] + sp[2] + sp[3];
}

// ==========================================================================================
// Velocity from the stream function (src/HO_2D.cpp:3174-3366) with the no-slip wall vorticity flux
// (update_diffusion_BC, src/HO_2D.cpp:2647-2664): the contravariant fluxes U, their normal traces on
// the faces (src/HO_2D.cpp:2332, 2489-2503; face-major [4][N][K]) and, where it is asked for, the
// Cartesian velocity.
// ==========================================================================================
template <int K, int GEO>
__global__ __launch_bounds__(kFineThreads) void k_velocity(int N, Tab T, Geo G, BCDev B,
                                                           const double* __restrict__ psi, double* __restrict__ vel,
                                                           double* __restrict__ U, double* __restrict__ tru,
                                                           double inv_dt_re, InstDev I, VelBatch vb) {
  constexpr int K2 = K * K;
  {  // probe blockIdx.y of a batch
    const size_t b = blockIdx.y;
    psi += b * vb.psi; U += b * vb.U; tru += b * vb.tru;
    B.vjump += b * vb.vjump; B.diff += b * vb.diff; B.pvel += b * vb.pvel;
  }
  __shared__ double lds[Lds<K>::N];
  const Lane<K> L(N);
  const int el = L.el, k = L.k;
  double *t = Lds<K>::tile(lds, L), *tf = Lds<K>::faces(lds, L);
  const size_t row = ((size_t)el * K + k) * K;
  double u[K], uc[K], bv[4], bg[4], vn[4], gn[4], cv[4], cg[4], dcv[4];
  const Nbrs<K> Nb(G, el, k);
  load_row<K>(psi + row, u);
  Nb.traces(T, psi, el, k, vn, gn);
  rows_to_cols<K>(t, k, u, uc);
  own_traces<K>(T, u, uc, bv, bg);
  common_faces<K, GEO, true>(T, G, Nb, el, k, tf, G.sw_psi, B.psi, true, bv, bg, vn, gn, cv, cg, dcv);
  // boundary side effects
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    if (Nb.nb[f] >= 0 || !L.live) continue;
    const int e = -1 - Nb.nb[f];
    const size_t i = (size_t)e * K + edge_fp<K>(f, k);
    const double an = G.fAn[((size_t)el * 4 + f) * K + k];
    const bool dir = G.sw_psi[e] == 0;
    double vj = 0.;
    if (dir) vj = cg[f] / an;
    else B.nvel[i] = (f < 2 ? dcv[f] : -dcv[f]) / an;
    if (G.no_slip[e]) {
      vj = (dir ? vj : B.vjump[i]) + G.esign[e] * B.pvel[i];
      B.diff[i] = vj * (I.inv_dt_re ? I.inv_dt_re[G.inst[el]] : inv_dt_re);
    }
    if (dir || G.no_slip[e]) B.vjump[i] = vj;
  }
  double tx[K], ty[K], fB[2], gB[2], tyc[K];
  gradient<K, GEO>(T, G, el, k, t, u, uc, bv, cv, cg, tx, tyc, fB, gB);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    tx[i] += fB[0] * T.rad[i][0] + fB[1] * T.rad[i][1];
    tyc[i] += gB[0] * T.rad[i][0] + gB[1] * T.rad[i][1];
  }
  cols_to_rows<K>(t, k, tyc, ty);
  double m[GEO == GEO_POINT ? 1 : 5];
  if constexpr (GEO != GEO_POINT) {
#pragma unroll
    for (int i = 0; i < 5; ++i) m[i] = G.gjm[(size_t)el * 5 + i];
  }
  double U1[K], U2[K], U2c[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    double xxi, xet, yxi, yet, J;
    if constexpr (GEO == GEO_POINT) {
      xxi = G.xxi[row + i]; xet = G.xeta[row + i]; yxi = G.yxi[row + i]; yet = G.yeta[row + i]; J = G.jac[row + i];
    } else {
      xxi = m[0]; xet = m[1]; yxi = m[2]; yet = m[3]; J = m[4];
    }
    const double vx = (tx[i] * yxi + ty[i] * yet) / J;   // u =  dpsi/dy
    const double vy = -((tx[i] * xxi + ty[i] * xet) / J);  // v = -dpsi/dx
    if (vel && L.live) {  // intermediate RK stages skip it
      const double v[2] = {vx, vy};
      store_row<2>(vel + 2 * (row + i), v);
    }
    U1[i] = vx * yet - vy * xet;   // J (xi_x u + xi_y v)
    U2[i] = -vx * yxi + vy * xxi;  // J (eta_x u + eta_y v)
  }
  rows_to_cols<K>(t, k, U2, U2c);
  if (!L.live) return;
  double* Ue = U + (size_t)el * 2 * K2 + k * K;
  store_row<K>(Ue, U1);
  store_row<K>(Ue + K2, U2);
#pragma unroll
  for (int ib = 0; ib < 2; ++ib) {
    double s = 0., s2 = 0.;
#pragma unroll
    for (int i = 0; i < K; ++i) { s += U1[i] * T.bb[i][ib]; s2 += U2c[i] * T.bb[i][ib]; }
    tru[((size_t)ib * N + el) * K + k] = s;
    tru[((size_t)(2 + ib) * N + el) * K + k] = s2;
  }
}

// ==========================================================================================
// The stage: diffusion (src/HO_2D.cpp:2666-2831), advection (src/HO_2D.cpp:2245-2645; ADV 1 the
// upwinded flux, ADV 2 the continuous volumetric flux of :2539-2546) and the RK combination.  omega is
// read at neighbours, so no output of the launch may be the array that it reads (launch_stage).
// MODE 1 records the upwind switches, MODE 2 (probes of the adjoint, in batches) uses them.
// ==========================================================================================
template <int K, int ADV, int GEO, int MODE>
__global__ __launch_bounds__(kFineThreads) void k_stage(int N, Tab T, Geo G, BCDev B, const double* __restrict__ omega,
                                                        const double* __restrict__ U, const double* __restrict__ tru,
                                                        double re_inv, double dt, InstDev I, StageOut so) {
  constexpr int K2 = K * K;
  if constexpr (MODE == 2) {  // probe blockIdx.y of a batch
    const size_t b = blockIdx.y;
    omega += b * so.bs_w; U += b * so.bs_U; tru += b * so.bs_tru; so.k += b * so.bs_k; B.diff += b * so.bs_diff;
  }
  __shared__ double lds[Lds<K>::N];
  const Lane<K> L(N);
  const int el = L.el, k = L.k;
  double *t = Lds<K>::tile(lds, L), *tf = Lds<K>::faces(lds, L);
  const size_t row = ((size_t)el * K + k) * K;
  const bool do_diff = MODE != 2 || !so.adv_only;  // zero vorticity and wall flux for the diffusion term
  const Nbrs<K> Nb(G, el, k);
  double w[K], wc[K], U1[K], U2[K], vn[4], gn[4], un[4], bv[4], bg[4], cv[4], cg[4];
  load_row<K>(omega + row, w);
  load_row<K>(U + (size_t)el * 2 * K2 + k * K, U1);
#pragma unroll
  for (int j = 0; j < K; ++j) U2[j] = U[(size_t)el * 2 * K2 + K2 + j * K + k];  // the column of U^2
#pragma unroll
  for (int f = 0; f < 4; ++f)
    un[f] = tru[((size_t)Nb.fn[f] * N + (Nb.nb[f] >= 0 ? Nb.nb[f] : el)) * K + Nb.kk[f]];
  Nb.traces(T, omega, el, k, vn, gn);
  rows_to_cols<K>(t, k, w, wc);
  own_traces<K>(T, w, wc, bv, bg);
  double rr[K], rc[K];  // diffusion, then everything: the row's and the column's shares
#pragma unroll
  for (int i = 0; i < K; ++i) { rr[i] = 0.; rc[i] = 0.; }
#pragma unroll
  for (int f = 0; f < 4; ++f) cv[f] = 0.;
  if (do_diff) {
    double ft[K], gt[K], fB[2], gB[2], none[1];
    common_faces<K, GEO, false>(T, G, Nb, el, k, tf, G.sw_diff, B.diff, false, bv, bg, vn, gn, cv, cg, none);
    gradient<K, GEO>(T, G, el, k, t, w, wc, bv, cv, cg, ft, gt, fB, gB);
    line_div<K>(T, ft, fB, rr);
    line_div<K>(T, gt, gB, rc);
    const double ri = I.re_inv ? I.re_inv[G.inst[el]] : re_inv;
#pragma unroll
    for (int i = 0; i < K; ++i) { rr[i] *= ri; rc[i] *= ri; }
  }
  // advective fluxes at the face points
  double bu[4], upw[4], cvf[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    double s = 0.;
#pragma unroll
    for (int i = 0; i < K; ++i) s += (f < 2 ? U1[i] : U2[i]) * T.bb[i][f & 1];
    bu[f] = s;
    cvf[f] = 0.;
    const size_t q = ((size_t)el * 4 + f) * K + k;
    if (Nb.nb[f] < 0) {  // boundary vorticity times the boundary's normal velocity
      const size_t i = (size_t)(-1 - Nb.nb[f]) * K + edge_fp<K>(f, k);
      const double an = G.fAn[q], nv = B.nvel[i];
      upw[f] = cv[f] * nv * an;
      if (ADV == 2) cvf[f] = nv * an;
      if constexpr (MODE != 2) {
        if (L.live) {
          B.vort[i] = cv[f];
          B.adv[i] = upw[f];
        }
      }
      continue;
    }
    const double sgn = face_sign(f, Nb.fn[f]);
    if (ADV == 1) {
      const double fo = bu[f] * bv[f], fnn = un[f] * vn[f];
      double up = 0.5 * (fo + sgn * fnn);
      const double dw = bv[f] - vn[f], df = fo - sgn * fnn, side = (f & 1) ? 1. : -1.;
      if constexpr (MODE == 2) {
        up += 0.5 * side * (double)so.sig[q] * df;
      } else {
        if (fabs(dw) > 1.e-4) up += 0.5 * side * fabs(df / dw) * dw;
        if constexpr (MODE == 1) {
          const int sd = dw > 0. ? 1 : -1, sf = df > 0. ? 1 : (df < 0. ? -1 : 0);
          if (L.live) so.sig[q] = (int8_t)(fabs(dw) > 1.e-4 ? sd * sf : 0);
        }
      }
      upw[f] = up;
    } else {
      const double c = 0.5 * (bu[f] + sgn * un[f]);
      const bool own = (f & 1) ? c > 0. : !(c > 0.);
      cvf[f] = c;
      upw[f] = c * (own ? bv[f] : vn[f]);
    }
  }
  // discontinuous fluxes U^1 w on the row, U^2 w on the column, and their end amplitudes
  double f1[K], f2[K], B1[2], B2[2], d1[K], d2[K];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    double a = U1[i], b = U2[i];
    if (ADV == 2) {
      a += (cvf[0] - bu[0]) * T.rad[i][0] + (cvf[1] - bu[1]) * T.rad[i][1];
      b += (cvf[2] - bu[2]) * T.rad[i][0] + (cvf[3] - bu[3]) * T.rad[i][1];
    }
    f1[i] = a * w[i];
    f2[i] = b * wc[i];
  }
#pragma unroll
  for (int ib = 0; ib < 2; ++ib) {
    double a = upw[ib], b = upw[2 + ib];
#pragma unroll
    for (int i = 0; i < K; ++i) { a -= f1[i] * T.bb[i][ib]; b -= f2[i] * T.bb[i][ib]; }
    B1[ib] = a;
    B2[ib] = b;
  }
  line_div<K>(T, f1, B1, d1);
  line_div<K>(T, f2, B2, d2);
  double kk[K];
#pragma unroll
  for (int i = 0; i < K; ++i) rc[i] -= d2[i];
  cols_to_rows<K>(t, k, rc, kk);
  const double dti = I.dt ? I.dt[G.inst[el]] : dt;
  double J[K];
  if constexpr (GEO == GEO_POINT) {
    load_row<K>(G.jac + row, J);
  } else {
    const double j = G.gjm[(size_t)el * 5 + 4];
#pragma unroll
    for (int i = 0; i < K; ++i) J[i] = j;
  }
#pragma unroll
  for (int i = 0; i < K; ++i) kk[i] = dti * ((kk[i] + (rr[i] - d1[i])) / J[i]);
  if (!L.live) return;
  // outputs: k, and the RK combination
  if (so.k) store_row<K>(so.k + row, kk);
  if (!so.next && !so.final_mode) return;
  double b[K], o[K];
  load_row<K>(so.base + row, b);
  if (so.next) {  // next stage input: base + c k
#pragma unroll
    for (int i = 0; i < K; ++i) o[i] = b[i] + so.c * kk[i];
    store_row<K>(so.next + row, o);
  }
  if (so.final_mode) {  // vorticity update
    double k1[K], k2[K], k3[K];
    load_row<K>(so.k1 + row, k1);
    if (so.final_mode == 4) {
      load_row<K>(so.k2 + row, k2);
      load_row<K>(so.k3 + row, k3);
    }
#pragma unroll
    for (int i = 0; i < K; ++i) {
      if (so.final_mode == 2) o[i] = b[i] + 0.5 * (k1[i] + kk[i]);
      else o[i] = b[i] + (k1[i] + 2. * k2[i] + 2. * k3[i] + kk[i]) / 6.;
    }
    store_row<K>(so.base + row, o);
  }
}

}  // namespace

#define HOC_K_SWITCH(KV, ...)            \
  switch (KV) {                          \
    case 2: { constexpr int KK = 2; __VA_ARGS__; } break; \
    case 3: { constexpr int KK = 3; __VA_ARGS__; } break; \
    case 4: { constexpr int KK = 4; __VA_ARGS__; } break; \
    case 5: { constexpr int KK = 5; __VA_ARGS__; } break; \
    case 6: { constexpr int KK = 6; __VA_ARGS__; } break; \
    default: return hipErrorInvalidValue; \
  }
#define HOC_GEO_SWITCH(GV, ...)          \
  switch (GV) {                          \
    case GEO_ORTHO: { constexpr int GG = GEO_ORTHO; __VA_ARGS__; } break; \
    case GEO_AFFINE: { constexpr int GG = GEO_AFFINE; __VA_ARGS__; } break; \
    case GEO_POINT: { constexpr int GG = GEO_POINT; __VA_ARGS__; } break; \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_rhs(int K, int geo, int N, const Tab& T, const Geo& G, const double* omega, const double* bcpsi,
                      double* bs, double* part, hipStream_t s) {
  if (N == 0) return hipSuccess;
  HOC_K_SWITCH(K, HOC_GEO_SWITCH(geo, hipLaunchKernelGGL((k_rhs<KK, GG>), dim3(fine_blocks(KK, N)), dim3(kFineThreads), 0,
                                                         s, N, T, G, omega, bcpsi, bs, part)));
  return hipGetLastError();
}

hipError_t launch_velocity(int K, int geo, int N, const Tab& T, const Geo& G, const BCDev& B, const double* psi,
                           double* vel, double* U, double* tru, double inv_dt_re, const InstDev& I, hipStream_t s,
                           int nbatch, const VelBatch& vb) {
  if (N == 0 || nbatch == 0) return hipSuccess;
  if (nbatch > 1 && vel) return hipErrorInvalidValue;  // a batch has no Cartesian velocity
  HOC_K_SWITCH(K, HOC_GEO_SWITCH(geo, hipLaunchKernelGGL((k_velocity<KK, GG>), dim3(fine_blocks(KK, N), nbatch),
                                                         dim3(kFineThreads), 0, s, N, T, G, B, psi, vel, U, tru,
                                                         inv_dt_re, I, vb)));
  return hipGetLastError();
}

hipError_t launch_stage(int K, int geo, int adv, int N, const Tab& T, const Geo& G, const BCDev& B,
                        const double* omega, const double* U, const double* tru, double re_inv, double dt,
                        const InstDev& I, const StageOut& so, hipStream_t s, int mode) {
  if (N == 0) return hipSuccess;
  // omega is read at neighbours while other elements are written
  if (omega == so.k || omega == so.next || (so.final_mode && omega == so.base)) return hipErrorInvalidValue;
#define HOC_STAGE(A, M)                                                                                               \
  HOC_K_SWITCH(K, HOC_GEO_SWITCH(geo, hipLaunchKernelGGL((k_stage<KK, A, GG, M>),                                      \
                                                         dim3(fine_blocks(KK, N), M == 2 ? so.nbatch : 1),            \
                                                         dim3(kFineThreads), 0, s, N, T, G, B, omega, U, tru, re_inv, \
                                                         dt, I, so)))
  if (adv == 1 && mode == 0) { HOC_STAGE(1, 0); }
  else if (adv == 2 && mode == 0) { HOC_STAGE(2, 0); }
  else if (adv == 1 && mode == 1) { HOC_STAGE(1, 1); }
  else if (adv == 1 && mode == 2) { HOC_STAGE(1, 2); }
  else return hipErrorInvalidValue;
#undef HOC_STAGE
  return hipGetLastError();
}

}  // namespace hoc
