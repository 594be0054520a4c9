// hoc_poisson.hip - the fine-level Poisson operator and smoother for gfx950.
//
// The operator is the second-order FR operator of src/HO_2D.cpp:1533-1804 (the diffusion term of
// :2666-2831 with zero boundary values), applied matrix-free.
//
// Mapping: K lanes per element, fine_epw(K) elements per wavefront.  Lane k of an element works on
// its row k (the xi line) and its column k (the eta line); rows become columns through a tile in
// LDS that only its own wavefront touches, so no barrier separates the two halves.  On each of the
// four faces lane k owns face point k, whose neighbour data is one line of the neighbour element
// (value and inward derivative at the shared face), read straight from the field.  That read
// comes from the L2 (the neighbour's line is in use by a nearby wavefront), where face traces
// stored by the kernel before cost 640 bytes of HBM traffic per element and application against
// the field's own 200 (K = 5, FP64); it also frees each application from a trace kernel.
//
// The smoother is the block Jacobi of the elements' own diagonal blocks, B, used as a damped
// Richardson step; a V-cycle takes degree-d Chebyshev polynomials in B As as d such steps with the
// roots as dampings.  A block of constant orthogonal metrics is W (x) a X + c Y (x) W with the
// one-dimensional line operators X, Y, so B = (S (x) S) (a lam_i + c lam_j)^-1 (S (x) S)^T with
// the generalised eigenvectors S of (X, W): 4 K^3 operations and no stored inverse (fast
// diagonalisation, R. E. Lynch, J. R. Rice and D. H. Thomas, Numer. Math. 6 (1964) 185-199).  S
// depends on what the two ends of the line are (interior, Dirichlet, Neumann: 9 tables); elsewhere
// a and c are the element's mean metrics.
#include "hoc_poisson.hpp"

#include "hoc_rowlane.hpp"
#include "hoc_status.hpp"

namespace hoc {

namespace {

// Even and odd parts of a line, and back.
template <int K, class R>
__device__ __forceinline__ void split(const R (&u)[K], R (&e)[3], R (&o)[3]) {
#pragma unroll
  for (int i = 0; i < K / 2; ++i) {
    e[i] = u[i] + u[K - 1 - i];
    o[i] = u[i] - u[K - 1 - i];
  }
  if (K & 1) e[K / 2] = u[K / 2];
}
template <int K, class R>
__device__ __forceinline__ void join(const R (&e)[3], const R (&o)[3], R (&u)[K]) {
#pragma unroll
  for (int i = 0; i < K / 2; ++i) {
    u[i] = e[i] + o[i];
    u[K - 1 - i] = e[i] - o[i];
  }
  if (K & 1) u[K / 2] = e[K / 2];
}

// 1 / x for the smoother's scales, x > 0 and normal: the hardware estimate and two Newton steps (to
// within an ulp or two; the quotient's exact rounding takes twice the instructions).
__device__ __forceinline__ double recip(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(fma(-x, r, 1.), r, r);
  return fma(fma(-x, r, 1.), r, r);
}
__device__ __forceinline__ float recip(float x) {
  const float r = __builtin_amdgcn_rcpf(x);
  return fmaf(fmaf(-x, r, 1.f), r, r);
}

// One face point of a lane: the neighbour line's value v and inward derivative g at the shared
// face; own and neighbour weights of the common flux (1/2, 1/2 inside; 1, 0 Dirichlet; 0, 0
// Neumann), and what the common value minus the own value is.
template <class R>
struct Face {
  R v = 0, g = 0;   // neighbour trace
  R an = 0;         // neighbour's normal metric
  int nb = -1;      // neighbour, or -1 - edge
  int fn = 0;       // its face
  int kk = 0;       // its point on that face
  bool neu = false;
};

// As u on the lane's row (without the weights -w_k w_i).  u: rows; uc: columns.  CONS: in conservation
// form (see line_cons); without it, the form for the V-cycle on elements with constant orthogonal metrics.
template <int K, int GEO, bool CONS, class R>
struct Op {
  // Common value minus own value at the two ends of a line, from the traces (value b., inward derivative
  // g.), and the common fluxes along it.
  static __device__ __forceinline__ void ends(const FineTab<R>& T, R a, R bl, R bu, R gl, R gu, const Face<R>& L,
                                              const Face<R>& U, R& dl, R& du, R& fl, R& fu) {
    dl = R(0.5) * (L.v - bl);
    du = R(0.5) * (U.v - bu);
    if (L.nb < 0) dl = L.neu ? gl * T.ig0 : -bl;
    if (U.nb < 0) du = U.neu ? gu * T.ig0 : -bu;
    const R tl = (gl - dl * T.g0) * a, tu = (gu - du * T.g0) * a;  // own inward fluxes
    fl = R(0.5) * (tl - (L.g + dl * T.g0) * L.an);
    fu = R(0.5) * ((U.g + du * T.g0) * U.an - tu);
    if (L.nb < 0) fl = L.neu ? R(0) : tl;
    if (U.nb < 0) fu = U.neu ? R(0) : -tu;
  }

  // One line of an element with constant orthogonal metrics: out = (a u'' + corrections) with the
  // two faces L (lower) and U (upper).  This is the operator whose solution is reported: the derivative of
  // the corrected derivative, so that the rounding of the tables enters through the flux and sums to
  // nothing over an element, and both sides' traces by the same sums, so that their difference has none.
  // With the second derivative as one table (line) a constant has a source of eps rho(A), of one sign in
  // every element; error of a solve whose solution is known: 3.0e-11 at 101 x 101, K = 6, 1.8e-11 at
  // 127 x 127, K = 5, 7.2e-11 at 256 x 256, K = 5; this way 3.4e-16, 9.3e-15 and 1.9e-14.
  static __device__ __forceinline__ void line_cons(const FineTab<R>& T, R a, const R (&u)[K], const Face<R>& L,
                                                   const Face<R>& U, R (&out)[K]) {
    constexpr int HE = (K + 1) / 2, HO = K / 2;
    R bl = 0, bu = 0, gl = 0, gu = 0, dl, du, fl, fu;
#pragma unroll
    for (int m = 0; m < K; ++m) {
      bl += u[m] * T.lv[m];
      gl += u[m] * T.ld[m];
      bu += u[K - 1 - m] * T.lv[m];
      gu += u[K - 1 - m] * T.ld[m];
    }
    ends(T, a, bl, bu, gl, gu, L, U, dl, du, fl, fu);
    R e[3], o[3];
    split<K>(u, e, o);
    const R se = dl - du, so = dl + du;
    // the flux's even and odd parts, from the odd and even parts of u
    R fe[3], fo[3];
#pragma unroll
    for (int i = 0; i < HE; ++i) {
      R t = se * T.gdE[i];
#pragma unroll
      for (int d = 0; d < HO; ++d) t += o[d] * T.DO[d][i];
      fe[i] = (2 * i + 1 == K ? a : R(2) * a) * t;
    }
#pragma unroll
    for (int i = 0; i < HO; ++i) {
      R t = so * T.gdO[i];
#pragma unroll
      for (int d = 0; d < HE; ++d) t += e[d] * T.DE[d][i];
      fo[i] = R(2) * a * t;
    }
    R ve = 0, vo = 0;  // its value at the lower end
#pragma unroll
    for (int i = 0; i < HE; ++i) ve += fe[i] * T.lvE[i];
#pragma unroll
    for (int i = 0; i < HO; ++i) vo += fo[i] * T.lvO[i];
    fl -= ve + vo;
    fu -= ve - vo;
    const R ce = fl - fu, co = fl + fu;
    R re[3], ro[3];
#pragma unroll
    for (int i = 0; i < HE; ++i) {
      R t = ce * T.gdE[i];
#pragma unroll
      for (int d = 0; d < HO; ++d) t += fo[d] * T.DO[d][i];
      re[i] = t;
    }
#pragma unroll
    for (int i = 0; i < HO; ++i) {
      R t = co * T.gdO[i];
#pragma unroll
      for (int d = 0; d < HE; ++d) t += fe[d] * T.DE[d][i];
      ro[i] = t;
    }
    join<K>(re, ro, out);
  }

  // The same for the V-cycle, a preconditioner whose rounding the iterations take up: half the products,
  // with the second derivative as one table.
  static __device__ __forceinline__ void line(const FineTab<R>& T, R a, const R (&u)[K], const Face<R>& L,
                                              const Face<R>& U, R (&out)[K]) {
    constexpr int HE = (K + 1) / 2, HO = K / 2;
    R e[3], o[3];
    split<K>(u, e, o);
    R ve = 0, vo = 0, ge = 0, go = 0;
#pragma unroll
    for (int i = 0; i < HE; ++i) { ve += e[i] * T.lvE[i]; ge += e[i] * T.ldE[i]; }
#pragma unroll
    for (int i = 0; i < HO; ++i) { vo += o[i] * T.lvO[i]; go += o[i] * T.ldO[i]; }
    const R bl = ve + vo, bu = ve - vo, gl = ge + go, gu = ge - go;
    R dl, du, fl, fu;
    ends(T, a, bl, bu, gl, gu, L, U, dl, du, fl, fu);
    fl -= a * (gl + dl * T.m0 - du * T.m1);
    fu -= a * (dl * T.m1 - gu - du * T.m0);
    const R se = a * (dl + du), so = a * (dl - du), ce = fl - fu, co = fl + fu;
    R re[3], ro[3];
#pragma unroll
    for (int i = 0; i < HE; ++i) {
      R t = 0;
#pragma unroll
      for (int d = 0; d < HE; ++d) t += e[d] * T.DDE[d][i];
      re[i] = a * t + (se * T.DgE[i] + ce * T.gdE[i]);
    }
#pragma unroll
    for (int i = 0; i < HO; ++i) {
      R t = 0;
#pragma unroll
      for (int d = 0; d < HO; ++d) t += o[d] * T.DDO[d][i];
      ro[i] = a * t + (so * T.DgO[i] + co * T.gdO[i]);
    }
    join<K>(re, ro, out);
  }

  static __device__ __forceinline__ void apply(const FineTab<R>& T, const FineGeo<R>& G, int el, int k, R* t, R* tf,
                                               const R (&u)[K], const R (&uc)[K], const Face<R> (&F)[4],
                                               R (&out)[K]) {
    if constexpr (GEO == GEO_ORTHO) {
      const R a = G.ac[(size_t)el * 2], c = G.ac[(size_t)el * 2 + 1];
      R oc[K], orw[K];
      if constexpr (CONS) {
        line_cons(T, c, uc, F[2], F[3], oc);
        line_cons(T, a, u, F[0], F[1], out);
      } else {
        line(T, c, uc, F[2], F[3], oc);
        line(T, a, u, F[0], F[1], out);
      }
      cols_to_rows<K>(t, k, oc, orw);
#pragma unroll
      for (int i = 0; i < K; ++i) out[i] += orw[i];
      return;
    } else {
      // common values: interior average, 0 on Dirichlet faces; Neumann faces from the K x K system
      // (src/HO_2D.cpp:2872-2927) solved at setup
      R bv[4], gi[4], cv[4], cg[4];
      for (int f = 0; f < 4; ++f) { bv[f] = 0; gi[f] = 0; }
#pragma unroll
      for (int m = 0; m < K; ++m) {
        bv[0] += u[m] * T.lv[m];
        gi[0] += u[m] * T.ld[m];
        bv[1] += u[K - 1 - m] * T.lv[m];
        gi[1] += u[K - 1 - m] * T.ld[m];
        bv[2] += uc[m] * T.lv[m];
        gi[2] += uc[m] * T.ld[m];
        bv[3] += uc[K - 1 - m] * T.lv[m];
        gi[3] += uc[K - 1 - m] * T.ld[m];
      }
      wave_fence();
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        cv[f] = F[f].nb >= 0 ? R(0.5) * (bv[f] + F[f].v) : R(0);
        tf[f * K + k] = F[f].nb < 0 && F[f].neu ? bv[f] + gi[f] * T.ig0 : cv[f];
      }
      wave_fence();
      R Dk[K];  // column k of the derivative matrix
#pragma unroll
      for (int d = 0; d < K; ++d) {
        R v = T.D[d][0];
#pragma unroll
        for (int i = 1; i < K; ++i) v = k == i ? T.D[d][i] : v;
        Dk[d] = v;
      }
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const R so = (f & 1) ? R(1) : R(-1);
        if (F[f].nb < 0 && F[f].neu) {
          const R* q = G.qn + ((size_t)(-1 - F[f].nb) * K + k) * K;
          R s = 0;
#pragma unroll
          for (int m = 0; m < K; ++m) s += q[m] * tf[f * K + m];
          cv[f] = s;
          cg[f] = 0;
          continue;
        }
        R cr = 0;
#pragma unroll
        for (int d = 0; d < K; ++d) cr += tf[f * K + d] * Dk[d];
        R fa, fb;
        if (GEO == GEO_AFFINE) {
          fa = G.gface[((size_t)el * 4 + f) * 2];
          fb = G.gface[((size_t)el * 4 + f) * 2 + 1];
        } else {
          fa = G.fa[((size_t)el * 4 + f) * K + k];
          fb = G.fb[((size_t)el * 4 + f) * K + k];
        }
        const R own = -so * (gi[f] - (cv[f] - bv[f]) * T.g0) * fa;
        if (F[f].nb < 0) {
          cg[f] = own;  // zero common value: no tangential part
        } else {
          const int fn = F[f].fn;
          R fan = F[f].an, fbn;
          if (GEO == GEO_AFFINE) fbn = G.gface[((size_t)F[f].nb * 4 + fn) * 2 + 1];
          else fbn = G.fb[((size_t)F[f].nb * 4 + fn) * K + F[f].kk];
          const bool rev = (f + fn - f / 2 - fn / 2 + 1) & 1;
          const R sg = (((f + fn) & 1) ? R(1) : R(-1)) * (rev ? R(-1) : R(1));
          cg[f] = R(0.5) * (own + so * (F[f].g - (cv[f] - F[f].v) * T.g0) * fan - cr * (fb + sg * fbn));
        }
      }
      // corrected contravariant gradient, its corrected divergence (src/HO_2D.cpp:2771-2816)
      R dx[K], de[K], der[K];
      const R d0 = cv[0] - bv[0], d1 = cv[1] - bv[1], d2 = cv[2] - bv[2], d3 = cv[3] - bv[3];
#pragma unroll
      for (int i = 0; i < K; ++i) {
        R s = 0, s2 = 0;
#pragma unroll
        for (int d = 0; d < K; ++d) {
          s += u[d] * T.D[d][i];
          s2 += uc[d] * T.D[d][i];
        }
        dx[i] = s + d0 * T.gd[i] - d1 * T.gd[K - 1 - i];
        de[i] = s2 + d2 * T.gd[i] - d3 * T.gd[K - 1 - i];
      }
      cols_to_rows<K>(t, k, de, der);
      R ft[K], gt[K], gtc[K];
      if (GEO == GEO_AFFINE) {
        const R a = G.gel[(size_t)el * 3], b = G.gel[(size_t)el * 3 + 1], c = G.gel[(size_t)el * 3 + 2];
#pragma unroll
        for (int i = 0; i < K; ++i) {
          ft[i] = dx[i] * a - der[i] * b;
          gt[i] = der[i] * c - dx[i] * b;
        }
      } else {
        R ga[K], gb[K], gc[K];
        const size_t q = ((size_t)el * K + k) * K;
        load_row<K>(G.Ga + q, ga);
        load_row<K>(G.Gb + q, gb);
        load_row<K>(G.Gc + q, gc);
#pragma unroll
        for (int i = 0; i < K; ++i) {
          ft[i] = dx[i] * ga[i] - der[i] * gb[i];
          gt[i] = der[i] * gc[i] - dx[i] * gb[i];
        }
      }
      rows_to_cols<K>(t, k, gt, gtc);
      R c0 = cg[0], c1 = cg[1], c2 = cg[2], c3 = cg[3];
#pragma unroll
      for (int m = 0; m < K; ++m) {
        c0 -= ft[m] * T.lv[m];
        c1 -= ft[K - 1 - m] * T.lv[m];
        c2 -= gtc[m] * T.lv[m];
        c3 -= gtc[K - 1 - m] * T.lv[m];
      }
      R oc[K], orw[K];
#pragma unroll
      for (int i = 0; i < K; ++i) {
        R s = 0, s2 = 0;
#pragma unroll
        for (int d = 0; d < K; ++d) {
          s += ft[d] * T.D[d][i];
          s2 += gtc[d] * T.D[d][i];
        }
        out[i] = s + c0 * T.gd[i] - c1 * T.gd[K - 1 - i];
        oc[i] = s2 + c2 * T.gd[i] - c3 * T.gd[K - 1 - i];
      }
      cols_to_rows<K>(t, k, oc, orw);
#pragma unroll
      for (int i = 0; i < K; ++i) out[i] += orw[i];
    }
  }
};

// r <- B r (rows): the element blocks' inverse by fast diagonalisation.  lamk: T.lam of the lane.
template <int K, class R>
__device__ __forceinline__ void block_inverse(const FineTab<R>& T, const FineGeo<R>& G, int el, int k, R lamk, R* t,
                                              R (&r)[K]) {
  const R a = G.ac[(size_t)el * 2], c = G.ac[(size_t)el * 2 + 1];
  const int ft = G.ftype[el];
  R s[K], q[K];
  if (__all(ft == 0)) {  // every element of the wavefront interior: even and odd eigenvectors
    constexpr int HE = (K + 1) / 2, HO = K / 2;
    R e[3], o[3];
    auto forward = [&](const R (&in)[K], R (&out)[K]) {
      split<K>(in, e, o);
#pragma unroll
      for (int b = 0; b < HE; ++b) {
        R v = 0;
#pragma unroll
        for (int i = 0; i < HE; ++i) v += T.SE[i][b] * e[i];
        out[b] = v;
      }
#pragma unroll
      for (int b = 0; b < HO; ++b) {
        R v = 0;
#pragma unroll
        for (int i = 0; i < HO; ++i) v += T.SO[i][b] * o[i];
        out[HE + b] = v;
      }
    };
    auto backward = [&](const R (&in)[K], R (&out)[K]) {
#pragma unroll
      for (int i = 0; i < HE; ++i) {
        R v = 0;
#pragma unroll
        for (int b = 0; b < HE; ++b) v += T.SE[i][b] * in[b];
        e[i] = v;
      }
#pragma unroll
      for (int i = 0; i < HO; ++i) {
        R v = 0;
#pragma unroll
        for (int b = 0; b < HO; ++b) v += T.SO[i][b] * in[HE + b];
        o[i] = v;
      }
      join<K>(e, o, out);
    };
    forward(r, s);
    rows_to_cols<K>(t, k, s, q);
    const R al = a * lamk;
    forward(q, s);
#pragma unroll
    for (int b = 0; b < K; ++b) s[b] *= recip(al + c * T.lam[b]);
    backward(s, q);
    cols_to_rows<K>(t, k, q, s);
    backward(s, r);
    return;
  }
  const R* fx = G.fdm + (ft & 15) * (K + K * K);
  const R* fy = G.fdm + (ft >> 4) * (K + K * K);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    R v = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) v += fx[K + j * K + i] * r[j];
    s[i] = v;
  }
  rows_to_cols<K>(t, k, s, q);
  const R al = a * fx[k];
#pragma unroll
  for (int b = 0; b < K; ++b) {
    R v = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) v += fy[K + j * K + b] * q[j];
    s[b] = v * recip(al + c * fy[b]);
  }
#pragma unroll
  for (int j = 0; j < K; ++j) {
    R v = 0;
#pragma unroll
    for (int b = 0; b < K; ++b) v += fy[K + j * K + b] * s[b];
    q[j] = v;
  }
  cols_to_rows<K>(t, k, q, s);
#pragma unroll
  for (int i = 0; i < K; ++i) {
    R v = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) v += fx[K + i * K + j] * s[j];
    r[i] = v;
  }
}

// Block sums of two per-lane values; thread 0 writes them to part[blk] and part[nblk + blk].
__device__ __forceinline__ void block_part(double a, double b, double* __restrict__ part, int blk, int nblk) {
  __shared__ double sa[kFineThreads / 64], sb[kFineThreads / 64];
  a = wave_sum(a);
  b = wave_sum(b);
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sa[w] = a; sb[w] = b; }
  __syncthreads();
  if (threadIdx.x == 0) {
    part[blk] = sa[0] + sa[1] + sa[2] + sa[3];
    part[nblk + blk] = sb[0] + sb[1] + sb[2] + sb[3];
  }
}

// The sum of np partials, the same in every thread of every block.
__device__ __forceinline__ double sum_parts(const double* __restrict__ part, int np) {
  __shared__ double sp[kFineThreads / 64];
  double s = 0.;
#pragma unroll 4
  for (int i = threadIdx.x; i < np; i += kFineThreads) s += part[i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sp[threadIdx.x >> 6] = s;
  __syncthreads();
  return sp[0] + sp[1] + sp[2] + sp[3];
}

// Sum of a per-lane value over the K lanes of each element, into part[el]; through the LDS that the
// block has done with.
template <int K>
__device__ __forceinline__ void element_part(double a, double* lds, int wv, int le, int k, bool live,
                                             double* __restrict__ part, int el) {
  double* s = lds + (wv * Lay<K>::EPW + le) * K;
  __syncthreads();
  s[k] = a;
  wave_fence();
  if (k != 0 || !live) return;
  double r = 0.;
#pragma unroll
  for (int i = 0; i < K; ++i) r += s[i];
  part[el] = r;
}

// sums of the first and of the second halves of 2 np partials, for thread 0 of the block
__device__ __forceinline__ void sum_pairs(const double* __restrict__ part, int np, double& a, double& b) {
  __shared__ double sa[kFineThreads / 64], sb[kFineThreads / 64];
  a = b = 0.;
#pragma unroll 4
  for (int i = threadIdx.x; i < np; i += kFineThreads) {
    a += part[i];
    b += part[np + i];
  }
  a = wave_sum(a);
  b = wave_sum(b);
  if ((threadIdx.x & 63) == 0) { sa[threadIdx.x >> 6] = a; sb[threadIdx.x >> 6] = b; }
  __syncthreads();
  a = sa[0] + sa[1] + sa[2] + sa[3];
  b = sb[0] + sb[1] + sb[2] + sb[3];
}

// The end of the iteration before, in a block of its own (FineArgs::chk_part): a launch of one
// block would hold the stream for 4.4 us.  The kernel's other blocks may or may not see the flag
// that it clears: what they write is not used then.
template <class A>
__device__ void check_block(const A& a) {
  int* F = a.chk_F;
  double* S = a.scal;
  const bool init = a.chk_phase == PH_INIT;
  const bool live = init || solve_live(F);  // uniform over the block
  double u = 0., v = 0., bb = 0.;
  if (live) sum_pairs(a.chk_part, a.chk_np, u, v);
  if (a.chk_bb) bb = sum_parts(a.chk_bb, a.chk_nbb);
  if (threadIdx.x) return;
  const int maxit = a.chk_maxit >= 0 ? a.chk_maxit : F[F_MAXIT];
  if (init) {
    if (a.chk_bb) S[S_BB] = bb;
    init_phase(u, v, v > S[S_TOL2] * S[S_BB], S, F, maxit);
  } else if (live) {
    check_phase(a.chk_phase, u, v, S, F, maxit);
  } else {
    F[F_ACTIVE] = 0;
  }
  if (!a.chk_mirror) return;
  const int seq = take_seq(a.chk_seq, F);
  publish(a.chk_mirror, seq, F[F_ACTIVE] && likely_last(S), S, F);
}

template <int K, int GEO, int IN, int EPI, class R, class RZ>
__global__ __launch_bounds__(kFineThreads) void k_fine(FineTab<R> T, FineGeo<R> G, FineArgs<R> A) {
  constexpr bool CHK = IN == IN_X && EPI == EPI_SMOOTH;
  // the test goes first, so that it ends in the shadow of the others; eight blocks, so that these keep
  // their XCDs
  const int nchk = CHK && A.chk_part ? 8 : 0, nblk = (int)gridDim.x - nchk;
  if (CHK && (int)blockIdx.x < nchk) {
    if (blockIdx.x == 0) check_block(A);
    return;
  }
  constexpr int EPW = Lay<K>::EPW, ES = Lay<K>::ES;
  constexpr int FS = GEO == GEO_ORTHO ? 0 : 4 * K;  // face values of one element
  __shared__ __align__(16) R lds[(kFineThreads / 64) * (Lay<K>::TILE + EPW * FS)];
  const int blk = xcd_block(blockIdx.x - nchk, nblk);
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  constexpr int EPB = EPW * (kFineThreads / 64);
  const int le = lane < EPW * K ? lane / K : EPW - 1;
  const int k = lane < EPW * K ? lane - le * K : K - 1;
  const int el0 = blk * EPB + wv * EPW + le;
  const bool live = lane < EPW * K && el0 < G.N;
  // lanes past the mesh follow its last element in a slot of their own, and the lanes past the last
  // slot its last row: the same reads, so the same values in LDS; neither writes to memory
  const int el = min(el0, G.N - 1);
  const bool go = !A.active || A.active[F_ACTIVE];
  if (A.ran && (int)blockIdx.x == nchk && threadIdx.x == 0) *A.ran = go ? 1 : 0;  // timed launches: did it work?
  if (!go) return;
  if (G.iact) {  // a block inside one stopped ensemble instance
    const int i0 = G.inst[blk * EPB];
    if (i0 == G.inst[min((blk + 1) * EPB, G.N) - 1] && !G.iact[i0]) return;
  }
  R* t = lds + wv * (Lay<K>::TILE + EPW * FS) + le * ES;
  R* tf = lds + wv * (Lay<K>::TILE + EPW * FS) + Lay<K>::TILE + le * FS;
  const size_t row = ((size_t)el * K + k) * K;
  const R wk = G.lane[4 * k], xk = G.lane[4 * k + 1], lamk = G.lane[4 * k + 2];
  (void)wk;
  (void)xk;
  (void)lamk;

  const int4 nbr = *reinterpret_cast<const int4*>(G.nb + (size_t)el * 4);
  const int nbf = G.nbf[el];
  // every global read of the kernel, issued before the arithmetic
  R u[K], z[K], b[K];
  (void)z;
  // a solve's first direction is z: the old one, of another solve, is not read
  const bool first_dir = IN == IN_PUPD && A.active[F_ITER] == 0;
  if (!first_dir) load_row<K>(A.x + row, u);
  R beta = 0;
  if constexpr (IN == IN_PUPD) {
    load_row<K>(static_cast<const RZ*>(A.z) + row, z);
    if (!A.rz) beta = (R)(A.scal_idx >= 0 ? A.scal[A.scal_idx] : A.scal[G.inst[el]]);
  }
  if constexpr (EPI == EPI_RESID || EPI == EPI_SMOOTH || EPI == EPI_RESTRICT || EPI == EPI_DOTS) load_row<K>(A.b + row, b);
  R xo[4] = {0, 0, 0, 0};  // IN_PROL: own vertex values
  if constexpr (IN == IN_PROL) {
    const int4 v = *reinterpret_cast<const int4*>(G.ev + (size_t)el * 4);
    xo[0] = A.xc[v.x]; xo[1] = A.xc[v.y]; xo[2] = A.xc[v.z]; xo[3] = A.xc[v.w];
  }
  // The four neighbours' lines through the lane's face points, from the shared face inward: all
  // loads unconditional (a boundary face reads the element's own line and ignores it), so that
  // their latencies overlap.
  Face<R> F[4];
  const int nbs[4] = {nbr.x, nbr.y, nbr.z, nbr.w};
  R l[4][K], pl[IN == IN_PUPD ? 4 : 1][K], cn[IN == IN_PROL ? 4 : 1][4];
  (void)pl;
  (void)cn;
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    const bool in = nbs[f] >= 0;
    const int nb = in ? nbs[f] : el, fn = in ? (nbf >> (8 * f)) & 3 : f ^ 1;
    F[f].nb = nbs[f];
    const bool opp = __all(fn == (f ^ 1));
    const int kk = opp ? k : face_point<K>(f, fn, k);
    if constexpr (IN == IN_PUPD) {
      nbr_line<K>(static_cast<const RZ*>(A.z), nb, f, fn, kk, k, opp, l[f]);
      if (!first_dir) nbr_line<K>(A.x, nb, f, fn, kk, k, opp, pl[f]);
    } else {
      nbr_line<K>(A.x, nb, f, fn, kk, k, opp, l[f]);
    }
    F[f].fn = opp ? (f ^ 1) : fn;
    F[f].kk = kk;
    if constexpr (IN == IN_PROL) {
      // vertex values at the corners of the shared face (along its parameter) and of the opposite one
      const int4 vn = *reinterpret_cast<const int4*>(G.ev + (size_t)nb * 4);
      cn[f][0] = A.xc[fn == 0 || fn == 2 ? vn.x : fn == 1 ? vn.y : vn.w];
      cn[f][1] = A.xc[fn == 0 ? vn.w : fn == 2 ? vn.y : vn.z];
      cn[f][2] = A.xc[fn == 0 ? vn.y : fn == 2 ? vn.w : vn.x];
      cn[f][3] = A.xc[fn == 0 || fn == 2 ? vn.z : fn == 1 ? vn.w : vn.y];
    }
    if (GEO == GEO_ORTHO) F[f].an = G.ac[(size_t)nb * 2 + (fn >> 1)];
    else if (GEO == GEO_AFFINE) F[f].an = G.gface[((size_t)nb * 4 + fn) * 2];
    else F[f].an = G.fa[((size_t)nb * 4 + fn) * K + F[f].kk];
  }
  if constexpr (IN == IN_PUPD) {
    if (A.rz) {  // behind the loads: the sum takes longer than they do
      const double rz = sum_parts(A.rz, A.np), be = A.active[F_ITER] > 0 ? rz / A.scal[S_RZ] : 0.;
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        A.scal[S_RZN] = rz;
        A.scal[S_BETA] = be;
      }
      // breakdown (z = 0 or an indefinite preconditioner): PRE_XR sees it by S_RZN
      if (!(rz > 0.) || !isfinite(rz)) return;
      beta = (R)be;
    }
  }
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    if (nbs[f] < 0) F[f].neu = G.sw[-1 - nbs[f]] != 0;
    if constexpr (IN == IN_PUPD)
      if (!first_dir)
#pragma unroll
        for (int m = 0; m < K; ++m) l[f][m] += beta * pl[f][m];
    R v = 0, g = 0;
#pragma unroll
    for (int m = 0; m < K; ++m) {
      v += l[f][m] * T.lv[m];
      g += l[f][m] * T.ld[m];
    }
    if constexpr (IN == IN_PROL) {  // the neighbour's bilinear correction on that line
      const R sk = R(0.5) * (R(1) + G.lane[4 * F[f].kk + 1]);
      const R near = cn[f][0] + sk * (cn[f][1] - cn[f][0]), far = cn[f][2] + sk * (cn[f][3] - cn[f][2]);
      v += near;
      g += R(0.5) * (far - near);
    }
    F[f].v = v;
    F[f].g = g;
  }
  if constexpr (IN == IN_PUPD) {
    if (first_dir) {
#pragma unroll
      for (int i = 0; i < K; ++i) u[i] = z[i];
    } else {
#pragma unroll
      for (int i = 0; i < K; ++i) u[i] = z[i] + beta * u[i];
    }
    if (live) store_row<K>(A.pn + row, u);
  }
  if constexpr (IN == IN_PROL) {
    const R sy = R(0.5) * (R(1) + xk);
    const R wl = xo[0] + sy * (xo[3] - xo[0]), wu = xo[1] + sy * (xo[2] - xo[1]);
#pragma unroll
    for (int i = 0; i < K; ++i) u[i] += wl + R(0.5) * (R(1) + T.x[i]) * (wu - wl);
  }
  R uc[K], out[K];
  rows_to_cols<K>(t, k, u, uc);
  Op<K, GEO, EPI != EPI_SMOOTH && EPI != EPI_RESTRICT, R>::apply(T, G, el, k, t, tf, u, uc, F, out);
  double p0 = 0., p1 = 0.;
  if constexpr (EPI == EPI_PLAIN) {
    if (live) store_row<K>(A.y + row, out);
    return;
  }
#pragma unroll
  for (int i = 0; i < K; ++i) out[i] *= -(wk * T.w[i]);
  if constexpr (EPI == EPI_DOTS) {
#pragma unroll
    for (int i = 0; i < K; ++i) {
      p0 += (double)b[i] * (double)out[i];
      p1 += (double)out[i] * (double)out[i];
    }
    if (live) store_row<K>(A.y + row, out);
  } else if constexpr (EPI == EPI_STORE) {
#pragma unroll
    for (int i = 0; i < K; ++i) p0 += (double)u[i] * (double)out[i];
    if (live) store_row<K>(A.y + row, out);
  } else {
    R res[K];
#pragma unroll
    for (int i = 0; i < K; ++i) res[i] = b[i] - out[i];
    if constexpr (EPI == EPI_RESID) {
#pragma unroll
      for (int i = 0; i < K; ++i) {
        const double v = res[i], uw = v / ((double)wk * (double)T.w[i]);
        p0 += v * v;
        p1 += uw * uw;
      }
      if (live) store_row<K>(A.y + row, res);
    } else if constexpr (EPI == EPI_RESTRICT) {
      R s0 = 0, s1 = 0;  // the row's share of its west and east ends
#pragma unroll
      for (int i = 0; i < K; ++i) {
        s0 += R(0.5) * (R(1) - T.x[i]) * res[i];
        s1 += R(0.5) * (R(1) + T.x[i]) * res[i];
      }
      wave_fence();
      t[2 * k] = s0;
      t[2 * k + 1] = s1;
      wave_fence();
#pragma unroll
      for (int c = 0; c < (3 + K) / K; ++c) {
        const int a = k + c * K;
        if (a < 4) {
          const int east = a == 1 || a == 2, north = a >= 2;
          R s = 0;
#pragma unroll
          for (int j = 0; j < K; ++j) s += R(0.5) * (north ? R(1) + T.x[j] : R(1) - T.x[j]) * t[2 * j + east];
          if (live) A.y[(size_t)el * 4 + a] = s;
        }
      }
    } else {  // EPI_SMOOTH
      block_inverse<K>(T, G, el, k, lamk, t, res);
      const R om = (R)A.omega;
#pragma unroll
      for (int i = 0; i < K; ++i) u[i] += om * res[i];
      if (A.part || A.elpart) {
        double bd[K];
        if constexpr (sizeof(R) == 4) {
          load_row<K>(A.b64 + row, bd);
        } else {
#pragma unroll
          for (int i = 0; i < K; ++i) bd[i] = b[i];
        }
#pragma unroll
        for (int i = 0; i < K; ++i) p0 += bd[i] * (double)u[i];
      }
      if (live) store_row<K>(A.y + row, u);
    }
  }
  if (A.elpart) element_part<K>(p0, reinterpret_cast<double*>(lds), wv, le, k, live, A.elpart, el);
  if (A.part) {
    if (!live) p0 = p1 = 0.;
    block_part(p0, p1, A.part, blk, nblk);
  }
}

template <int K, int UPD, class R>
__global__ __launch_bounds__(kFineThreads) void k_pre(FineTab<R> T, FineGeo<R> G, PreArgs<R> A) {
  constexpr bool XR = UPD == PRE_XR;
  if (A.active && !A.active[F_ACTIVE]) return;
  constexpr int EPW = Lay<K>::EPW, ES = Lay<K>::ES, EPB = EPW * (kFineThreads / 64);
  __shared__ __align__(16) R lds[(kFineThreads / 64) * Lay<K>::TILE];
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (G.iact) {
    const int i0 = G.inst[blk * EPB];
    if (i0 == G.inst[min((blk + 1) * EPB, G.N) - 1] && !G.iact[i0]) return;
  }
  const int le = lane < EPW * K ? lane / K : EPW - 1;
  const int k = lane < EPW * K ? lane - le * K : K - 1;
  const int el0 = blk * EPB + wv * EPW + le;
  const bool live = lane < EPW * K && el0 < G.N;
  const int el = min(el0, G.N - 1);
  R* t = lds + wv * Lay<K>::TILE + le * ES;
  const size_t row = ((size_t)el * K + k) * K;
  double r[K];
  load_row<K>(A.r + row, r);
  double p0 = 0., p1 = 0.;
  if constexpr (XR) {
    double x[K], p[K], q[K];
    load_row<K>(A.q + row, q);
    load_row<K>(A.p + row, p);
    load_row<K>(A.x + row, x);
    double al;
    if (A.pq) {
      const double pq = sum_parts(A.pq, A.np), num = A.scal[A.num];
      al = num / pq;
      const bool first = blockIdx.x == 0 && threadIdx.x == 0;
      // the same in every wavefront of every block, as F_ACTIVE at entry is: none clears it here
      if (pq == 0. || (A.spd && !(pq > 0. && num > 0.)) || !isfinite(al)) {
        if (first) A.active[F_BREAK] = 1;
        return;
      }
      if (first) {
        A.scal[S_PQ] = pq;
        A.scal[S_ALPHA] = al;
        A.scal[A.keep] = num;
      }
    } else {
      al = A.scal_idx >= 0 ? A.scal[A.scal_idx] : A.scal[G.inst[el]];
    }
    if (al != 0.) {
#pragma unroll
      for (int i = 0; i < K; ++i) {
        x[i] += al * p[i];
        r[i] -= al * q[i];
      }
      if (live) {
        store_row<K>(A.x + row, x);
        store_row<K>(A.r + row, r);
      }
    }
    const double wk = A.iwl[k];
#pragma unroll
    for (int i = 0; i < K; ++i) {
      const double uw = r[i] * (wk * A.iw[i]);
      p0 += r[i] * r[i];
      p1 += uw * uw;
    }
  }
  if constexpr (UPD == PRE_BICGP) {
    double p[K], q[K];
    load_row<K>(A.q + row, q);
    load_row<K>(A.p + row, p);
    const double om = A.scal[S_OMEGA];
    double be;
    if (A.pq) {
      const double rho = sum_parts(A.pq, A.np);
      be = (rho / A.scal[S_RHO]) * (A.scal[S_ALPHA] / om);
      if (blockIdx.x == 0 && threadIdx.x == 0) {
        A.scal[S_RHON] = rho;
        A.scal[S_BETA] = be;
      }
    } else {
      be = A.scal[S_BETA];
    }
#pragma unroll
    for (int i = 0; i < K; ++i) r[i] += be * (p[i] - om * q[i]);
    if (live) store_row<K>(A.pw + row, r);
  }
  if constexpr (UPD == PRE_BICG0) {
    if (live) {
      store_row<K>(A.pw + row, r);
      store_row<K>(A.rh + row, r);
    }
  }
  R v[K];
#pragma unroll
  for (int i = 0; i < K; ++i) v[i] = (R)r[i];
  if constexpr (sizeof(R) == 4) {
    if (live) store_row<K>(A.r32 + row, v);
  }
  block_inverse<K>(T, G, el, k, G.lane[4 * k + 2], t, v);
  const R om = (R)A.omega;
#pragma unroll
  for (int i = 0; i < K; ++i) v[i] *= om;
  if (live) store_row<K>(A.z + row, v);
  if (XR && A.elpart) element_part<K>(p1, reinterpret_cast<double*>(lds), wv, le, k, live, A.elpart, el);
  if (XR && A.part) {
    if (!live) p0 = p1 = 0.;
    block_part(p0, p1, A.part, blk, gridDim.x);
  }
}

// Element rows over the lanes as in the kernels around it, so that its partial sums are as many.
template <int K>
__global__ __launch_bounds__(kFineThreads) void k_bicg_x(int N, BicgArgs A) {
  if (!A.active[F_ACTIVE]) return;
  constexpr int EPW = Lay<K>::EPW, EPB = EPW * (kFineThreads / 64);
  const int blk = xcd_block(blockIdx.x, gridDim.x);
  const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int le = min(lane / K, EPW - 1), k = lane - le * K, el0 = blk * EPB + wv * EPW + le;
  const bool live = k < K && el0 < N;
  const size_t row = ((size_t)min(el0, N - 1) * K + min(k, K - 1)) * K;
  double x[K], r[K], sh[K], t[K], rh[K];
  load_row<K>(A.t + row, t);
  load_row<K>(A.r + row, r);
  load_row<K>(A.sh + row, sh);
  load_row<K>(A.x + row, x);
  load_row<K>(A.rh + row, rh);
  double om;
  if (A.ts) {
    double ts, tt;
    sum_pairs(A.ts, A.np, ts, tt);
    om = tt != 0. ? ts / tt : 0.;
    if (!isfinite(om)) om = 0.;
    if (blockIdx.x == 0 && threadIdx.x == 0) A.scal[S_OMEGA] = om;
  } else {
    om = A.scal[S_OMEGA];
  }
  double p0 = 0., p1 = 0.;
  const double wk = A.iwl[min(k, K - 1)];
#pragma unroll
  for (int i = 0; i < K; ++i) {
    x[i] += om * sh[i];
    r[i] -= om * t[i];
    const double uw = r[i] * (wk * A.iw[i]);
    p0 += rh[i] * r[i];
    p1 += uw * uw;
  }
  if (live) {
    store_row<K>(A.x + row, x);
    store_row<K>(A.r + row, r);
  } else {
    p0 = p1 = 0.;
  }
  block_part(p0, p1, A.part, blk, gridDim.x);
}

}  // namespace

#define HOC_K_SWITCH(KV, ...)                      \
  switch (KV) {                                    \
    case 2: { constexpr int KK = 2; __VA_ARGS__; } break; \
    case 3: { constexpr int KK = 3; __VA_ARGS__; } break; \
    case 4: { constexpr int KK = 4; __VA_ARGS__; } break; \
    case 5: { constexpr int KK = 5; __VA_ARGS__; } break; \
    case 6: { constexpr int KK = 6; __VA_ARGS__; } break; \
    default: return hipErrorInvalidValue;          \
  }
#define HOC_GEO_SWITCH(GV, ...)                             \
  switch (GV) {                                             \
    case GEO_ORTHO: { constexpr int GG = GEO_ORTHO; __VA_ARGS__; } break;   \
    case GEO_AFFINE: { constexpr int GG = GEO_AFFINE; __VA_ARGS__; } break; \
    case GEO_POINT: { constexpr int GG = GEO_POINT; __VA_ARGS__; } break;   \
    default: return hipErrorInvalidValue;                   \
  }

template <int K, int GEO, int IN, int EPI, class R, class RZ>
static void go_fine(const FineTab<R>& T, const FineGeo<R>& G, const FineArgs<R>& A, hipStream_t s) {
  hipLaunchKernelGGL((k_fine<K, GEO, IN, EPI, R, RZ>), dim3(fine_blocks(K, G.N) + (A.chk_part ? 8 : 0)),
                     dim3(kFineThreads), 0, s, T, G, A);
}

template <int K, int GEO, class R>
static hipError_t fine_kg(int in, int epi, const FineTab<R>& T, const FineGeo<R>& G, const FineArgs<R>& A,
                          hipStream_t s) {
  if (in == IN_X && epi == EPI_SMOOTH) go_fine<K, GEO, IN_X, EPI_SMOOTH, R, R>(T, G, A, s);
  else if (in == IN_PROL && epi == EPI_SMOOTH) go_fine<K, GEO, IN_PROL, EPI_SMOOTH, R, R>(T, G, A, s);
  else if (in == IN_X && epi == EPI_RESTRICT) go_fine<K, GEO, IN_X, EPI_RESTRICT, R, R>(T, G, A, s);
  else if constexpr (sizeof(R) == 8) {
    if (in == IN_X && epi == EPI_STORE) go_fine<K, GEO, IN_X, EPI_STORE, R, R>(T, G, A, s);
    else if (in == IN_X && epi == EPI_RESID) go_fine<K, GEO, IN_X, EPI_RESID, R, R>(T, G, A, s);
    else if (in == IN_X && epi == EPI_PLAIN) go_fine<K, GEO, IN_X, EPI_PLAIN, R, R>(T, G, A, s);
    else if (in == IN_X && epi == EPI_DOTS) go_fine<K, GEO, IN_X, EPI_DOTS, R, R>(T, G, A, s);
    else if (in == IN_PUPD && epi == EPI_STORE) go_fine<K, GEO, IN_PUPD, EPI_STORE, R, R>(T, G, A, s);
    else return hipErrorInvalidValue;
  } else return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_fine(int K, int geo, int in, int epi, const FineTab<double>& T, const FineGeo<double>& G,
                       const FineArgs<double>& A, hipStream_t s) {
  HOC_K_SWITCH(K, HOC_GEO_SWITCH(geo, return (fine_kg<KK, GG, double>(in, epi, T, G, A, s))));
  return hipErrorInvalidValue;
}
hipError_t launch_fine(int K, int geo, int in, int epi, const FineTab<float>& T, const FineGeo<float>& G,
                       const FineArgs<float>& A, hipStream_t s) {
  HOC_K_SWITCH(K, HOC_GEO_SWITCH(geo, return (fine_kg<KK, GG, float>(in, epi, T, G, A, s))));
  return hipErrorInvalidValue;
}
hipError_t launch_fine_pupd_f32z(int K, int geo, const FineTab<double>& T, const FineGeo<double>& G,
                                 const FineArgs<double>& A, hipStream_t s) {
  HOC_K_SWITCH(K, HOC_GEO_SWITCH(geo, (go_fine<KK, GG, IN_PUPD, EPI_STORE, double, float>(T, G, A, s))));
  return hipGetLastError();
}

template <class R>
static hipError_t launch_pre_t(int K, const FineTab<R>& T, const FineGeo<R>& G, const PreArgs<R>& A, hipStream_t s) {
  HOC_K_SWITCH(K, {
    const dim3 grid(fine_blocks(KK, G.N)), block(kFineThreads);
    switch (A.up) {
      case PRE_NONE: hipLaunchKernelGGL((k_pre<KK, PRE_NONE, R>), grid, block, 0, s, T, G, A); break;
      case PRE_XR: hipLaunchKernelGGL((k_pre<KK, PRE_XR, R>), grid, block, 0, s, T, G, A); break;
      case PRE_BICGP: hipLaunchKernelGGL((k_pre<KK, PRE_BICGP, R>), grid, block, 0, s, T, G, A); break;
      case PRE_BICG0: hipLaunchKernelGGL((k_pre<KK, PRE_BICG0, R>), grid, block, 0, s, T, G, A); break;
      default: return hipErrorInvalidValue;
    }
  });
  return hipGetLastError();
}
hipError_t launch_pre(int K, const FineTab<double>& T, const FineGeo<double>& G, const PreArgs<double>& A,
                      hipStream_t s) {
  return launch_pre_t<double>(K, T, G, A, s);
}
hipError_t launch_pre(int K, const FineTab<float>& T, const FineGeo<float>& G, const PreArgs<float>& A,
                      hipStream_t s) {
  return launch_pre_t<float>(K, T, G, A, s);
}
hipError_t launch_bicg_x(int K, int N, const BicgArgs& A, hipStream_t s) {
  HOC_K_SWITCH(K, hipLaunchKernelGGL((k_bicg_x<KK>), dim3(fine_blocks(KK, N)), dim3(kFineThreads), 0, s, N, A));
  return hipGetLastError();
}

}  // namespace hoc
