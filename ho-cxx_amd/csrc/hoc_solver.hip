// hoc_solver.hip - device state, Poisson solver, RK driver and the C ABI (include/hoc.h).
//
// Per RK stage (src/HO_2D.cpp:1806-1839):
//   update_BCs(t)            k_update_bcs
//   solve_Poisson            k_rhs, then PCG or BiCGSTAB on As = -W A (W = Gauss weights
//                            w_i w_j, which makes As symmetric on affine meshes) with a
//                            V-cycle: matrix-free fine level + Chebyshev smoothing with the
//                            element blocks' inverse (degree by order and shape), continuous
//                            bilinear coarse space on the element corners (Ac = Pc^T As Pc
//                            assembled from probes of As), then Ruge-Stueben coarsening below
//   velocity, wall vorticity k_velocity
//   diffusion + advection    k_stage (fused with k = dt (adv + diff) and the RK update)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <thread>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <system_error>
#include <type_traits>
#include <vector>

#include "../../include/hoc.h"
#include "hoc_adj.hpp"
#include "hoc_dev.hpp"
#include "hoc_fr.hpp"
#include "hoc_host.hpp"
#include "hoc_la.hpp"
#include "hoc_out.hpp"
#include "hoc_poisson.hpp"

namespace hoc {

// The largest mesh hoc_apply_laplacian_device takes: face traces (n_elem * 8 * K doubles) of this
// many bytes, the entry point's documented limit.
constexpr size_t kNoAllocMaxTraceBytes = size_t(64) << 20;

// Fine-level state in working precision R: tables and metrics of the operator and its smoother,
// the Krylov and smoother vectors, and the V-cycle hierarchy.  FP64 (R = double) serves the Krylov
// method and setup probing; FP32 (R = float) is the mixed solve's V-cycle.
template <class R>
struct Prec {
  FineTab<R> T{};
  FineGeo<R> G{};
  DBuf<R> Ga, Gb, Gc, fa, fb, gel, gface;  // FP32 copies (unused for FP64)
  DBuf<R> ac, fdm, qn, lane;
  // PCG ping-pongs its direction between p and v; t: the smoother's second iterate
  DBuf<R> r, z, p, q, rh, v, ph, sh, t, ec, xc;
  DevVHierarchy<R> lv;  // Q1 vertex level and below
  int prof_off = 0;  // offset of this precision's entries in the live kernel profile
  // set only while the iterations of a batched ensemble PCG are queued: the instances' live flags;
  // fine-level blocks of a stopped instance then return at once.  They go with a launch's copy of G
  // (masked): G itself has none, so that an operator application beside or after a solve works on every
  // instance.
  const int* iact = nullptr;
  FineGeo<R> masked() const {
    FineGeo<R> g = G;
    g.iact = iact;
    return g;
  }
  // vectors of the Krylov method (krylov) and of the V-cycle alone (the FP32 state)
  void alloc_vectors(size_t D, int N, bool krylov) {
    for (auto* f : {&r, &z, &t}) f->alloc(D);
    for (auto* f : {&p, &q, &rh, &v, &ph, &sh}) f->alloc(krylov ? D : 0);
    ec.alloc((size_t)N * 4 + 1);  // and a zero for the gather's padding (setup)
  }
};

// Large results to the caller's memory.  A caller's array is usually fresh, so that the copy's time is
// that of its page faults, taken by one thread (52 MB: 3.5 to 5 ms, against 1.8 ms the other way).
// Here the device writes chunks to a ring of pinned slots and a few threads, which live for the call,
// move them on and take the faults.  Used from kMin bytes on, where starting the threads (0.1 ms) pays, and
// for memory that the runtime does not know: into pinned memory the device writes by itself (52 MB:
// 0.93 ms, through the ring 1.73).
class HostCopy {
 public:
  static constexpr size_t kMin = size_t(8) << 20;

  static bool takes(const void* dst, size_t bytes) {
    if (bytes < kMin) return false;
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, dst) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
    (void)hipGetLastError();  // not known to the runtime
    return true;
  }
  ~HostCopy() {
    for (auto& e : ev_)
      if (e) (void)hipEventDestroy(e);
    if (pin_) (void)hipHostFree(pin_);
  }
  // false: no events, pinned memory or threads to be had, and nothing copied
  bool d2h(int device, hipStream_t s, char* dst, const char* src, size_t bytes) {
    if (!ring()) return false;
    const size_t n = (bytes + kChunk - 1) / kChunk;
    std::atomic<size_t> issued{0};
    std::atomic<int> err{hipSuccess};
    std::vector<std::atomic<bool>> done(n);
    for (auto& d : done) d = false;
    // thread t moves the chunks t, t + kThreads, ..; chunk c is in slot c % kSlots
    auto move = [&](size_t t) {
      (void)hipSetDevice(device);
      for (size_t c = t; c < n; c += kThreads) {
        while (issued.load(std::memory_order_acquire) <= c)
          if (err.load() != hipSuccess) return;
          else std::this_thread::yield();
        const hipError_t e = hipEventSynchronize(ev_[c % kSlots]);
        if (e != hipSuccess) { err = e; return; }
        const size_t o = c * kChunk;
        std::memcpy(dst + o, pin_ + (c % kSlots) * kChunk, std::min(kChunk, bytes - o));
        done[c].store(true, std::memory_order_release);
      }
    };
    std::vector<std::thread> th;
    struct Join {
      std::vector<std::thread>& t;
      std::atomic<int>& err;
      bool ok = false;
      ~Join() {  // an exception of this thread ends the others' waits
        if (!ok) err = hipErrorUnknown;
        for (auto& x : t)
          if (x.joinable()) x.join();
      }
    } join{th, err};
    try {
      for (size_t t = 0; t < kThreads; ++t) th.emplace_back(move, t);
    } catch (const std::system_error&) {
      return false;
    }
    for (size_t c = 0; c < n && err.load() == hipSuccess; ++c) {
      if (c >= kSlots)
        while (!done[c - kSlots].load(std::memory_order_acquire) && err.load() == hipSuccess) std::this_thread::yield();
      const size_t o = c * kChunk;
      HIPCHK(hipMemcpyAsync(pin_ + (c % kSlots) * kChunk, src + o, std::min(kChunk, bytes - o), hipMemcpyDeviceToHost, s));
      HIPCHK(hipEventRecord(ev_[c % kSlots], s));
      issued.store(c + 1, std::memory_order_release);
    }
    join.ok = true;
    for (auto& x : th) x.join();
    HIPCHK(static_cast<hipError_t>(err.load()));
    return true;
  }

 private:
  static constexpr size_t kChunk = size_t(1) << 20, kSlots = 16, kThreads = 4;
  // The events and then the slots; what a failed call has made, the next one keeps.
  bool ring() {
    for (auto& e : ev_)
      if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        e = nullptr;
        return false;
      }
    if (!pin_ && hipHostMalloc(reinterpret_cast<void**>(&pin_), kSlots * kChunk) != hipSuccess) {
      (void)hipGetLastError();
      pin_ = nullptr;
      return false;
    }
    return true;
  }
  char* pin_ = nullptr;
  hipEvent_t ev_[kSlots] = {};
};

constexpr int kMaxCheb = 8;

struct Solver {
  hoc_config cfg{};
  int device = 0;
  hipStream_t stream = nullptr;
  HostCopy host_copy;
  std::string err;

  // host
  Mesh mesh;
  bool mesh_loaded = false, ready = false;
  Tables tab;
  Geometry geo;
  BCs bch;
  int K = 0, K2 = 0, N = 0, E = 0;
  size_t D = 0;
  double time = 0., re_inv = 0.;
  Tab T{};
  VecArgs VA{};
  DBuf<double> d_iw;    // 1/w_k
  DBuf<double> d_winv;  // 1/(w_j w_i), the inverse quadrature weights VA.winv points at
  bool mixed = false;

  // device: geometry and connectivity
  DBuf<double> d_jac, d_xxi, d_xeta, d_yxi, d_yeta, d_Ga, d_Gb, d_Gc, d_fa, d_fb, d_fA, d_fjac, d_fAn;
  DBuf<int32_t> d_nb;
  DBuf<int8_t> d_nbf, d_swpsi, d_swdiff, d_noslip;
  DBuf<double> d_esign, d_gel, d_gface, d_gjm;
  Geo G{};
  // boundary values
  DBuf<double> b_psi, b_diff, b_nvel, b_pvel, b_vj, b_vort, b_adv;
  DBuf<double> b_psi0, b_psi_r, b_diff0, b_diff_r, b_nvel0, b_nvel_r, b_pvel0, b_pvel_r;
  BCDev B{};
  // fields
  DBuf<double> w, psi, vel, U, k1, k2, k3, k4, vort, vort2, kscratch, bs;
  DBuf<double> tru;      // normal traces of U
  DBuf<double> d_dcol, d_wrow;
  // Poisson solver: FP64 state (the Krylov method, the initial residual, probing) and FP32
  // state (the mixed-precision V-cycle); S/F = scalars and flags of the Krylov solve.
  Prec<double> P64;
  Prec<float> P32;
  DBuf<double> part, part2, S;  // part2: p.q partials, and ||b||^2's before the first residual
  DBuf<int> F;
  // Krylov progress and results published by the end-of-iteration finalize kernel, in pinned coherent
  // host memory; the status' number counts iterations over the handle's lifetime (hoc_seq.hpp).
  MirrorState* mirror = nullptr;
  MirrorState* mirror_dev = nullptr;
  int seq_next = kSeqStart;
  int nparts = 0;
  int nv = 0;                             // Q1 coarse space: element-corner vertices
  DBuf<int32_t> d_ev, d_vinc, d_voff;     // element -> 4 vertices; vertex -> (element*4+corner), gather_pack
  Corners corners{};
  // Chebyshev smoother of degree cheb_m in B As (B: the element blocks' inverse) as damped
  // Richardson steps x += cheb_w[k] B (r - As x)
  int cheb_m = 2;
  // Lower end of the smoothing interval over 1.1 lambda_max(B As).
  double cheb_lo = .1;
  // Degree and interval by order and shape of the elements: what the bilinear functions leave to the
  // smoother reaches down to a part of the spectrum that shrinks with the order and, far more, with the
  // elements' aspect ratio, where three steps down to 1/20 (order 6: 0.06) save a third of the iterations
  // for 4 of about 29 launches each.  ms per solve to 1e-11 (iterations), degree 2 at 1/10 | degree 2 at the
  // table's end (order 6: 0.08) | degree 3.  Squares: 48x48 K=2 0.52 (10) | 0.46 (9) | 0.63 (10), K=4 0.58 (11) | 0.56 (11) | 0.70 (11),
  // K=5 0.72 (12) | same | 0.77 (11), K=6 0.90 (15) | 0.92 (15) | 0.82 (11); jittered 128x128 K=5 1.98 (9)
  // | same | 2.19 (9).  Ratio 1.9, 128x16: K=2 0.53 | 0.44 | 0.64, K=3 0.65 | 0.67 | 0.64, K=4 0.83 | 0.93
  // | 0.74, K=5 1.12 | same | 0.98.  Ratio 3.8, 96x24: K=2 0.70 | 0.77 | 0.68, K=3 1.17 | 1.29 | 0.93, K=5
  // 2.2 (39) | same | 1.8 (27); jittered 2.97 (25) | same | 2.78 (17); ratio 7.5, 96x48: K=5 4.6 (78) |
  // same | 3.8 (53).  Degree 1 takes about twice the iterations of degree 2 throughout.
  // Further out degree 4 at 0.03 gains on degree 3: ratio 1.9, 128x16: K=3 0.64 -> 0.74, K=4 0.74 -> 0.79,
  // K=5 0.98 -> 0.92, K=6 1.36 -> 1.16; jittered K=5 1.38 -> 1.26, K=6 1.87 -> 1.53.  Ratio 2.5, 256x42: K=3
  // 0.96 -> 1.02, K=4 1.23 -> 1.19, K=5 1.75 -> 1.49, K=6 2.34 -> 2.03; jittered K=3 1.06 -> 1.21, K=4 1.59 ->
  // 1.60, K=5 2.22 -> 1.93, K=6 3.11 -> 2.52.  Ratio 3.8, 96x24: K=2 0.68 -> 0.72, K=3 0.93 -> 0.88, K=4 1.31
  // -> 1.17, K=5 1.82 -> 1.56, K=6 2.36 -> 2.04.
  void choose_smoother(double aspect) {
    static const double two[4] = {.15, .15, .12, .1};
    if (cfg.cheb_degree > 0) {
      cheb_m = cfg.cheb_degree;
      cheb_lo = .1;
    } else if (K > 2 && aspect > (K < 5 ? 3. : 1.8)) {
      cheb_m = 4;
      cheb_lo = .03;
    } else if (K == 6 || aspect > (K == 2 ? 3. : 1.5)) {
      cheb_m = 3;
      cheb_lo = K == 6 ? .06 : .05;
    } else {
      cheb_m = 2;
      cheb_lo = two[K - 2];
    }
    if (cfg.cheb_lower > 0.) cheb_lo = cfg.cheb_lower;
  }
  // Mean ratio of the elements' sides: the longer to the shorter pair's sum.
  double mean_aspect() const {
    double sum = 0.;
    for (int e = 0; e < N; ++e) {
      const int32_t* nd = &mesh.elem[(size_t)e * mesh.lnod * mesh.lnod];
      double side[4];
      for (int k = 0; k < 4; ++k) {
        const double *p = &mesh.xy[2 * (size_t)nd[k]], *q = &mesh.xy[2 * (size_t)nd[(k + 1) & 3]];
        side[k] = std::hypot(q[0] - p[0], q[1] - p[1]);
      }
      const double a = side[0] + side[2], b = side[1] + side[3];
      sum += std::max(a, b) / std::max(std::min(a, b), 1e-300);
    }
    return sum / N;
  }
  double cheb_w[kMaxCheb] = {0};
  double lam_max = 0.;
  int geo_kind = GEO_POINT;          // what the fine-level kernels are instantiated for
  DBuf<uint16_t> d_ftype;            // kinds of each element's line ends
  int krylov = HOC_KRYLOV_BICGSTAB;
  // live kernel timing (hoc_profile_*)
  struct Prof {
    bool on = false;
    int every = 1;      // record every every-th launch
    int64_t seen = 0;   // launches since profiling was turned on
    std::vector<hipEvent_t> e0, e1;
    std::vector<int> var;
    std::vector<double> nbytes;
    DBuf<int> ran;        // per recorded launch: 1 when it worked, 0 when it was a predicated no-op
    int64_t skipped = 0;  // recorded launches left out as no-ops
    int n = 0;
    double ms[HOC_PROF_VARIANTS] = {0};
    double bytes[HOC_PROF_VARIANTS] = {0};
    int64_t cnt[HOC_PROF_VARIANTS] = {0};
  } prof;
  // stats
  // hybrid operation (problem_type 11): values carried by boundary edges, outer-step window,
  // open-boundary edges in driver order, start/end values and blend targets
  std::vector<double> edge_nvel_in;
  std::vector<int8_t> edge_has_nvel;
  double time_start = 0., time_end = 0.;
  std::vector<int32_t> open_edges;
  std::vector<double> h_vn1, h_vp1, h_vw1;
  DBuf<uint8_t> d_hkind;
  DBuf<double> d_hinlet, d_vn0, d_vn1, d_vp0, d_vp1, d_vw0, d_vw1, d_hw0, d_hw1, d_hwgt;
  HybridDev H{};
  // ensembles: instance i owns elements [inst_off[i], inst_off[i+1]) and has its own Re, dt, clock
  int n_inst = 1;
  std::vector<int32_t> inst_off;
  std::vector<double> inst_re, inst_dt, inst_time;
  DBuf<int32_t> d_inst, d_einst, d_ioff;
  DBuf<double> d_ireinv, d_idt, d_iidr, d_iramp, d_inorm;
  InstDev I{};
  int last_iters = 0, last_outer = 0;
  double last_rel = 0.;
  int64_t total_iters = 0, n_solves = 0;
  double setup_seconds = 0.;

  ~Solver() {
    clear_graphs();
    for (auto e : prof.e0) (void)hipEventDestroy(e);
    for (auto e : prof.e1) (void)hipEventDestroy(e);
    if (mirror) (void)hipHostFree(mirror);
    if (stream) (void)hipStreamDestroy(stream);
  }

  // ---------------------------------------------------------------------------------------
  void setup() {
    auto t0 = std::chrono::steady_clock::now();
    HIPCHK(hipSetDevice(device));
    if (!stream) HIPCHK(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
    clear_graphs();
    connect(mesh);
    build_tables(cfg.K, mesh.lnod, tab);
    build_geometry(mesh, tab, geo);
    std::vector<int32_t> edge_inst;
    if (n_inst > 1 && (int)inst_off.size() == n_inst + 1) {
      edge_inst.resize(mesh.n_bedges);
      for (int e = 0; e < mesh.n_bedges; ++e)
        edge_inst[e] = (int32_t)(std::upper_bound(inst_off.begin(), inst_off.end(), mesh.be_elem[e]) - inst_off.begin() - 1);
    }
    build_bcs(mesh, tab, cfg.problem_type, bch, edge_inst, edge_nvel_in, edge_has_nvel);
    K = cfg.K; K2 = K * K; N = mesh.n_elem; E = mesh.n_bedges; D = (size_t)N * K2;
    re_inv = cfg.Re > 1.e-3 ? 1. / cfg.Re : -1.;  // src/HO_2D.cpp:255
    // tables
    std::memset(&T, 0, sizeof(T));
    for (int m = 0; m < K; ++m) {
      for (int s = 0; s < 2; ++s) {
        T.bb[m][s] = tab.bb[m][s]; T.bgb[m][s] = tab.bgb[m][s];
        T.rad[m][s] = tab.rad[m][s]; T.grad[m][s] = tab.grad[m][s];
      }
      for (int k = 0; k < K; ++k) T.D[m][k] = tab.D[m][k];
      T.w[m] = tab.wgt[m];
      T.x[m] = tab.sps[m];
    }
    T.gp[0] = tab.gprime[0]; T.gp[1] = tab.gprime[1];
    {
      std::vector<double> wi((size_t)K * K);
      for (int j = 0; j < K; ++j)
        for (int i = 0; i < K; ++i) wi[(size_t)j * K + i] = 1. / (tab.wgt[j] * tab.wgt[i]);
      d_winv.upload(wi);
      std::vector<double> iw(K);
      for (int k = 0; k < K; ++k) iw[k] = 1. / tab.wgt[k];
      d_iw.upload(iw);
      VA.K = K;
      VA.winv = d_winv.p;
    }
    for (size_t v = 0; v < D; ++v)
      if (!(geo.jac[v] > 0.)) throw StatusError(HOC_EMESH, "non-positive Jacobian at a solution point (element orientation must be CCW)");
    // geometry upload
    std::vector<double> Ga(D), Gb(D), Gc(D);
    for (size_t v = 0; v < D; ++v) {
      const double J = geo.jac[v];
      Ga[v] = (geo.xeta[v] * geo.xeta[v] + geo.yeta[v] * geo.yeta[v]) / J;
      Gb[v] = (geo.xxi[v] * geo.xeta[v] + geo.yxi[v] * geo.yeta[v]) / J;
      Gc[v] = (geo.xxi[v] * geo.xxi[v] + geo.yxi[v] * geo.yxi[v]) / J;
    }
    std::vector<double> fa(geo.fA.size()), fb(geo.fA.size());
    for (size_t i = 0; i < fa.size(); ++i) { fa[i] = geo.fA[i] / geo.fjac[i]; fb[i] = geo.fB[i] / geo.fjac[i]; }
    d_jac.upload(geo.jac); d_xxi.upload(geo.xxi); d_xeta.upload(geo.xeta); d_yxi.upload(geo.yxi); d_yeta.upload(geo.yeta);
    d_Ga.upload(Ga); d_Gb.upload(Gb); d_Gc.upload(Gc);
    d_fa.upload(fa); d_fb.upload(fb); d_fA.upload(geo.fA); d_fjac.upload(geo.fjac); d_fAn.upload(geo.fAn);
    d_nb.upload(mesh.nb);
    d_nbf.upload(mesh.nb_face);
    std::vector<int8_t> swp(E), swd(E), ns(E);
    for (int e = 0; e < E; ++e) { swp[e] = (int8_t)bch.sw_psi[e]; swd[e] = (int8_t)bch.sw_diff[e]; ns[e] = (int8_t)bch.no_slip_edge[e]; }
    d_swpsi.upload(swp); d_swdiff.upload(swd); d_noslip.upload(ns);
    d_esign.upload(bch.edge_sign);
    // affine fast path: every element's metrics constant over its sps and faces
    // (tolerances relative to each element's metric scale: rounding leaves ~1e-16 noise
    // in components that vanish on rectangles)
    bool affine = true;
    std::vector<double> gel((size_t)N * 3), gface((size_t)N * 8), gjm((size_t)N * 5);
    for (int e = 0; e < N && affine; ++e) {
      const size_t b0 = (size_t)e * K2;
      const double sc = std::max(std::fabs(Ga[b0]), std::fabs(Gc[b0]));
      gel[(size_t)e * 3] = Ga[b0]; gel[(size_t)e * 3 + 1] = Gb[b0]; gel[(size_t)e * 3 + 2] = Gc[b0];
      const double* jm[5] = {geo.xxi.data(), geo.xeta.data(), geo.yxi.data(), geo.yeta.data(), geo.jac.data()};
      const double sj = std::max(std::max(std::fabs(jm[0][b0]), std::fabs(jm[1][b0])),
                                 std::max(std::fabs(jm[2][b0]), std::fabs(jm[3][b0])));
      for (int c = 0; c < 5; ++c) gjm[(size_t)e * 5 + c] = jm[c][b0];
      for (int m = 1; m < K2 && affine; ++m) {
        affine = std::fabs(Ga[b0 + m] - Ga[b0]) <= 1e-12 * sc && std::fabs(Gb[b0 + m] - Gb[b0]) <= 1e-12 * sc &&
                 std::fabs(Gc[b0 + m] - Gc[b0]) <= 1e-12 * sc;
        for (int c = 0; c < 4 && affine; ++c) affine = std::fabs(jm[c][b0 + m] - jm[c][b0]) <= 1e-12 * sj;
        affine = affine && std::fabs(jm[4][b0 + m] - jm[4][b0]) <= 1e-12 * std::fabs(jm[4][b0]);
      }
      for (int f = 0; f < 4 && affine; ++f) {
        const size_t q0 = ((size_t)e * 4 + f) * K;
        const double fs = std::max(std::fabs(fa[q0]), 1e-300);
        gface[((size_t)e * 4 + f) * 2] = fa[q0]; gface[((size_t)e * 4 + f) * 2 + 1] = fb[q0];
        for (int k = 1; k < K && affine; ++k)
          affine = std::fabs(fa[q0 + k] - fa[q0]) <= 1e-12 * fs && std::fabs(fb[q0 + k] - fb[q0]) <= 1e-12 * fs;
      }
    }
    {
      std::vector<double> dc((size_t)K2), wr(tab.wgt, tab.wgt + K);
      for (int k = 0; k < K; ++k)
        for (int d = 0; d < K; ++d) dc[(size_t)k * K + d] = tab.D[d][k];
      d_dcol.upload(dc); d_wrow.upload(wr);
    }
    if (affine) { d_gel.upload(gel); d_gface.upload(gface); d_gjm.upload(gjm); }
    G = Geo{N, E, d_jac, d_xxi, d_xeta, d_yxi, d_yeta, d_Ga, d_Gb, d_Gc, d_fa, d_fb, d_fA, d_fjac, d_fAn,
            affine ? d_gel.p : nullptr, affine ? d_gface.p : nullptr, affine ? d_gjm.p : nullptr,
            d_nb, d_nbf, d_swpsi, d_swdiff, d_noslip, d_esign, nullptr, d_dcol, d_wrow, nullptr};
    setup_instances();
    setup_hybrid();
    P64.prof_off = 0;
    setup_fine(P64, affine, Ga, Gb, Gc, fa, fb, gel, gface);
    G.qn = P64.qn;
    const size_t EK = std::max<size_t>((size_t)E * K, 1);
    for (auto* b : {&b_psi, &b_diff, &b_nvel, &b_pvel, &b_vj, &b_vort, &b_adv}) b->alloc(EK);
    auto upl = [&](DBuf<double>& d, const std::vector<double>& h) { if (h.empty()) d.alloc(1); else d.upload(h); };
    upl(b_psi0, bch.psi); upl(b_psi_r, bch.psi_ramp); upl(b_diff0, bch.diff); upl(b_diff_r, bch.diff_ramp);
    upl(b_nvel0, bch.nvel); upl(b_nvel_r, bch.nvel_ramp); upl(b_pvel0, bch.pvel); upl(b_pvel_r, bch.pvel_ramp);
    B = BCDev{b_psi, b_diff, b_nvel, b_pvel, b_vj, b_vort, b_adv, b_psi0, b_psi_r, b_diff0, b_diff_r, b_nvel0, b_nvel_r, b_pvel0, b_pvel_r};
    // fields
    for (auto* f : {&w, &psi, &k1, &k2, &k3, &k4, &vort, &vort2, &kscratch, &bs}) f->alloc(D);
    vel.alloc(2 * D); U.alloc(2 * D);
    tru.alloc((size_t)N * 4 * K);
    mixed = cfg.precision == HOC_MIXED;
    P64.alloc_vectors(D, N, true);
    if (mixed) {  // FP32 tables and metrics of the V-cycle's fine operator
      P32.prof_off = HOC_PROF_VARIANTS / 2;
      setup_fine(P32, affine, Ga, Gb, Gc, fa, fb, gel, gface);
      P32.alloc_vectors(D, N, false);
    }
    nparts = std::max(fine_blocks(K, N), vec_grid(D));
    part.alloc(2 * (size_t)nparts);
    part2.alloc(2 * (size_t)nparts);
    S.alloc(S_COUNT); F.alloc(F_COUNT);
    if (!mirror) {
      HIPCHK(hipHostMalloc((void**)&mirror, sizeof(MirrorState), hipHostMallocCoherent | hipHostMallocMapped));
      __atomic_store_n(&mirror->status, status_word(seq_add(seq_next, -1), false, false), __ATOMIC_RELEASE);
      HIPCHK(hipHostGetDevicePointer((void**)&mirror_dev, mirror, 0));
    }
    build_hierarchy();
    // initial-guess history (its mode depends on the Krylov method chosen above)
    psi_prev.alloc(guess_mode() >= 2 ? D : 0);
    for (auto& b : rkS) b.alloc(guess_mode() >= 3 ? D : 0);
    for (auto& b : rkQ) b.alloc(guess_mode() >= 4 ? D : 0);
    proj_fwd.X.alloc(0); proj_fwd.AX.alloc(0); proj_fwd.m = 0;
    proj_adj.X.alloc(0); proj_adj.AX.alloc(0); proj_adj.m = 0;
    reset_adjoint();
    ensure_segments();  // (the timed iterations of an ensemble run its per-instance test)
    tune_launch_mode();
    invalidate_guess();
    const double tol2 = cfg.tol * cfg.tol;
    h2d(S.p + S_TOL2, &tol2, sizeof(double));
    time = 0.;
    smooth_ready = false;
    n_sp = 0;
    ready = true;
    HIPCHK(hipStreamSynchronize(stream));
    setup_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  }

  // Tables, metrics and connectivity of the fine-level kernels in the precision of P.
  template <class R>
  void setup_fine(Prec<R>& P, bool affine, const std::vector<double>& Ga, const std::vector<double>& Gb,
                  const std::vector<double>& Gc, const std::vector<double>& fa, const std::vector<double>& fb,
                  const std::vector<double>& gel, const std::vector<double>& gface) {
    FineTables ft;
    fine_tables(tab, ft);
    FineTab<R>& F = P.T;
    F = FineTab<R>{};
    const int HE = (K + 1) / 2, HO = K / 2;
    auto even = [&](const double* v, int i) { return 2 * i + 1 == K ? v[i] : 0.5 * (v[i] + v[K - 1 - i]); };
    auto odd = [&](const double* v, int i) { return 0.5 * (v[i] - v[K - 1 - i]); };
    double lv[kMaxK], ld[kMaxK], gd[kMaxK];
    for (int i = 0; i < K; ++i) {
      lv[i] = tab.bb[i][0];
      ld[i] = tab.bgb[i][0];
      gd[i] = tab.grad[i][0];
      F.lv[i] = (R)lv[i];
      F.ld[i] = (R)ld[i];
      F.gd[i] = (R)gd[i];
      F.w[i] = (R)tab.wgt[i];
      F.x[i] = (R)tab.sps[i];
      for (int j = 0; j < K; ++j) F.D[i][j] = (R)tab.D[i][j];
    }
    for (int i = 0; i < HE; ++i) {
      F.lvE[i] = (R)even(lv, i); F.ldE[i] = (R)even(ld, i); F.gdE[i] = (R)even(gd, i); F.DgE[i] = (R)even(ft.Dg, i);
      for (int d = 0; d < HE; ++d) F.DDE[d][i] = (R)even(ft.DD[d], i);
      for (int d = 0; d < HO; ++d) F.DO[d][i] = (R)even(tab.D[d], i);
    }
    for (int i = 0; i < HO; ++i) {
      F.lvO[i] = (R)odd(lv, i); F.ldO[i] = (R)odd(ld, i); F.gdO[i] = (R)odd(gd, i); F.DgO[i] = (R)odd(ft.Dg, i);
      for (int d = 0; d < HO; ++d) F.DDO[d][i] = (R)odd(ft.DD[d], i);
      for (int d = 0; d < HE; ++d) F.DE[d][i] = (R)odd(tab.D[d], i);
    }
    // interior eigenvectors, even ones first (the line operator commutes with the reflection)
    for (int q = 0, ne = 0, no = 0; q < K; ++q) {
      double v[kMaxK], se = 0., so = 0.;
      for (int i = 0; i < K; ++i) v[i] = ft.fdm[K + i * K + q];
      for (int i = 0; i < HO; ++i) { se += std::fabs(v[i] + v[K - 1 - i]); so += std::fabs(v[i] - v[K - 1 - i]); }
      if (se >= so && ne < HE) {
        F.lam[ne] = (R)ft.fdm[q];
        for (int i = 0; i < HE; ++i) F.SE[i][ne] = (R)even(v, i);
        ++ne;
      } else {
        F.lam[HE + no] = (R)ft.fdm[q];
        for (int i = 0; i < HO; ++i) F.SO[i][no] = (R)odd(v, i);
        ++no;
      }
    }
    F.m0 = (R)ft.m0; F.m1 = (R)ft.m1; F.g0 = (R)(-tab.gprime[0]); F.ig0 = (R)(-1. / tab.gprime[0]);
    std::vector<R> lane((size_t)4 * K, R(0));
    for (int k = 0; k < K; ++k) { lane[4 * k] = F.w[k]; lane[4 * k + 1] = F.x[k]; lane[4 * k + 2] = F.lam[k]; }
    P.lane.upload(lane);
    P.fdm.upload_as(ft.fdm);
    // orthogonal elements: the off-diagonal metric is rounding noise of the affine test's size
    bool ortho = affine;
    for (int e = 0; e < N && ortho; ++e) {
      const double* g = &gel[(size_t)e * 3];
      ortho = std::fabs(g[1]) <= 1e-12 * std::max(std::fabs(g[0]), std::fabs(g[2]));
    }
    geo_kind = ortho ? GEO_ORTHO : affine ? GEO_AFFINE : GEO_POINT;
    std::vector<double> ac((size_t)N * 2);
    for (int e = 0; e < N; ++e) {
      double a = 0., c = 0.;
      if (affine) {
        a = gel[(size_t)e * 3];
        c = gel[(size_t)e * 3 + 2];
      } else {
        for (int m = 0; m < K2; ++m) {  // quadrature means over the reference square
          const double ww = 0.25 * tab.wgt[m / K] * tab.wgt[m % K];
          a += ww * Ga[(size_t)e * K2 + m];
          c += ww * Gc[(size_t)e * K2 + m];
        }
      }
      ac[(size_t)e * 2] = a;
      ac[(size_t)e * 2 + 1] = c;
    }
    P.ac.upload_as(ac);
    if constexpr (std::is_same<R, double>::value) {
      std::vector<uint16_t> types(N);
      for (int e = 0; e < N; ++e) {
        int kind[4];
        for (int f = 0; f < 4; ++f) {
          const int nb = mesh.nb[(size_t)e * 4 + f];
          kind[f] = nb >= 0 ? 0 : bch.sw_psi[-1 - nb] ? 2 : 1;
        }
        types[e] = (uint16_t)((kind[0] * 3 + kind[1]) + 16 * (kind[2] * 3 + kind[3]));
      }
      d_ftype.upload(types);
    }
    // Neumann faces with tangential metrics: common values from the K x K system of
    // src/HO_2D.cpp:2872-2927, inverted here
    std::vector<double> qn;
    if (geo_kind != GEO_ORTHO) {
      qn.assign((size_t)std::max(E, 1) * K2, 0.);
      for (int e = 0; e < E; ++e) {
        if (!bch.sw_psi[e] && !bch.sw_diff[e]) continue;
        const int f = mesh.be_ijp[e];
        const size_t q = ((size_t)mesh.be_elem[e] * 4 + f) * K;
        const double gp = tab.gprime[f & 1];
        std::vector<double> M((size_t)K2), rhs((size_t)K2, 0.);
        for (int k = 0; k < K; ++k) {
          for (int i = 0; i < K; ++i) M[(size_t)k * K + i] = -geo.fB[q + k] * tab.D[i][k];
          M[(size_t)k * K + k] += geo.fA[q + k] * gp;
          rhs[(size_t)k * K + k] = geo.fA[q + k] * gp;
        }
        solve_dense(K, K, M.data(), rhs.data());
        std::copy(rhs.begin(), rhs.end(), qn.begin() + (size_t)e * K2);
      }
    }
    P.qn.upload_as(qn);
    FineGeo<R>& G2 = P.G;
    G2 = FineGeo<R>{};
    if constexpr (std::is_same<R, double>::value) {
      G2.gel = G.gel; G2.gface = G.gface;
      G2.Ga = G.Ga; G2.Gb = G.Gb; G2.Gc = G.Gc; G2.fa = G.fa; G2.fb = G.fb;
    } else if (affine) {
      P.gel.upload_as(gel); P.gface.upload_as(gface);
      G2.gel = P.gel; G2.gface = P.gface;
    } else {
      P.Ga.upload_as(Ga); P.Gb.upload_as(Gb); P.Gc.upload_as(Gc); P.fa.upload_as(fa); P.fb.upload_as(fb);
      G2.Ga = P.Ga; G2.Gb = P.Gb; G2.Gc = P.Gc; G2.fa = P.fa; G2.fb = P.fb;
    }
    G2.N = N;
    G2.ac = P.ac; G2.fdm = P.fdm; G2.lane = P.lane; G2.qn = P.qn; G2.ftype = d_ftype;
    G2.nb = d_nb; G2.nbf = reinterpret_cast<const int32_t*>(d_nbf.p); G2.sw = d_swpsi;
    G2.inst = G.inst;
  }

  // Fine-level operator launch in precision R, bracketed by events when profiling.
  template <class R>
  void fine(Prec<R>& P, int in, int epi, FineArgs<R> A) {
    const bool rec = prof.on && (prof.seen++ % prof.every) == 0;
    if (rec) HIPCHK(hipEventRecord(prof.e0[prof.n], stream));
    A.ran = rec ? prof.ran.p + prof.n : nullptr;
    HIPCHK(launch_fine(K, geo_kind, in, epi, P.T, P.masked(), A, stream));
    const double b64 = epi == EPI_SMOOTH && A.b64 && (A.part || A.elpart) ? 8. * D : 0.;  // FP32: b in FP64 too
    if (rec) prof_mark(P.prof_off + prof_variant(in, epi), lap_bytes(in, epi, (double)sizeof(R), (double)sizeof(R)) + b64);
  }
  void prof_mark(int variant, double bytes) {
    HIPCHK(hipEventRecord(prof.e1[prof.n], stream));
    prof.var[prof.n] = variant;
    prof.nbytes[prof.n] = bytes;
    if (++prof.n == (int)prof.e0.size()) prof_flush();
  }
  // Entry of the live kernel profile: apply, residual, smoothing step, first smoothing step after the
  // coarse correction, restriction.
  static int prof_variant(int in, int epi) {
    return epi == EPI_RESID ? 1 : epi == EPI_SMOOTH ? (in == IN_PROL ? 3 : 2) : epi == EPI_RESTRICT ? 4 : 0;
  }
  // p = z + beta p and q = As p in one launch (z in FP32 from the mixed-precision V-cycle).
  void direction_apply(Prec<double>& P, const void* z, bool z32, const double* p, double* pn, double* q,
                       double* scal, int scal_idx, const double* rz, double* partp,
                       int* active) {
    FineArgs<double> A;
    A.x = p; A.z = z; A.pn = pn; A.y = q; A.scal = scal; A.scal_idx = scal_idx; A.active = active;
    (P.iact ? A.elpart : A.part) = partp;
    A.rz = rz; A.np = rz ? fine_blocks(K, N) : 0;
    if (!z32) { fine(P, IN_PUPD, EPI_STORE, A); return; }
    const bool rec = prof.on && (prof.seen++ % prof.every) == 0;
    if (rec) HIPCHK(hipEventRecord(prof.e0[prof.n], stream));
    A.ran = rec ? prof.ran.p + prof.n : nullptr;
    HIPCHK(launch_fine_pupd_f32z(K, geo_kind, P.T, P.masked(), A, stream));
    if (rec) prof_mark(0, lap_bytes(IN_PUPD, EPI_STORE, 8., 4.));
  }
  // Only launches that worked count: a launch predicated off after convergence returns at once
  // and would book its algorithmic bytes against a near-zero duration.
  void prof_flush() {
    if (prof.n == 0) return;
    HIPCHK(hipEventSynchronize(prof.e1[prof.n - 1]));
    std::vector<int> ran(prof.n);
    HIPCHK(hipMemcpy(ran.data(), prof.ran.p, prof.n * sizeof(int), hipMemcpyDeviceToHost));
    for (int i = 0; i < prof.n; ++i) {
      if (!ran[i]) { ++prof.skipped; continue; }
      float ms = 0.f;
      HIPCHK(hipEventElapsedTime(&ms, prof.e0[i], prof.e1[i]));
      prof.ms[prof.var[i]] += ms;
      prof.cnt[prof.var[i]] += 1;
      prof.bytes[prof.var[i]] += prof.nbytes[i];
    }
    prof.n = 0;
  }
  // Algorithmic HBM bytes of one fine-operator launch for values of vb bytes (z: zb): every field,
  // metric and connectivity array once (the neighbours' lines are other wavefronts' own rows).
  double lap_bytes(int in, int epi, double vb = 8., double zb = 8.) const {
    const double vec = (double)N * K2 * vb;
    double b = vec + (double)N * (4 * 4 + 4);          // x; nb, nbf
    if (geo_kind == GEO_ORTHO) b += (double)N * 2 * vb;
    else if (geo_kind == GEO_AFFINE) b += (double)N * (3 + 8) * vb;
    else b += 3 * vec + (double)N * 4 * K * 2 * vb;
    if (in == IN_PUPD) b += vec + (double)N * K2 * zb; // z, p out
    if (in == IN_PROL) b += (double)N * 4 * 4 + (double)nv * vb;
    switch (epi) {
      case EPI_STORE: case EPI_PLAIN: b += vec; break;                      // y
      case EPI_RESID: case EPI_DOTS: b += 2 * vec; break;                   // b, y
      case EPI_SMOOTH: b += 2 * vec + (double)N * (geo_kind == GEO_ORTHO ? 2. : 2. + 2 * vb); break;  // b, y; types, scales
      case EPI_RESTRICT: b += vec + (double)N * 4 * vb; break;              // b, corner sums
    }
    return b;
  }

  // y = As x, and y = b - As x with the partial sums of its norms when partp is set (FP64).
  void apply_As(const double* x, double* y) {
    FineArgs<double> A;
    A.x = x; A.y = y;
    fine(P64, IN_X, EPI_STORE, A);
  }
  void residual_As(const double* x, const double* b, double* y, double* partp) {
    FineArgs<double> A;
    A.x = x; A.b = b; A.y = y; A.part = partp;
    fine(P64, IN_X, EPI_RESID, A);
  }

  // Stream-ordered copies that return when the data has arrived.
  void d2h(void* dst, const void* src, size_t bytes) {
    if (HostCopy::takes(dst, bytes) &&
        host_copy.d2h(device, stream, static_cast<char*>(dst), static_cast<const char*>(src), bytes))
      return;
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, stream));
    HIPCHK(hipStreamSynchronize(stream));
  }
  void h2d(void* dst, const void* src, size_t bytes) {
    HIPCHK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream));
    HIPCHK(hipStreamSynchronize(stream));
  }

  // Fine-level diagonal and the Q1 operator by probing, then the levels below it.
  void build_hierarchy() {
    std::vector<int32_t> col1, col2;
    const int nc1 = color_elements(mesh, 1, col1);
    const int nc2 = color_elements(mesh, 2, col2);
    DBuf<int32_t> dcol1, dcol2;
    dcol1.upload(col1); dcol2.upload(col2);
    for (int c = 0; c < nc1; ++c)
      for (int rs = 0; rs < K2; ++rs) {
        probe_set(stream, N, K2, dcol1, c, rs, P64.z);
        apply_As(P64.z, P64.q);
        probe_diag(stream, N, K2, dcol1, c, rs, P64.q, P64.t);
      }
    // Continuous bilinear coarse space on the element corners: Pc interpolates vertex values
    // to every element's solution points; Ac = Pc^T As Pc is assembled from probes of As.
    std::vector<int32_t> vid((size_t)mesh.n_nodes, -1), ev((size_t)N * 4);
    nv = 0;
    for (int e = 0; e < N; ++e)
      for (int a = 0; a < 4; ++a) {
        const int nd = mesh.elem[(size_t)e * mesh.lnod * mesh.lnod + a];
        if (vid[nd] < 0) vid[nd] = nv++;
        ev[(size_t)e * 4 + a] = vid[nd];
      }
    std::vector<int32_t> vptr(nv + 1, 0), vinc((size_t)N * 4);
    for (int32_t v : ev) vptr[v + 1]++;
    for (int v = 0; v < nv; ++v) vptr[v + 1] += vptr[v];
    {
      std::vector<int32_t> pos(vptr.begin(), vptr.end() - 1);
      for (int e = 0; e < N; ++e)
        for (int a = 0; a < 4; ++a) vinc[pos[ev[(size_t)e * 4 + a]]++] = e * 4 + a;
    }
    std::vector<int32_t> voff, inc;
    gather_pack(vptr, vinc, N * 4, corners.w, voff, inc);
    d_ev.upload(ev); d_vinc.upload(inc); d_voff.upload(voff);
    corners.off = d_voff;
    corners.inc = d_vinc;
    P64.G.ev = d_ev;
    P32.G.ev = d_ev;
    inst_coupled = false;  // an ensemble whose instances share a corner vertex
    if (n_inst > 1 && (int)inst_off.size() == n_inst + 1) {
      auto inst_of = [&](int e) { return std::upper_bound(inst_off.begin(), inst_off.end(), e) - inst_off.begin() - 1; };
      for (int v = 0; v < nv && !inst_coupled; ++v)
        for (int k = vptr[v] + 1; k < vptr[v + 1]; ++k)
          if (inst_of(vinc[k] / 4) != inst_of(vinc[vptr[v]] / 4)) { inst_coupled = true; break; }
    }
    std::vector<std::vector<std::pair<int, double>>> rows(nv);
    auto add = [&](int r, int c, double val) {
      for (auto& pr : rows[r]) if (pr.first == c) { pr.second += val; return; }
      rows[r].push_back({c, val});
    };
    DBuf<double> dM;
    dM.alloc((size_t)N * 16);
    std::vector<double> hM((size_t)N * 16);
    for (int c = 0; c < nc2; ++c) {
      HIPCHK(hipMemsetAsync(dM.p, 0, (size_t)N * 16 * sizeof(double), stream));
      for (int rs = 0; rs < K2; ++rs) {
        probe_set(stream, N, K2, dcol2, c, rs, P64.z);
        apply_As(P64.z, P64.q);
        q1_probe_accum(stream, N, K, T, rs, P64.q, dM);
      }
      d2h(hM.data(), dM.p, hM.size() * sizeof(double));
      for (int f = 0; f < N; ++f) {
        int e = -1;
        if (col2[f] == c) e = f;
        else
          for (int k = 0; k < 4; ++k) {
            const int nb = mesh.nb[(size_t)f * 4 + k];
            if (nb >= 0 && col2[nb] == c) { e = nb; break; }
          }
        if (e < 0) continue;
        for (int a = 0; a < 4; ++a)
          for (int b = 0; b < 4; ++b) {
            const double val = hM[(size_t)f * 16 + a * 4 + b];
            if (val != 0.) add(ev[(size_t)f * 4 + a], ev[(size_t)e * 4 + b], val);
          }
      }
    }
    CSR A1;
    A1.n = A1.m = nv;
    A1.ptr.assign(nv + 1, 0);
    for (int r0 = 0; r0 < nv; ++r0) {
      std::sort(rows[r0].begin(), rows[r0].end());
      for (auto& pr : rows[r0]) { A1.col.push_back(pr.first); A1.val.push_back(pr.second); }
      A1.ptr[r0 + 1] = (int)A1.col.size();
    }
    VHierarchy H;
    build_vhierarchy(A1, kCoarseDense, H);
    std::vector<double> ci;
    coarse_inverse(H.coarse, ci);
    if (mixed) { P32.lv.upload(H, ci); P32.xc.alloc(nv); }
    else { P64.lv.upload(H, ci); P64.xc.alloc(nv); }
    std::vector<double> hd(D);
    d2h(hd.data(), P64.t.p, D * sizeof(double));
    for (size_t i = 0; i < D; ++i)
      if (!(hd[i] > 0.)) throw StatusError(HOC_EINVAL, "Poisson operator has a non-positive diagonal entry");
    // Chebyshev interval from lambda_max(B As) by power iteration
    std::vector<double> hx(D);
    uint64_t st = 88172645463325252ull;
    for (size_t i = 0; i < D; ++i) { st ^= st << 13; st ^= st >> 7; st ^= st << 17; hx[i] = (double)(st % 2000001) / 1e6 - 1.; }
    h2d(P64.z.p, hx.data(), D * sizeof(double));
    double lam = 0.;
    const int vg = vec_grid(D);
    for (int it = 0; it < 30; ++it) {
      // z <- B As z / lam: the norm over one step estimates lambda_max (B As is similar to a
      // symmetric operator on affine meshes)
      apply_As(P64.z, P64.q);
      PreArgs<double> A = pre_args<double>(P64.q.p, P64.t.p, it > 0 ? 1. / lam : 1.);
      HIPCHK(launch_pre(K, P64.T, P64.G, A, stream));
      double nn[2] = {0., 0.};
      for (int k = 0; k < 2; ++k) {
        double* v = k == 0 ? P64.z.p : P64.t.p;
        vec<double>(stream, VOP_DOT2, VA, D, v, v, v, v, nullptr, nullptr, nullptr, part);
        finalize(stream, PH_BB, part, vg, S, F, 0);
        d2h(&nn[k], S.p + S_BB, sizeof(double));
      }
      lam = (it > 0 ? lam : 1.) * std::sqrt(nn[1] / nn[0]);
      std::swap(P64.z.p, P64.t.p);
    }
    lam_max = lam;
    // symmetry of As decides the Krylov method
    krylov = cfg.krylov;
    if (krylov == HOC_KRYLOV_AUTO) {
      std::vector<double> hx2(D), hAx(D), hAy(D);
      for (size_t i = 0; i < D; ++i) { st ^= st << 13; st ^= st >> 7; st ^= st << 17; hx2[i] = (double)(st % 2000001) / 1e6 - 1.; }
      for (size_t i = 0; i < D; ++i) { st ^= st << 13; st ^= st >> 7; st ^= st << 17; hx[i] = (double)(st % 2000001) / 1e6 - 1.; }
      h2d(P64.z.p, hx.data(), D * sizeof(double));
      apply_As(P64.z, P64.q);
      d2h(hAx.data(), P64.q.p, D * sizeof(double));
      h2d(P64.z.p, hx2.data(), D * sizeof(double));
      apply_As(P64.z, P64.q);
      d2h(hAy.data(), P64.q.p, D * sizeof(double));
      double a = 0., b = 0., na = 0., nb = 0.;
      for (size_t i = 0; i < D; ++i) { a += hx2[i] * hAx[i]; b += hx[i] * hAy[i]; na += std::fabs(hx2[i] * hAx[i]); nb += std::fabs(hx[i] * hAy[i]); }
      krylov = std::fabs(a - b) <= 1e-12 * std::max(na, nb) ? HOC_KRYLOV_PCG : HOC_KRYLOV_BICGSTAB;
    }
    choose_smoother(mean_aspect());
    const double lmax = 1.1 * lam, lmin = lmax * cheb_lo;
    const double theta = 0.5 * (lmax + lmin), delta = 0.5 * (lmax - lmin);
    // The dampings are the inverse roots of the Chebyshev polynomial on [lmin, lmax], large and small in
    // turn.
    std::vector<double> root(cheb_m);
    for (int k = 0; k < cheb_m; ++k) root[k] = theta + delta * std::cos(M_PI * (k + 0.5) / cheb_m);
    for (int k = 0; k < cheb_m; ++k) cheb_w[k] = 1. / ((k & 1) ? root[cheb_m - 1 - k / 2] : root[k / 2]);
    HIPCHK(hipMemsetAsync(P64.z.p, 0, D * sizeof(double), stream));
    HIPCHK(hipStreamSynchronize(stream));
  }

  // ---------------------------------------------------------------------------------------
  // Coarsening stops at this many unknowns, solved by their dense inverse: one launch in place of
  // two per level below.  1200, 1700 and 2450: cavity 127 x 127, K = 5 (coarsest 258, or 1213) 23.0, 22.0
  // and 21.9 ms a pass, step 384 x 64 (294, or 1209) 21.3, 20.3 and 20.5, cylinder 96 x 96 (288, or 1235)
  // 7.3, 7.0 and 7.2; where 2450 takes one of 2401 instead of 695 (hybrid 48 x 48) 5.0 ms stay 5.0 and
  // the setup doubles.
  static constexpr int kCoarseDense = 1700;
  // The dense inverse of the coarsest matrix, by the GPU's unpivoted elimination; a result that does
  // not reproduce a vector to 1e-6 is replaced by the host's pivoted one.
  void coarse_inverse(const CSR& A, std::vector<double>& ci) {
    const int n = A.n;
    ci.assign((size_t)n * n, 0.);
    if (n == 0) return;
    for (int i = 0; i < n; ++i)
      for (int j = A.ptr[i]; j < A.ptr[i + 1]; ++j) ci[(size_t)i * n + A.col[j]] += A.val[j];
    DBuf<double> d, wk;
    d.upload(ci);
    wk.alloc(dense_invert_work(n));
    dense_invert(stream, n, d, wk);
    HIPCHK(hipGetLastError());
    d2h(ci.data(), d.p, ci.size() * sizeof(double));
    std::vector<double> x(n), b(n, 0.);
    for (int i = 0; i < n; ++i) x[i] = 1. + std::sin(1.7 * i);
    for (int i = 0; i < n; ++i)
      for (int j = A.ptr[i]; j < A.ptr[i + 1]; ++j) b[i] += A.val[j] * x[A.col[j]];
    double e = 0., xx = 0.;
    for (int i = 0; i < n; ++i) {
      double y = 0.;
      for (int j = 0; j < n; ++j) y += ci[(size_t)i * n + j] * b[j];
      e += (y - x[i]) * (y - x[i]);
      xx += x[i] * x[i];
    }
    if (!(e <= 1e-12 * xx)) dense_inverse(A, ci);
  }

  // The first smoothing step of a V-cycle, z = omega B r (see PreArgs).
  template <class R>
  PreArgs<R> pre_args(const double* r, R* z, double omega) const {
    PreArgs<R> A;
    A.r = const_cast<double*>(r);  // written only with the PCG update in front of the step
    A.z = z;
    A.omega = omega;
    for (int k = 0; k < K; ++k) A.iw[k] = 1. / tab.wgt[k];
    A.iwl = d_iw;
    return A;
  }
  // The test of an iteration's end by the second smoothing step of the next V-cycle (FineArgs).
  struct Check {
    const double* part;
    int np, phase, maxit, seq;
    MirrorState* mirror;
    double* S;
    int* F;
    const double* bb;  // PH_INIT: partials of ||b||^2 (fine_blocks), or null
  };
  enum { WHOLE = 0, HEAD, REST };
  // The rest of the V-cycle for the residual rr after its first smoothing step has left the first
  // iterate in P.t: the iterate ping-pongs between P.t and zout and ends in zout; if partp != nullptr,
  // partials of r64.zout (r64: the residual in FP64) are left there, per element while an ensemble's masks
  // are set.  HEAD: the second smoothing step only; REST: what follows it.
  template <class R>
  void vcycle_rest(Prec<R>& P, const R* rr, const double* r64, R* zout, double* partp, int* Fp, int part_of = WHOLE,
                   const Check* chk = nullptr) {
    R *cur = P.t.p, *nxt = zout;
    FineArgs<R> A;
    A.b = rr;
    A.active = Fp;
    if constexpr (std::is_same<R, float>::value) A.b64 = r64;
    auto smooth = [&](int in, double omega, double* pp) {
      A.x = cur; A.y = nxt; A.omega = omega; (P.iact ? A.elpart : A.part) = pp;
      fine(P, in, EPI_SMOOTH, A);
      std::swap(cur, nxt);
    };
    for (int k = 1; k < cheb_m; ++k) {
      if (k == 1 && chk) {
        A.chk_part = chk->part; A.chk_np = chk->np; A.chk_phase = chk->phase; A.chk_maxit = chk->maxit;
        A.chk_seq = chk->seq; A.chk_mirror = chk->mirror; A.scal = chk->S; A.chk_F = chk->F;
        A.chk_bb = chk->bb; A.chk_nbb = chk->bb ? fine_blocks(K, N) : 0;
        if (chk->phase == PH_INIT) A.active = nullptr;  // the flags are of an earlier solve
      }
      if (k > 1 || part_of != REST) smooth(IN_X, cheb_w[k], nullptr);
      else std::swap(cur, nxt);
      A.chk_part = nullptr;
      A.active = Fp;
      if (part_of == HEAD) return;
    }
    // restrict the residual to the corner vertices
    A.x = cur; A.y = P.ec.p; A.part = nullptr;
    fine(P, IN_X, EPI_RESTRICT, A);
    if (P.lv.dense_only() && nv <= kDenseGather) {
      dense_gather<R>(stream, nv, P.lv.inv, corners, P.ec, P.xc.p, Fp);
    } else {
      q1_gather<R>(stream, nv, corners, P.ec, P.lv.rhs(), Fp);
      P.lv.cycle(stream, P.xc.p, Fp);
    }
    // prolongate and post-smooth, the dampings in reverse: the cycle stays symmetric
    A.xc = P.xc.p;
    for (int k = cheb_m - 1; k >= 0; --k)
      smooth(k == cheb_m - 1 ? IN_PROL : IN_X, cheb_w[k], k == 0 ? partp : nullptr);
  }

  // z = M r, begun by a first smoothing step (krylov_pre): the rest of the V-cycle in
  // its precision, for a mixed-precision handle with a promotion of z at the end.
  void precond_rest(const double* rin, double* zout, int* Fp, int part_of, const Check* chk) {
    if (mixed) {
      vcycle_rest(P32, (const float*)P32.r.p, rin, P32.z.p, nullptr, Fp, part_of, chk);
      if (part_of != HEAD) promote(stream, D, P32.z.p, zout, Fp);
    } else {
      vcycle_rest(P64, rin, rin, zout, nullptr, Fp, part_of, chk);
    }
  }

  // Wait, lag iterations behind (none when final_wait), until the finalize kernel of the
  // iteration numbered seq has published its status; returns false when the solve ended.
  // seq_first: the first iteration of this solve (no wait before it has run).  The wait spins
  // on the pinned word and checks the stream every 4096 reads, so an idle stream without the
  // expected status (or a device error) ends it with an error instead of a hang.
  bool poll(int seq, int seq_first, bool final_wait, int lag = 1, bool* near = nullptr) {
    const int target = final_wait ? seq : seq_add(seq, -lag);
    if (near) *near = false;
    if (!seq_reached(target, seq_first)) return true;
    for (unsigned spin = 1;; ++spin) {
      const uint32_t v = __atomic_load_n(&mirror->status, __ATOMIC_ACQUIRE);
      if (seq_reached(status_seq(v), target)) {
        if (near) *near = status_near(v);
        return status_active(v);
      }
      if ((spin & 4095) == 0) {
        const hipError_t q = hipStreamQuery(stream);
        if (q == hipSuccess) {
          const uint32_t v2 = __atomic_load_n(&mirror->status, __ATOMIC_ACQUIRE);
          if (seq_reached(status_seq(v2), target)) {
            if (near) *near = status_near(v2);
            return status_active(v2);
          }
          throw HipError("Krylov status of an iteration was not published");
        }
        if (q != hipErrorNotReady) HIPCHK(q);
      }
    }
  }

  // Preconditioned Krylov iterations on As x = r in precision R, from the state left by
  // PH_INIT in (Sp, Fp): r holds the residual of x.  PCG when As is symmetric, else
  // right-preconditioned BiCGSTAB.  Every kernel is predicated on Fp's active flag.
  // maxit bounds the host loop; maxit_dev is the device budget (< 0: Fp[F_MAXIT]).
  //
  // Launches.  An iteration is queued in two pieces, up to its test (krylov_iter) and the rest of the
  // next one's V-cycle (krylov_tail), and the host reads the status in between.  What bounds small
  // meshes is the chain of dependent launches, 5 to 6 us each: every vector update, dot product and
  // test rides on a kernel that needs its result or on the one that made its operands (32 x 32
  // elements, K = 4: 9 launches and 50.3 us a PCG iteration with the test and the vertices' gather as
  // launches of their own, now 7 and 42.0; BiCGSTAB on 384 x 64 elements, K = 5: 43 launches and 256 us,
  // now 33 and 213).
  // Direct mode launches the kernels, graph mode the pieces as captured hipGraphs (two for the
  // iteration, by which of the direction buffers is the old one), whose test takes its number from the
  // device counter F[F_SEQ].  The kernels and their order are the same, so both modes give the same
  // iterates; graphs pay where the host's launch cost exceeds the kernels' run time, and setup chooses
  // by timing both (launch_mode 0).
  static constexpr int kTuneIters = 8;
  struct KGraph {
    hipGraph_t g = nullptr;
    hipGraphExec_t e = nullptr;
    const void* key[6] = {nullptr, nullptr, nullptr, nullptr, nullptr, nullptr};
    int maxit = 0;
    int piece = 0;  // 0, 1: krylov_iter (odd 0, 1); 2: krylov_tail
  };
  std::vector<KGraph> kgraphs;
  bool use_graphs = false;
  double launch_tune_ratio = 0.;  // graph / direct time of the same iterations at setup (0: not timed)
  void clear_graphs() {
    for (auto& k : kgraphs) {
      if (k.e) (void)hipGraphExecDestroy(k.e);
      if (k.g) (void)hipGraphDestroy(k.g);
    }
    kgraphs.clear();
  }
  // Whether the blocks of the kernels sum the partials of the kernel before themselves: past
  // kInlineParts partials every block's sum costs more than the finalize launch that it saves.
  bool inline_sums() const { return fine_blocks(K, N) <= kInlineParts; }
  // Whether an iteration's test rides on the next smoothing step (512 x 512 elements, K = 5: 5462 pairs in
  // the shadow of a kernel of 45 us, 6.5 us as a launch).  BiCGSTAB's also gives the next beta, which the
  // kernel before that step needs: a launch where that kernel's blocks do not sum.
  bool inline_check() const { return cheb_m > 1 && !ens_pcg() && (krylov == HOC_KRYLOV_PCG || inline_sums()); }
  // The first smoothing step of a V-cycle behind a Krylov update.
  template <class Set>
  void krylov_pre(const double* r, Set&& set) {
    auto go = [&](auto& P) {
      using R = std::remove_reference_t<decltype(*P.t.p)>;
      PreArgs<R> A = pre_args<R>(r, P.t.p, cheb_w[0]);
      if constexpr (std::is_same<R, float>::value) A.r32 = P.r.p;
      set(A);
      HIPCHK(launch_pre(K, P.T, P.masked(), A, stream));
    };
    if (mixed) go(P32);
    else go(P64);
  }
  // Before the first iteration, from the residual r with its norms' partials in part: its V-cycle (an
  // iteration ends with the next one's), and the start of the solve's state where that is not a launch of
  // its own (outer_residual).  The first
  // direction needs no clearing, beta = 0 leaves the old one out.
  // pbb: partials of ||b||^2 for S[S_BB] (null: it is set).
  void krylov_begin(double* r, const double* pbb, double* Sp, int* Fp, int maxit) {
    krylov_pre(r, [&](auto& A) {
      if (krylov != HOC_KRYLOV_PCG) { A.up = PRE_BICG0; A.pw = P64.p; A.rh = P64.rh; }
      A.active = inline_check() ? nullptr : Fp;
    });
    const Check init{part.p, fine_blocks(K, N), PH_INIT, maxit, 0, nullptr, Sp, Fp, pbb};
    krylov_vcycle(r, Sp, Fp, maxit, WHOLE, inline_check() ? &init : nullptr);
  }
  // The V-cycle of the next iteration, or a part of it, after its first smoothing step.
  void krylov_vcycle(double* r, double* Sp, int* Fp, int maxit, int part_of, const Check* chk) {
    Prec<double>& P = P64;
    if (krylov != HOC_KRYLOV_PCG) {
      precond_rest(P.p.p, P.ph.p, Fp, part_of, chk);
      return;
    }
    if (ens_batched()) {
      EnsMask mask(*this);
      vcycle_pcg(r, ens_part.p, Fp, part_of, chk);
      ens_finalize(ENS_RZ, Sp, Fp, maxit);
      return;
    }
    // r.z from the V-cycle's last sweep; in mixed precision the direction update reads z in FP32
    vcycle_pcg(r, part.p, Fp, part_of, chk);
    if (part_of != HEAD && !inline_sums()) finalize(stream, PH_RZ, part, fine_blocks(K, N), Sp, Fp, maxit);
  }
  void vcycle_pcg(double* r, double* partp, int* Fp, int part_of, const Check* chk) {
    if (mixed) vcycle_rest(P32, (const float*)P32.r.p, r, P32.z.p, partp, Fp, part_of, chk);
    else vcycle_rest(P64, r, r, P64.z.p, partp, Fp, part_of, chk);
  }
  // One iteration up to its test and the publication of its status (seq >= 0: as seq; seq < 0: as the
  // next number of F[F_SEQ]); with inline_check() that takes the second smoothing step of the next
  // V-cycle along.  krylov_tail: the rest of that V-cycle.  odd: which of the two direction buffers of
  // PCG is the old one.
  void krylov_iter(double* x, double* r, double* Sp, int* Fp, int maxit, int seq, bool odd) {
    Prec<double>& P = P64;
    const int fb = fine_blocks(K, N);
    const bool inl = inline_sums(), ichk = inline_check();
    double* pold = odd ? P.v.p : P.p.p;
    double* pnew = odd ? P.p.p : P.v.p;
    if (ens_batched()) {
      ens_iter(x, r, pold, pnew, Sp, Fp, maxit, seq);
      return;
    }
    Check chk{part.p, fb, PH_UPD, maxit, seq, mirror_dev, Sp, Fp, nullptr};
    if (krylov == HOC_KRYLOV_PCG) {
      direction_apply(P, mixed ? (const void*)P32.z.p : P.z.p, mixed, pold, pnew, P.q.p, Sp, S_BETA,
                      inl ? part.p : nullptr, part2.p, Fp);
      if (!inl) finalize(stream, PH_PQ, part2, fb, Sp, Fp, maxit);
      krylov_pre(r, [&](auto& A) {
        A.up = PRE_XR; A.x = x; A.p = pnew; A.q = P.q; A.scal = Sp; A.scal_idx = S_ALPHA; A.part = part; A.active = Fp;
        if (inl) { A.pq = part2; A.np = fb; A.num = S_RZN; A.keep = S_RZ; }
      });
      if (ens_pcg()) {  // every instance against its own right-hand side
        seg_norm2(stream, pseg, VA, r, Fp, ens_part.p, ens_rr.p);
        finalize(stream, PH_UPD, part, fb, Sp, Fp, maxit, mirror_dev, seq, ens_rr.p, ens_bb.p, pseg.nseg);
      } else if (!ichk) {
        finalize(stream, PH_UPD, part, fb, Sp, Fp, maxit, mirror_dev, seq);
      }
    } else {
      // BiCGSTAB, right-preconditioned: v = As M p, alpha = rho / rh.v, s = r - alpha v, t = As M s,
      // omega = t.s / t.t; every vector update rides on the kernel that needs its result
      FineArgs<double> A;
      A.active = Fp;
      A.x = P.ph.p; A.y = P.v.p; A.b = P.rh.p; A.part = part2;
      fine(P, IN_X, EPI_DOTS, A);
      if (!inl) finalize(stream, PH_ALPHA, part2, fb, Sp, Fp, maxit);
      krylov_pre(r, [&](auto& B) {
        B.up = PRE_XR; B.x = x; B.p = P.ph; B.q = P.v; B.scal = Sp; B.scal_idx = S_ALPHA; B.part = part; B.active = Fp;
        B.spd = false;
        if (inl) { B.pq = part2; B.np = fb; B.num = S_RHON; B.keep = S_RHO; }
      });
      const Check half{part.p, fb, PH_BHALF, maxit, 0, nullptr, Sp, Fp, nullptr};
      if (!ichk) finalize(stream, PH_BHALF, part, fb, Sp, Fp, maxit);
      precond_rest(r, P.sh.p, Fp, WHOLE, ichk ? &half : nullptr);
      A.x = P.sh.p; A.y = P.q.p; A.b = r; A.part = part2;
      fine(P, IN_X, EPI_DOTS, A);
      if (!inl) finalize(stream, PH_OMEGA, part2, fb, Sp, Fp, maxit);
      BicgArgs B;
      B.x = x; B.r = r; B.sh = P.sh; B.t = P.q; B.rh = P.rh; B.scal = Sp; B.part = part; B.active = Fp;
      if (inl) { B.ts = part2; B.np = fb; }
      for (int k = 0; k < K; ++k) B.iw[k] = 1. / tab.wgt[k];
      B.iwl = d_iw;
      HIPCHK(launch_bicg_x(K, N, B, stream));
      if (!ichk) finalize(stream, PH_BNEXT, part, fb, Sp, Fp, maxit, mirror_dev, seq);
      chk.phase = PH_BNEXT;
      krylov_pre(r, [&](auto& C) {
        C.up = PRE_BICGP; C.p = P.p; C.pw = P.p; C.q = P.v; C.scal = Sp; C.active = Fp;
        if (ichk) { C.pq = part; C.np = fb; }  // else PH_BNEXT has left beta
      });
    }
    if (ichk) krylov_vcycle(r, Sp, Fp, maxit, HEAD, &chk);
  }
  void krylov_tail(double* r, double* Sp, int* Fp, int maxit) {
    krylov_vcycle(r, Sp, Fp, maxit, inline_check() ? REST : WHOLE, nullptr);
  }
  struct EnsMask {  // the masks hold for the launches in its scope only
    Solver& s;
    explicit EnsMask(Solver& so) : s(so) { s.P64.iact = s.P32.iact = s.ens_act.p; }
    ~EnsMask() { s.P64.iact = s.P32.iact = nullptr; }
  };
  // A phase of the batched ensemble PCG from the elements' sums in ens_part.  Up to kEnsInline elements the
  // phase's own block sums them, past that one block per instance does first (35152 elements, a pass of 12
  // solves: 18.4 ms without that launch, 17.7 with it).
  static constexpr int kEnsInline = 16384;
  void ens_finalize(int phase, double* Sp, int* Fp, int maxit, MirrorState* mir = nullptr, int seq = 0) {
    EnsKry E = ensk();
    if (phase == ENS_UPD) E.in = ens_rr.p;
    if (N > kEnsInline) {
      seg_sum(stream, pseg.nseg, d_ioff, ens_part, E.in, ens_act);
      E.part = nullptr;
    }
    finalize_ens(stream, phase, E, Sp, Fp, maxit, mir, seq);
  }
  // One iteration of the batched ensemble PCG (ens_batched): PCG with a step length and a
  // direction coefficient per instance (r_i.z_i, p_i.q_i and ||r_i|| by segment), each instance
  // stopping on its own test; while an instance is stopped, the fine-level kernels skip the
  // blocks that hold only its elements, and its x and r stay as they are.  The coarse levels run
  // over every instance: with no Q1 vertex shared between instances they stay block-diagonal.
  void ens_iter(double* x, double* r, const double* pold, double* pnew, double* Sp, int* Fp, int maxit, int seq) {
    EnsMask mask(*this);
    Prec<double>& P = P64;
    direction_apply(P, mixed ? (const void*)P32.z.p : P.z.p, mixed, pold, pnew, P.q.p, ens_beta.p, -1, nullptr,
                    ens_part.p, Fp);
    ens_finalize(ENS_PQ, Sp, Fp, maxit);
    krylov_pre(r, [&](auto& A) {
      A.up = PRE_XR; A.x = x; A.p = pnew; A.q = P.q; A.scal = ens_alpha; A.scal_idx = -1; A.active = Fp;
      A.elpart = ens_part;
    });
    // ||r_i||^2 into ens_rr, where a stopped instance keeps its last value (its r no longer changes)
    ens_finalize(ENS_UPD, Sp, Fp, maxit, mirror_dev, seq);
  }
  // The instantiated graph of a piece of an iteration on these buffers (captured on first use).
  hipGraphExec_t krylov_graph(double* x, double* r, double* Sp, int* Fp, int maxit, int piece) {
    const void* key[6] = {&P64, x, r, Sp, Fp, mixed ? (const void*)&P32 : nullptr};
    for (auto& k : kgraphs)
      if (k.maxit == maxit && k.piece == piece && std::equal(key, key + 6, k.key)) return k.e;
    KGraph kg;
    std::copy(key, key + 6, kg.key);
    kg.maxit = maxit;
    kg.piece = piece;
    HIPCHK(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    try {
      if (piece < 2) krylov_iter(x, r, Sp, Fp, maxit, -1, piece);
      else krylov_tail(r, Sp, Fp, maxit);
    } catch (...) {
      hipGraph_t g = nullptr;
      (void)hipStreamEndCapture(stream, &g);
      if (g) (void)hipGraphDestroy(g);
      throw;
    }
    HIPCHK(hipStreamEndCapture(stream, &kg.g));
    HIPCHK(hipGraphInstantiate(&kg.e, kg.g, nullptr, nullptr, 0));
    kgraphs.push_back(kg);
    return kg.e;
  }
  void krylov_solve(double* x, double* r, const double* pbb, double* Sp, int* Fp, int maxit_host, int maxit_dev) {
    const int maxit = maxit_dev;
    const int seq0 = seq_next;
    krylov_begin(r, pbb, Sp, Fp, maxit);
    const bool graphs = use_graphs && !prof.on;
    hipGraphExec_t ge[3] = {nullptr, nullptr, nullptr};
    if (graphs) {
      for (int k = 0; k < 3; ++k) ge[k] = krylov_graph(x, r, Sp, Fp, maxit, k);
      set_int(stream, Fp + F_SEQ, seq_add(seq_next, -1));
    }
    // The host runs ahead by an iteration up to its test: while it waits for the status of the one
    // before, the rest of a V-cycle and that iteration are queued.  Where that status says that the
    // iteration is likely the last (near), its own is waited for before the next V-cycle is queued,
    // which would run predicated off.
    for (int it = 0;; ++it) {
      const int seq = seq_next;
      seq_next = seq_add(seq_next, 1);
      if (graphs) HIPCHK(hipGraphLaunch(ge[it & 1], stream));
      else krylov_iter(x, r, Sp, Fp, maxit, seq, it & 1);
      bool near = false;
      if (!poll(seq, seq0, it > maxit_host + 2, 1, &near) || it > maxit_host + 4) break;
      // (before the first iteration there is no status to go by: as the solve before, which ended there)
      if ((near || (it == 0 && last_iters == 1)) && !poll(seq, seq0, true)) break;
      if (graphs) HIPCHK(hipGraphLaunch(ge[2], stream));
      else krylov_tail(r, Sp, Fp, maxit);
    }
  }

  // Launch mode (launch_mode 0): the same kTuneIters iterations of a solve on a random right-hand
  // side, queued directly and replayed from the captured graphs; graphs are used when they take under
  // 85% of the direct time.  The solve's state is reset afterwards.
  void tune_launch_mode() {
    clear_graphs();
    use_graphs = cfg.launch_mode == 2;
    launch_tune_ratio = 0.;
    if (cfg.launch_mode != 0) return;
    std::vector<double> hb(D);
    uint64_t st = 0x9E3779B97F4A7C15ull;
    for (size_t i = 0; i < D; ++i) { st ^= st << 13; st ^= st >> 7; st ^= st << 17; hb[i] = (double)(st % 2000001) / 1e6 - 1.; }
    h2d(bs.p, hb.data(), D * sizeof(double));
    const double sv[2] = {1., 0.};  // S_BB = 1, S_TOL2 = 0: every tuning iteration stays active
    h2d(S.p + S_BB, &sv[0], sizeof(double));
    h2d(S.p + S_TOL2, &sv[1], sizeof(double));
    const int maxit = std::max(cfg.maxiter, 2 * kTuneIters);
    auto run = [&](bool graph) {
      HIPCHK(hipMemsetAsync(psi.p, 0, D * sizeof(double), stream));
      outer_residual(nullptr);
      krylov_begin(P64.r.p, nullptr, S.p, F.p, maxit);
      hipGraphExec_t ge[3] = {nullptr, nullptr, nullptr};
      for (int k = 0; k < 3 && graph; ++k) ge[k] = krylov_graph(psi.p, P64.r.p, S.p, F.p, maxit, k);
      HIPCHK(hipStreamSynchronize(stream));
      const auto t0 = std::chrono::steady_clock::now();
      if (graph) set_int(stream, F.p + F_SEQ, seq_add(seq_next, -1));
      for (int i = 0; i < kTuneIters; ++i, seq_next = seq_add(seq_next, 1)) {
        if (graph) {
          HIPCHK(hipGraphLaunch(ge[i & 1], stream));
          HIPCHK(hipGraphLaunch(ge[2], stream));
        } else {
          krylov_iter(psi.p, P64.r.p, S.p, F.p, maxit, seq_next, i & 1);
          krylov_tail(P64.r.p, S.p, F.p, maxit);
        }
      }
      HIPCHK(hipStreamSynchronize(stream));
      return std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    };
    run(false);  // warm-up
    const double td = run(false);
    run(true);   // capture and warm-up
    const double tg = run(true);
    launch_tune_ratio = td > 0. ? tg / td : 0.;
    use_graphs = tg < 0.85 * td;
    HIPCHK(hipMemsetAsync(psi.p, 0, D * sizeof(double), stream));
    HIPCHK(hipMemsetAsync(bs.p, 0, D * sizeof(double), stream));
    HIPCHK(hipStreamSynchronize(stream));
  }

  // FP64 residual r = bs - As psi with the reference's unscaled norm, and the solve's
  // convergence state in (S, F).
  // pbb (may be null): fine_blocks(K, N) partials of ||b||^2 for S[S_BB].
  void outer_residual(const double* pbb) {
    const int lb = fine_blocks(K, N);
    residual_As(psi.p, bs.p, P64.r.p, part.p);
    if (ens_pcg()) {
      seg_norm2(stream, pseg, VA, P64.r.p, nullptr, ens_part.p, ens_rr.p);
      finalize(stream, PH_INIT, part, lb, S, F, cfg.maxiter, nullptr, 0, ens_rr.p, ens_bb.p, pseg.nseg, pbb,
               fine_blocks(K, N));
      if (ens_batched()) {
        EnsKry E = ensk();
        E.in = ens_rr.p;
        E.part = nullptr;
        finalize_ens(stream, ENS_INIT, E, S, F, cfg.maxiter);
      }
    } else if (!inline_check()) {
      finalize(stream, PH_INIT, part, lb, S, F, cfg.maxiter, nullptr, 0, nullptr, nullptr, 0, pbb, fine_blocks(K, N));
    }
  }

  // solve_Poisson (src/HO_2D.cpp:1841-1977) for omega at the current boundary values.
  //  FP64:  PCG/BiCGSTAB with the FP64 V-cycle on the scaled system, stopping on the
  //         reference's ||b - A psi|| <= tol ||b||.
  //  mixed: the same FP64 Krylov method, the same operator and the same stopping test, with
  //         the V-cycle in FP32 as its preconditioner: the residual is demoted at the cycle's
  //         entry and the cycle's output enters the FP64 direction update (PCG's reads it in FP32,
  //         BiCGSTAB's after a promotion, precond_rest).
  const double* rhs_bc = nullptr;  // boundary stream-function values of the next solve (null: b_psi)

  // Initial guess of the stage solves.  Mode 1: the previous solution, as the reference
  // (src/HO_2D.cpp:1949-1953).  Mode 2: psi is affine in omega and the RK stage inputs advance
  // smoothly in the stage time tau = steps + c, so the guess at tau is the linear extrapolation
  // psi_a + (tau - tau_a) / (tau_a - tau_b) (psi_a - psi_b) from the solutions at the last two
  // distinct stage times (the previous solution where tau = tau_a).  Only the iteration count
  // changes: every solve still stops on the same residual test.
  DBuf<double> psi_prev;        // psi_b
  double tau_a = 0., tau_b = 0.;
  int n_hist = 0;               // solutions in the history (0: psi is not a stage solution)
  int64_t step_count = 0;
  double stage_tau = std::nan("");  // stage time of the solve in progress (NaN: not a stage solve)
  // default: the projection (mode 5)
  int guess_mode() const { return cfg.psi_guess != 0 ? cfg.psi_guess : 5; }
  // Mode 3 (RK4): psi(omega_n + c k) = psi(omega_n) + c Psi(k) with Psi linear, so the stage
  // solutions S1..S4 of a step give Psi(k1) = 2 (S2 - S1), Psi(k2) = 2 (S3 - S1), Psi(k3) = S4 - S1,
  // and the next step's first solve is S1 + (Psi(k1) + 2 Psi(k2) + 2 Psi(k3) + Psi(k4)) / 6 with
  // Psi(k4) ~ Psi(k3): (-3 S1 + 2 S2 + 4 S3 + 3 S4) / 6.  Its solution T1 then gives Psi(k4) exactly,
  // and the second stage, T1 + Psi(k1') / 2 with Psi(k1') ~ Psi(k4): 4 T1 + S1 - S2 - 2 S3 - S4.
  // Stages 3 and 4 as in mode 2 (S2; 2 S3 - S1).  Other integrators use mode 2 under modes 3 and 4.
  DBuf<double> rkS[4];
  DBuf<double> rkQ[4];            // mode 4: Psi(k1..k4) of the step before S1..S4's
  int rk_stage = -1, rk_cur = 0;  // stage index of the RK4 solve in progress; stages of this step solved
  bool rk_full = false;           // S1..S4 hold a complete step
  bool rk_qok = false;            // rkQ holds a complete step (mode 4)
  // Mode 4: as mode 3, with each predicted Psi(k) corrected by the same stage difference one step
  // earlier (Q = Psi(k) of that step): stage 1 Psi(k4) ~ Psi(k3) + Q4 - Q3; stage 2
  // Psi(k1') ~ Psi(k4) + Q1 - Q4; stage 3 Psi(k2') ~ Psi(k1') + Q2 - Q1; stage 4 Psi(k3') ~ Psi(k2') + Q3 - Q2.
  void rk4_guess_before() {
    const int st = rk_stage;
    double* S[4] = {rkS[0], rkS[1], rkS[2], rkS[3]};
    double* Q[4] = {rkQ[0], rkQ[1], rkQ[2], rkQ[3]};
    const double q = rk_qok ? 1. : 0.;
    if (st == 0 && rk_full) {
      const double a[6] = {-0.5, 1. / 3., 2. / 3., 0.5, q / 6., -q / 6.};
      const double* x[6] = {S[0], S[1], S[2], S[3], Q[3], Q[2]};
      psi_combine(stream, D, rk_qok ? 6 : 4, a, x, psi, nullptr);
    } else if (st == 1 && rk_cur == 1) {
      if (rk_full) {
        // T1 = psi; guess 4 T1 - 2 S3 - S4 - Q4/2 (Q4 of the older step), then the Q history of the
        // completed step: Q1 = 2 (S2 - S1), Q2 = 2 (S3 - S1), Q3 = S4 - S1, Q4 = 6 T1 + 2 S1 - 2 S2 - 4 S3 - 2 S4
        // (mode 3's guess 4 T1 + S1 - S2 - 2 S3 - S4 while Q holds no complete step), and S1 = T1, in one pass
        rk4_history(stream, D, rk_qok ? 1 : 0, psi, S, Q);
        rk_qok = true;
      } else {
        dcopy(rkS[0], psi, D);
      }
    } else if (st == 2 && rk_cur == 2 && rk_qok) {
      const double a[3] = {1., 0.5, -0.5};
      const double* x[3] = {psi, Q[1], Q[0]};
      psi_combine(stream, D, 3, a, x, psi, nullptr);
    } else if (st == 3 && rk_cur == 3) {
      const double a[4] = {2., -1., q, -q};
      const double* x[4] = {psi, rkS[0], Q[2], Q[1]};
      psi_combine(stream, D, rk_qok ? 4 : 2, a, x, psi, nullptr);
    }
  }
  void rk_guess_before() {
    if (guess_mode() >= 4) { rk4_guess_before(); return; }
    const int st = rk_stage;
    if (st == 0 && rk_full) {
      const double a[4] = {-0.5, 1. / 3., 2. / 3., 0.5};
      const double* x[4] = {rkS[0], rkS[1], rkS[2], rkS[3]};
      psi_combine(stream, D, 4, a, x, psi, nullptr);
    } else if (st == 1 && rk_cur == 1) {
      if (rk_full) {
        const double a[5] = {4., 1., -1., -2., -1.};
        const double* x[5] = {psi, rkS[0], rkS[1], rkS[2], rkS[3]};
        psi_combine(stream, D, 5, a, x, psi, rkS[0]);
      } else {
        dcopy(rkS[0], psi, D);
      }
    } else if (st == 3 && rk_cur == 3) {
      const double a[2] = {2., -1.};
      const double* x[2] = {psi, rkS[0]};
      psi_combine(stream, D, 2, a, x, psi, nullptr);
    }
  }
  // Whether the stage solution in psi continues the history, and where its copy goes (null: nowhere).
  bool rk_continues() const { return !(rk_stage != rk_cur % 4 || (rk_stage > 0 && rk_cur != rk_stage)); }
  double* rk_copy() {
    return guess_mode() >= 3 && rk_stage >= 1 && !std::isnan(stage_tau) && rk_continues() ? rkS[rk_stage].p : nullptr;
  }
  void rk_guess_after(bool copied) {
    const int st = rk_stage;
    if (!rk_continues()) { rk_full = false; rk_qok = false; rk_cur = 0; return; }
    if (st >= 1 && !copied) dcopy(rkS[st], psi, D);
    rk_cur = st + 1;
    if (st == 3) { rk_full = true; rk_cur = 0; }
  }
  // Mode 5: projection for successive right-hand sides (P. F. Fischer, Comput. Methods Appl. Mech.
  // Engrg. 163 (1998) 193-204), applied to the correction of mode 4's guess x0 (with Euler and RK2,
  // whose stiff modes alternate in sign from step to step: of the previous solution).  A basis X of
  // up to M = kProjVectors vectors spanning earlier stage solutions, with their images AX = As X and Gram
  // matrix G = Y^T AX, gives the start x0 + X c with c = G^-1 Y^T (b - As x0):
  //   symmetric As (PCG): Y = X, the As-norm best correction in the span;
  //   otherwise (BiCGSTAB): Y = AX, the least-squares residual.
  // Either is never worse than x0 in its norm.  A new solution x is appended after its solve as
  // x - X e with e = G^-1 Y^T As x = G^-1 (Y^T b - Y^T r); the Y^T b part is formed before the
  // solve in the pass that forms c, and the Y^T r part (within the solve's tolerance) is left in
  // place.  The appended vector's image is applied by the operator (one apply per solve): images
  // inferred from the solve's recursive residual, b - r - AX e, carried the residual's drift, and
  // the projection built on them degraded as the basis aged.  Its Gram column is then measured
  // exactly, so the basis is not kept orthogonal and needs no second pass or normalisation.
  // Each appended solution's coefficients in the basis are kept (W).  A full basis restarts from
  // the span of its newest kProjKeep solutions: their coefficient columns, orthonormalised on the
  // host in the inner product of G (every column of it measured: at an append, or after the last
  // restart), recombine the basis in one pass; a pass over the recombined vectors then measures
  // their Gram matrix (about I), so the start of every solve is projected on at least kProjKeep
  // earlier solutions.  24 kept 12 took fewer iterations than 16 kept 8 for less than the extra
  // upkeep (at 512^2, K = 5: 2.05 against 2.44 per solve, 463 against 438 FP64 Mdof-steps/s);
  // 32 kept 16 took 1.89 for the same throughput.
  static constexpr int kProjVectors = 24;
  static constexpr int kProjKeep = 12;
  static constexpr int kProjLdg = kProjVectors + 1;  // Gram column: M entries and the solution's norm
  static constexpr int kProjCoef = 2 * kProjMax;      // c and e of one segment
  static_assert(2 * kProjKeep <= kProjVectors && kProjVectors <= kProjMax, "basis restart sizes");
  struct ProjBasis {
    DBuf<double> X, AX;
    // per segment: Gram columns (M x kProjLdg), solution coefficients (M x M), restart combination
    // or measured Gram matrix (M x M)
    DBuf<double> G, W, C;
    DBuf<double> L;  // per segment: the Gram matrix's Cholesky factor (k_proj_solve)
    int fact = 0;    // its rows
    int m = 0;       // vectors held
    int e_m = -1;    // basis size the coefficients e of the solve in progress were formed for
    int v_slot = -1; // the slot holding -X e for the append after the solve in progress (or -1)
    // the newest slot, whose Gram column and solution norm (partials in pnorm) the next projected solve forms
    int gcol_pending = -1;
    DBuf<double> pnorm;
    int nseg = 0;    // segments the per-segment arrays were sized for
    int restarts = 0;
  };
  ProjBasis proj_fwd, proj_adj;     // stage solves; adjoint (transposed) solves
  ProjBasis* proj_cur = &proj_fwd;  // the basis of the solve in progress
  bool proj_force = false;          // project a solve that is not a stage solve (adjoint solves)
  DBuf<double> pcoef, ppart, ptmp;  // pcoef: per segment c (m) and e (m)
  // The projection's dof segments: one per ensemble instance (each projects on its own
  // coefficients), one for a single problem.
  ProjSeg pseg;
  DBuf<int32_t> pseg_blk, pseg_bbeg;
  DBuf<int64_t> pseg_sbeg;
  std::vector<int64_t> pseg_key;  // the segments' first dofs the map was built for
  bool proj_on() const { return guess_mode() >= 5; }
  bool proj_mr() const { return krylov != HOC_KRYLOV_PCG; }  // minimal-residual form
  // The segment map (rebuilt when the mesh or the instances change) and the per-instance norms
  // of an ensemble's convergence test.
  DBuf<double> ens_part, ens_rr, ens_bb;
  bool ens_pcg() const { return n_inst > 1 && krylov == HOC_KRYLOV_PCG; }
  // The batched ensemble PCG (ens_iter) when no Q1 vertex is shared between instances (else the
  // joint PCG with the per-instance stopping test).
  bool inst_coupled = false;
  bool ens_batched() const { return ens_pcg() && !inst_coupled; }
  DBuf<double> ens_in, ens_rz, ens_alpha, ens_beta;
  DBuf<int> ens_act;
  EnsKry ensk() {
    return EnsKry{ens_in.p, ens_rz.p, ens_alpha.p, ens_beta.p, ens_bb.p, ens_act.p, pseg.nseg, ens_part.p, d_ioff.p};
  }
  void ensure_segments() {
    std::vector<int64_t> sb;
    if (n_inst > 1 && (int)inst_off.size() == n_inst + 1)
      for (int32_t e : inst_off) sb.push_back((int64_t)e * K2);
    else
      sb = {0, (int64_t)D};
    if (sb == pseg_key) return;
    std::vector<int32_t> bbeg, blk;
    proj_seg_layout(sb, bbeg, blk);
    pseg_sbeg.upload(sb); pseg_bbeg.upload(bbeg); pseg_blk.upload(blk);
    pseg.nseg = (int)sb.size() - 1;
    pseg.nb = (int)blk.size();
    pseg.maxb = 0;
    for (int i = 0; i < pseg.nseg; ++i) pseg.maxb = std::max(pseg.maxb, bbeg[i + 1] - bbeg[i]);
    pseg.blk_seg = pseg_blk.p; pseg.bbeg = pseg_bbeg.p; pseg.sbeg = pseg_sbeg.p;
    pseg_key = sb;
    ptmp.alloc(0);
    ens_part.alloc(std::max(N, pseg.nb)); ens_rr.alloc(pseg.nseg); ens_bb.alloc(pseg.nseg);
    for (auto* b : {&ens_in, &ens_rz, &ens_alpha, &ens_beta}) b->alloc(pseg.nseg);
    ens_act.alloc(pseg.nseg);
    HIPCHK(hipMemsetAsync(ens_alpha.p, 0, pseg.nseg * sizeof(double), stream));
    HIPCHK(hipMemsetAsync(ens_act.p, 0, pseg.nseg * sizeof(int), stream));
  }
  void proj_alloc() {
    ensure_segments();
    if (ptmp.n < D) {  // t of proj_before; coefficients; partial sums
      ptmp.alloc(D);
      pcoef.alloc((size_t)pseg.nseg * kProjCoef);
      ppart.alloc((size_t)pseg.nb * std::max(2 * kProjMax + 2, kProjVectors * kProjVectors));
    }
  }
  // c, e: the coefficients of the first m vectors; sums: proj_dots3's are still to be formed
  void proj_coefs(ProjBasis& P, int m, bool sums) {
    proj_solve(stream, pseg, m, P.fact, P.G.p, kProjLdg, kProjVectors * kProjLdg, P.L, pcoef, kProjCoef,
               sums ? ppart.p : nullptr, sums ? P.pnorm.p : nullptr);
    P.fact = m;
  }
  void proj_before(const double* b) {
    ProjBasis& P = *proj_cur;
    P.e_m = -1;
    P.v_slot = -1;
    if (P.m == 0) return;
    proj_alloc();
    if (P.nseg != pseg.nseg) { P.m = 0; return; }
    double* t = ptmp.p;
    residual_As(psi.p, b, t, nullptr);  // t = b - As x0
    const double* Y = proj_mr() ? P.AX.p : P.X.p;
    if (P.gcol_pending >= 0 && P.gcol_pending == P.m - 1) {  // Y^T t, Y^T b and the newest Gram column
      const int j = P.m - 1;
      double* gcol = P.G.p + (size_t)j * kProjLdg;
      proj_dots3(stream, D, pseg, P.m, Y, P.AX.p + (size_t)j * D, t, b, ppart, pcoef, kProjCoef, gcol,
                 kProjVectors * kProjLdg);
      const bool inl = proj_inline(pseg);  // the solve sums what the dots left
      if (!inl) proj_sum(stream, pseg, P.pnorm, gcol + P.m, kProjVectors * kProjLdg);
      proj_coefs(P, P.m, inl);
    } else {
      proj_dots2(stream, D, pseg, P.m, Y, t, b, ppart, pcoef, kProjCoef);  // Y^T t, Y^T b
      proj_coefs(P, P.m, false);
    }
    P.gcol_pending = -1;
    // with a free slot, the same pass leaves -X e there for the append after this solve
    const bool pre = P.m < kProjVectors;
    proj_combine(stream, D, pseg, P.m, P.X.p, pcoef, kProjCoef, psi, pre ? P.X.p + (size_t)P.m * D : nullptr);
    P.e_m = P.m;
    P.v_slot = pre ? P.m : -1;
  }
  // A full basis: keep, per segment, the span of the newest kProjKeep appended solutions
  // (columns M - kProjKeep .. M - 1 of W: with kProjKeep <= M / 2 these were all appended after
  // the last restart).  The new basis is orthonormalised in the inner product of the Gram matrix
  // held in G's columns, and the new vectors' Gram matrix, measured after the recombination,
  // replaces it; a segment whose newest solutions span fewer than the most vectors kept by any
  // segment gets zero vectors in the remaining slots (left out of its solves).
  void proj_restart(ProjBasis& P) {
    constexpr int M = kProjVectors, KP = kProjKeep, LG = kProjLdg;
    const int ns = pseg.nseg;
    P.m = 0;
    P.e_m = -1;
    P.v_slot = -1;
    P.gcol_pending = -1;
    P.fact = 0;
    ++P.restarts;
    if (KP == 0) return;
    std::vector<double> w((size_t)ns * M * M), gc((size_t)ns * M * LG), gm((size_t)M * M);
    HIPCHK(hipStreamSynchronize(stream));
    d2h(w.data(), P.W.p, w.size() * sizeof(double));
    d2h(gc.data(), P.G.p, gc.size() * sizeof(double));
    std::vector<std::vector<double>> cs(ns);
    int kk = 0;
    for (int sg = 0; sg < ns; ++sg) {
      const double* W = w.data() + (size_t)sg * M * M;
      const double* Gc = gc.data() + (size_t)sg * M * LG;
      for (int j = 0; j < M; ++j)  // the symmetric Gram matrix from its columns (upper triangle)
        for (int i = 0; i <= j; ++i) gm[(size_t)i * M + j] = gm[(size_t)j * M + i] = Gc[(size_t)j * LG + i];
      const int k = proj_restart_basis(M, KP, Gc, LG, gm.data(), W, cs[sg]);
      kk = std::max(kk, k);
    }
    if (kk == 0) return;
    // combinations (zero rows pad a segment to kk), then the recombined vectors' Gram matrix
    std::vector<double> ca((size_t)ns * M * M, 0.), gn((size_t)ns * kk * kk), gi((size_t)ns * M * LG, 0.);
    for (int sg = 0; sg < ns; ++sg) std::copy(cs[sg].begin(), cs[sg].end(), ca.begin() + (size_t)sg * M * M);
    HIPCHK(hipMemcpyAsync(P.C.p, ca.data(), ca.size() * sizeof(double), hipMemcpyHostToDevice, stream));
    proj_reseed(stream, D, pseg, M, kk, P.C.p, M * M, P.X.p, P.AX.p);
    proj_gram(stream, D, pseg, kk, proj_mr() ? P.AX.p : P.X.p, P.AX.p, ppart, P.C.p);  // kk x kk per segment
    HIPCHK(hipStreamSynchronize(stream));  // (ca is a local)
    d2h(gn.data(), P.C.p, gn.size() * sizeof(double));
    // the Gram columns of the new vectors, each with a unit solution norm (zero vectors padding a
    // segment have G_jj = 0 and are left out)
    for (int sg = 0; sg < ns; ++sg)
      for (int j = 0; j < kk; ++j) {
        double* col = gi.data() + (size_t)sg * M * LG + (size_t)j * LG;
        for (int i = 0; i <= j; ++i) col[i] = gn[(size_t)sg * kk * kk + (size_t)i * kk + j];
        col[j + 1] = 1.;
      }
    HIPCHK(hipMemcpyAsync(P.G.p, gi.data(), gi.size() * sizeof(double), hipMemcpyHostToDevice, stream));
    HIPCHK(hipStreamSynchronize(stream));  // (gi is a local)
    P.m = kk;
  }
  // save (may be null): where a copy of psi is wanted; true when the append's pass has made it.
  bool proj_after(const double* b, double* save) {
    constexpr int M = kProjVectors;
    bool saved = false;
    ProjBasis& P = *proj_cur;
    proj_alloc();
    if (P.X.n < (size_t)M * D || P.nseg != pseg.nseg) {
      P.X.alloc((size_t)M * D); P.AX.alloc((size_t)M * D);
      const size_t ns = pseg.nseg;
      P.G.alloc(ns * M * kProjLdg); P.W.alloc(ns * M * M); P.C.alloc(ns * M * M);
      P.L.alloc(ns * kProjL);
      P.nseg = pseg.nseg;
      P.m = 0;
    }
    if (P.pnorm.n < (size_t)pseg.nb) P.pnorm.alloc(pseg.nb);
    proj_flush_gcol(P);
    if (P.m >= M) proj_restart(P);
    const int j = P.m;
    P.fact = std::min(P.fact, j);
    if (j > 0 && P.e_m != j) {  // e = G^-1 Y^T b
      proj_dots2(stream, D, pseg, j, proj_mr() ? P.AX.p : P.X.p, b, b, ppart, pcoef, kProjCoef);
      proj_coefs(P, j, false);
    }
    // x = psi - X e into slot j, its exact image As x, and its Gram column
    double* xj = P.X.p + (size_t)j * D;
    double* axj = P.AX.p + (size_t)j * D;
    if (P.v_slot == j && P.e_m == j) {  // slot j holds -X e from proj_before's pass
      proj_append(stream, D, pseg, j, proj_mr() ? 1 : 0, pcoef.p + j, kProjCoef, psi, b, xj, P.pnorm,
                  P.W.p + (size_t)j * M, M * M, M, save);
      saved = save != nullptr;
    } else {
      proj_ortho(stream, D, pseg, j, proj_mr() ? 1 : 0, P.X.p, pcoef.p + j, kProjCoef, psi, b, xj, P.pnorm,
                 P.W.p + (size_t)j * M, M * M, M);
    }
    apply_As(xj, axj);
    // its Gram column (Y_i . axj, i <= j) comes from the next projected solve's pass over Y
    // (proj_dots3), or from proj_flush_gcol when the basis is used otherwise first
    P.m = j + 1;
    P.e_m = -1;
    P.v_slot = -1;
    P.gcol_pending = j;
    return saved;
  }
  // The Gram column of the newest vector when it is still pending (its vector and image are in
  // their slots); a pending column of a basis since reset is dropped.
  void proj_flush_gcol(ProjBasis& P) {
    const int j = P.gcol_pending;
    P.gcol_pending = -1;
    if (j < 0 || j != P.m - 1) return;
    constexpr int M = kProjVectors;
    proj_gcol(stream, D, pseg, j, proj_mr() ? 1 : 0, proj_mr() ? P.AX.p : P.X.p, P.X.p + (size_t)j * D,
              P.AX.p + (size_t)j * D, ppart, P.G.p + (size_t)j * kProjLdg, M * kProjLdg);
    proj_sum(stream, pseg, P.pnorm, P.G.p + (size_t)j * kProjLdg + j + 1, M * kProjLdg);
  }
  // The adjoint's colouring, velocity map, buffers and recorded trajectory belong to one mesh and
  // one set-up: a new mesh or set-up rebuilds them on the next adjoint call.
  void reset_adjoint() {
    adj.init = false;
    adj.have_forward = false;
    adj.zn = 0;
    proj_adj.m = 0;
  }
  // Called when the state is set from outside: the histories restart, so that the same state gives
  // the same iterations (the projection basis would stay valid, holding solutions of As x = b only).
  void invalidate_guess() {
    proj_fwd.m = 0;
    n_hist = 0;
    rk_full = false;
    rk_qok = false;
    rk_cur = 0;
  }
  void guess_before_solve() {
    if (guess_mode() >= 3 && rk_stage >= 0 && !std::isnan(stage_tau)) { rk_guess_before(); return; }
    if (guess_mode() < 2 || guess_mode() == 5 || std::isnan(stage_tau)) return;
    const double tau = stage_tau;
    if (n_hist == 0 || tau == tau_a) return;  // no history, or the same stage time: the previous solution
    const bool ok = n_hist == 2 && tau > tau_a && tau - tau_a <= 1. && tau_a > tau_b && tau_a - tau_b <= 1.;
    psi_predict(stream, D, ok ? (tau - tau_a) / (tau_a - tau_b) : 0., ok ? 1 : 0, psi, psi_prev);
  }
  // copied: rk_copy's copy has been made
  void guess_after_solve(bool copied) {
    if (guess_mode() >= 3 && rk_stage >= 0 && !std::isnan(stage_tau)) { rk_guess_after(copied); return; }
    rk_full = false;
    rk_qok = false;
    rk_cur = 0;
    if (guess_mode() < 2 || std::isnan(stage_tau)) { n_hist = 0; return; }
    if (n_hist >= 1 && stage_tau == tau_a) return;
    if (n_hist == 0) { tau_a = stage_tau; n_hist = 1; return; }
    tau_b = tau_a;
    tau_a = stage_tau;
    n_hist = 2;
  }

  void poisson(const double* omega) {
    guess_before_solve();
    const int maxit = cfg.maxiter;
    HIPCHK(launch_rhs(K, geo_kind, N, T, G, omega, rhs_bc ? rhs_bc : b_psi.p, bs, part2, stream));
    const bool proj = proj_on() && (!std::isnan(stage_tau) || proj_force);
    if (proj) proj_before(bs);
    bool have_bb = false;
    if (ens_pcg()) {
      // PCG: the iterations continue while some instance has ||r_i|| > tol ||b_i||
      ensure_segments();
      seg_norm2(stream, pseg, VA, bs, nullptr, ens_part.p, ens_bb.p);
    } else if (n_inst > 1) {
      finalize(stream, PH_BB, part2, fine_blocks(K, N), S, F, maxit);
      have_bb = true;
      // BiCGSTAB: ||b - A psi|| <= tol min_i ||b_i|| bounds every instance's own relative residual
      // (instances with a zero right-hand side are left out of the minimum)
      inst_norms(stream, VA, n_inst, d_ioff, K2, bs, d_inorm);
      std::vector<double> bi(n_inst);
      double bb = 0.;
      HIPCHK(hipMemcpyAsync(bi.data(), d_inorm.p, n_inst * sizeof(double), hipMemcpyDeviceToHost, stream));
      HIPCHK(hipMemcpyAsync(&bb, S.p + S_BB, sizeof(double), hipMemcpyDeviceToHost, stream));
      HIPCHK(hipStreamSynchronize(stream));
      double mx = 0., mn = HUGE_VAL;
      for (double v : bi) mx = std::max(mx, v);
      for (double v : bi) if (v > 1e-30 * mx) mn = std::min(mn, v);
      const double tol2 = cfg.tol * cfg.tol;
      const double t2 = (bb > 0. && mn < HUGE_VAL) ? tol2 * mn / bb : tol2;
      HIPCHK(hipMemcpyAsync(S.p + S_TOL2, &t2, sizeof(double), hipMemcpyHostToDevice, stream));
      HIPCHK(hipStreamSynchronize(stream));
    }
    const double* pbb = have_bb ? nullptr : part2.p;
    outer_residual(pbb);
    // FP64: the FP64 V-cycle; mixed: the FP32 V-cycle; the Krylov vectors, the operator
    // application and the stopping test in FP64 either way.  The results arrive with the status of
    // the last iteration, so the stream goes on without a copy or a wait for it to drain.
    krylov_solve(psi.p, P64.r.p, pbb, S.p, F.p, maxit, maxit);
    const MirrorState res = *mirror;
    // a zero right-hand side: psi = 0, as the reference's solver returns
    if (res.zero) HIPCHK(hipMemsetAsync(psi.p, 0, D * sizeof(double), stream));
    // statistics
    last_iters = res.iter;
    last_outer = 0;
    if (!std::isfinite(res.bb) || !std::isfinite(res.rr)) {
      last_rel = std::nan("");
      throw StatusError(HOC_ENAN, "NaN/Inf in the Poisson right-hand side or residual");
    }
    last_rel = res.bb > 0. ? std::sqrt(res.rr / res.bb) : 0.;
    if (res.zero) last_rel = 0.;
    total_iters += last_iters;
    ++n_solves;
    bool copied = false;
    if (proj && !res.zero) copied = proj_after(bs, rk_copy());
    guess_after_solve(copied);
    if (!std::isfinite(last_rel)) throw StatusError(HOC_ENAN, "NaN/Inf in the Poisson solve");
    if (cfg.fail_on_noconv && last_rel > cfg.tol)
      throw StatusError(HOC_ENOCONV, "Poisson solve did not converge: rel residual " + std::to_string(last_rel));
  }

  // ---- node-averaged output and sample points ---------------------------------------------
  DBuf<int32_t> d_elnodes, d_nptr, d_ninc, d_sel;
  DBuf<double> d_bmet, d_elemout, d_nodeout, d_sshape, d_sval;
  bool smooth_ready = false;
  int n_sp = 0;
  std::vector<double> sp_xy, sp_loc;
  std::vector<int32_t> sp_elem;

  // Element node lists, node incidences in element order and the boundary faces' metrics,
  // uploaded on the first output call.
  void smooth_setup() {
    if (smooth_ready) return;
    const int L2 = mesh.lnod * mesh.lnod;
    d_elnodes.upload(mesh.elem);
    std::vector<int32_t> ptr((size_t)mesh.n_nodes + 1, 0), inc((size_t)N * L2);
    for (int32_t nd : mesh.elem) ptr[(size_t)nd + 1]++;
    for (int i = 0; i < mesh.n_nodes; ++i) ptr[i + 1] += ptr[i];
    std::vector<int32_t> pos(ptr.begin(), ptr.end() - 1);
    for (int el = 0; el < N; ++el)
      for (int l = 0; l < L2; ++l) inc[pos[mesh.elem[(size_t)el * L2 + l]]++] = el * L2 + l;
    d_nptr.upload(ptr);
    d_ninc.upload(inc);
    std::vector<double> bm((size_t)std::max(E, 1) * K * 4, 0.);
    for (int e = 0; e < E; ++e)
      for (int k = 0; k < K; ++k) {
        const size_t q = ((size_t)mesh.be_elem[e] * 4 + mesh.be_ijp[e]) * K + k;
        double* o = &bm[((size_t)e * K + k) * 4];
        o[0] = geo.fxxi[q]; o[1] = geo.fxeta[q]; o[2] = geo.fyxi[q]; o[3] = geo.fyeta[q];
      }
    d_bmet.upload(bm);
    d_elemout.alloc((size_t)N * L2 * 4);
    d_nodeout.alloc((size_t)mesh.n_nodes * 4);
    smooth_ready = true;
  }
  // What the reference's main loop runs before each dump (src/HO_2D.cpp:1411-1414): boundary
  // values at the current time, the stream function and the velocity of the current vorticity.
  void refresh_fields() {
    update_bcs(0.);
    poisson(w);
    HIPCHK(launch_velocity(K, geo_kind, N, T, G, B, psi, vel, U, tru, 1. / (cfg.dt * re_inv), I, stream));
  }
  // Node-averaged vorticity, psi and velocity into d_nodeout (save_smooth_vtk,
  // src/HO_2D.cpp:3369-3531).
  void node_fields(bool refresh) {
    smooth_setup();
    if (refresh) refresh_fields();
    SmoothArgs A{};
    A.N = N; A.K = K; A.L = mesh.lnod;
    for (int k = 0; k < K; ++k)  // sps_gps_basis (src/HO_2D.cpp:571-583)
      for (int l = 0; l < A.L; ++l) {
        double num = 1., den = 1.;
        for (int j = 0; j < K; ++j) {
          if (j == k) continue;
          den *= tab.sps[k] - tab.sps[j];
          num *= tab.gps[l] - tab.sps[j];
        }
        A.sgb[k][l] = num / den;
      }
    for (int j = 0; j < A.L; ++j)
      for (int i = 0; i < A.L; ++i) A.slot[j * A.L + i] = gmsh_slot(A.L, i, j);
    A.w = w; A.psi = psi; A.vel = vel; A.nb = d_nb;
    A.bvort = b_vort; A.bnvel = b_nvel; A.bpvel = b_pvel; A.bmet = d_bmet; A.elemout = d_elemout;
    HIPCHK(launch_smooth_elem(A, stream));
    HIPCHK(launch_smooth_nodes(mesh.n_nodes, d_nptr, d_ninc, d_elemout, d_nodeout, stream));
  }
  void set_sample_points(int n, const double* xy) {
    std::vector<double> shape;
    try {
      locate_sample_points(mesh, tab, n, xy, sp_elem, sp_loc, shape);
    } catch (const std::runtime_error& e) {
      throw StatusError(HOC_EINVAL, e.what());
    }
    sp_xy.assign(xy, xy + 2 * (size_t)n);
    n_sp = n;
    if (n > 0) { d_sel.upload(sp_elem); d_sshape.upload(shape); d_sval.alloc(3 * (size_t)n); }
  }
  void sample_values(bool refresh, double* out) {
    node_fields(refresh);
    HIPCHK(launch_sample(n_sp, mesh.lnod * mesh.lnod, d_sel, d_sshape, d_elnodes, d_nodeout, d_sval, stream));
    if (n_sp > 0) d2h(out, d_sval.p, 3 * (size_t)n_sp * sizeof(double));
    else HIPCHK(hipStreamSynchronize(stream));
  }

  // Validates a mesh given as arrays or read from a file and makes it the handle's mesh.
  void accept_mesh(Mesh&& m) {
    for (int32_t v : m.elem) if (v < 0 || v >= m.n_nodes) throw StatusError(HOC_EINVAL, "element node id out of range");
    for (auto& e : m.edges)
      for (int32_t v : e) if (v < 0 || v >= m.n_nodes) throw StatusError(HOC_EINVAL, "edge node id out of range");
    for (int32_t b : m.bedge_bdry)
      if (b < 0 || b >= (int)m.bnames.size()) throw StatusError(HOC_EINVAL, "boundary id out of range");
    mesh = std::move(m);
    mesh_loaded = true;
    ready = false;
    reset_adjoint();
    n_inst = 1;
    inst_off.clear(); inst_re.clear(); inst_dt.clear(); inst_time.clear();
    edge_nvel_in.clear(); edge_has_nvel.clear();
  }

  double ramp(double t) const { return bch.time_dependent ? 2. * std::fabs(std::sin(M_PI / 40. * t)) : 1.; }

  // Boundary values at stage fraction c of the step (each instance at its own clock), or at
  // the absolute time t_abs for all instances when t_abs is given.
  void update_bcs(double c, double t_abs = std::nan("")) {
    if (cfg.problem_type == 11) {
      const double t = std::isnan(t_abs) ? time + c * cfg.dt : t_abs;
      const double span = time_end - time_start;
      const double fac1 = span > 0. ? (t - time_start) / span : 0.;
      HIPCHK(launch_update_bcs_hybrid(E * K, K, B, H, fac1, 1. - fac1, stream));
      HIPCHK(launch_hybrid_blend(D, w, H, fac1, 1. - fac1, stream));
      return;
    }
    if (n_inst > 1 && std::isnan(t_abs)) {
      std::vector<double> r(n_inst);
      for (int i = 0; i < n_inst; ++i) r[i] = ramp(inst_time[i] + c * inst_dt[i]);
      HIPCHK(hipMemcpyAsync(d_iramp.p, r.data(), n_inst * sizeof(double), hipMemcpyHostToDevice, stream));
      HIPCHK(launch_update_bcs(E * K, K, B, 1., I, stream));
    } else {
      InstDev I0 = I;
      I0.ramp = nullptr;
      HIPCHK(launch_update_bcs(E * K, K, B, ramp(std::isnan(t_abs) ? time + c * cfg.dt : t_abs), I0, stream));
    }
  }

  // Euler_time_integrate (src/HO_2D.cpp:1806-1839) on input win; boundary values already set.
  double* capture_psi = nullptr;  // when set, RK4 stage s copies its solution to capture_psi + s D
  void stage_body(const double* win, const StageOut& so) {
    poisson(win);
    if (capture_psi && rk_stage >= 0) dcopy(capture_psi + (size_t)rk_stage * D, psi, D);
    // the Cartesian velocity is an output of the step's last stage only (what the getters and
    // writers read); intermediate RK stages need the contravariant fluxes U alone
    HIPCHK(launch_velocity(K, geo_kind, N, T, G, B, psi, so.inner ? nullptr : vel.p, U, tru, 1. / (cfg.dt * re_inv), I,
                           stream));
    HIPCHK(launch_stage(K, geo_kind, cfg.advection_type, N, T, G, B, win, U, tru, re_inv, cfg.dt, I, so, stream));
  }
  void stage(const double* win, double c, const StageOut& so) {
    update_bcs(c);
    stage_tau = (double)step_count + c;
    try {
      stage_body(win, so);
    } catch (...) {
      stage_tau = std::nan("");
      rk_stage = -1;
      n_hist = 0;
      rk_full = false;
      rk_qok = false;
      rk_cur = 0;
      throw;
    }
    stage_tau = std::nan("");
  }

  // solve_advection_diffusion (src/HO_2D.cpp:1465-1531)
  void rk_step() {
    StageOut so;
    // a stage's input is none of its outputs: the inputs alternate between vort and vort2
    if (cfg.time_integration_type == 1) {
      so.next = vort; so.c = 1.; so.base = w;
      stage(w, 0., so);
      std::swap(w.p, vort.p);  // nothing keeps either address from one launch to the next
    } else if (cfg.time_integration_type == 2) {
      so.k = k1; so.next = vort; so.c = 1.; so.base = w; so.inner = true;
      stage(w, 0., so);
      StageOut s2; s2.base = w; s2.final_mode = 2; s2.k1 = k1;
      stage(vort, 1., s2);
    } else if (cfg.time_integration_type == 4) {
      const double c[4] = {0., 0.5, 0.5, 1.};
      double* ks[3] = {k1, k2, k3};
      rk_stage = 0;
      stage_rk4(w, c[0], ks[0], 0.5, vort);
      rk_stage = 1;
      stage_rk4(vort, c[1], ks[1], 0.5, vort2);
      rk_stage = 2;
      stage_rk4(vort2, c[2], ks[2], 1.0, vort);
      StageOut s4; s4.base = w; s4.final_mode = 4; s4.k1 = k1; s4.k2 = k2; s4.k3 = k3;
      rk_stage = 3;
      stage(vort, c[3], s4);
      rk_stage = -1;
    } else {
      throw StatusError(HOC_EINVAL, "time_integration_type must be 1, 2 or 4");
    }
    time += cfg.dt;
    ++step_count;
    for (int i = 0; i < n_inst && n_inst > 1; ++i) inst_time[i] += inst_dt[i];
  }
  void stage_rk4(const double* win, double c, double* kout, double cnext, double* next) {
    StageOut so; so.k = kout; so.next = next; so.c = cnext; so.base = w; so.inner = true;
    stage(win, c, so);
  }

  // Hybrid tables: edge kinds, open-boundary order, zero start/end values and targets.
  void setup_hybrid() {
    H = HybridDev{};
    open_edges.clear();
    time_start = time_end = 0.;
    if (cfg.problem_type != 11) return;
    for (int b = 0; b < (int)mesh.bnames.size(); ++b)
      if (mesh.bnames[b] == "open")
        for (int e = 0; e < E; ++e) if (mesh.bedge_bdry[e] == b) open_edges.push_back(e);
    const size_t EK = std::max<size_t>((size_t)E * K, 1);
    d_hkind.upload(bch.hybrid_kind);
    d_hinlet.upload(bch.inlet_nvel);
    for (auto* b : {&d_vn0, &d_vn1, &d_vp0, &d_vp1, &d_vw0, &d_vw1}) b->alloc(EK);
    for (auto* b : {&d_hw0, &d_hw1, &d_hwgt}) b->alloc(D);
    h_vn1.assign(EK, 0.); h_vp1.assign(EK, 0.); h_vw1.assign(EK, 0.);
    H = HybridDev{d_hkind, d_hinlet, d_esign, d_swdiff, d_vn0, d_vn1, d_vp0, d_vp1, d_vw0, d_vw1, d_hw0, d_hw1, d_hwgt};
  }
  void need_hybrid() const {
    if (cfg.problem_type != 11) throw StatusError(HOC_ESTATE, "hybrid driver calls need problem_type 11");
  }
  // getopenpts_d (src/HO_2D.cpp:4007-4046): K points along each open edge, edge node order
  void open_points(double* xy) const {
    const int L = mesh.lnod;
    for (size_t i = 0; i < open_edges.size(); ++i) {
      const auto& nd = mesh.edges[open_edges[i]];  // tensor order after connect()
      for (int j = 0; j < K; ++j) {
        double x = 0., y = 0.;
        for (int l = 0; l < L; ++l) {
          x += tab.gsb[l][j] * mesh.xy[2 * (size_t)nd[l]];
          y += tab.gsb[l][j] * mesh.xy[2 * (size_t)nd[l] + 1];
        }
        xy[2 * (i * K + j)] = x; xy[2 * (i * K + j) + 1] = y;
      }
    }
  }
  // setopenvels_d (src/HO_2D.cpp:4050-4117): start = end, then the new Cartesian velocities
  // as outward-normal and tangential components with the owner face's metrics
  void set_open_velocities(const double* uv) {
    const size_t EK = std::max<size_t>((size_t)E * K, 1);
    HIPCHK(hipMemcpyAsync(d_vn0.p, d_vn1.p, EK * sizeof(double), hipMemcpyDeviceToDevice, stream));
    HIPCHK(hipMemcpyAsync(d_vp0.p, d_vp1.p, EK * sizeof(double), hipMemcpyDeviceToDevice, stream));
    for (size_t i = 0; i < open_edges.size(); ++i) {
      const int e = open_edges[i];
      const int el = mesh.be_elem[e], ijp = mesh.be_ijp[e];
      const double coeff = 2. * (ijp % 2) - 1.;
      for (int j = 0; j < K; ++j) {
        const size_t q = ((size_t)el * 4 + ijp) * K + j;
        const double u = uv[2 * (i * K + j)], v = uv[2 * (i * K + j) + 1];
        double nx, ny;
        if (ijp / 2 == 1) { nx = -geo.fyxi[q]; ny = geo.fxxi[q]; }
        else { nx = geo.fyeta[q]; ny = -geo.fxeta[q]; }
        nx *= coeff / geo.fAn[q];
        ny *= coeff / geo.fAn[q];
        h_vn1[(size_t)e * K + j] = nx * u + ny * v;
        h_vp1[(size_t)e * K + j] = nx * v - ny * u;
      }
    }
    h2d(d_vn1.p, h_vn1.data(), EK * sizeof(double));
    h2d(d_vp1.p, h_vp1.data(), EK * sizeof(double));
  }
  // setopenvort_d (src/HO_2D.cpp:4120-4141)
  void set_open_vorticity(const double* wv) {
    const size_t EK = std::max<size_t>((size_t)E * K, 1);
    HIPCHK(hipMemcpyAsync(d_vw0.p, d_vw1.p, EK * sizeof(double), hipMemcpyDeviceToDevice, stream));
    for (size_t i = 0; i < open_edges.size(); ++i)
      for (int j = 0; j < K; ++j) h_vw1[(size_t)open_edges[i] * K + j] = wv[K * i + j];
    h2d(d_vw1.p, h_vw1.data(), EK * sizeof(double));
  }
  // setsolnvort_d (src/HO_2D.cpp:4144-4166)
  void set_vorticity_target(const double* wv) {
    HIPCHK(hipMemcpyAsync(d_hw0.p, d_hw1.p, D * sizeof(double), hipMemcpyDeviceToDevice, stream));
    h2d(d_hw1.p, wv, D * sizeof(double));
  }

  // ---- discrete adjoint of the RK4 trajectory -------------------------------------------
  // One stage maps omega_s to k_s = dt R(omega_s), with psi_s = A^-1 b(omega_s) and
  // b = -omega J - (boundary source).  Its transpose is applied as
  //   omega_bar  = (dk/domega)^T lam                 (probes: omega, 1-ring)
  //   U_bar      = (dk/dU)^T lam,  diff_bar = (dk/ddiff)^T lam   (probes: velocity, wall flux)
  //   pvel_bar  += sign idr diff_bar                 (no-slip walls: diff = (vjump + sign pvel) idr)
  //   psi_bar    = (dU/dpsi)^T U_bar + (ddiff/dpsi)^T diff_bar   (assembled once: the map is linear
  //                                                              and state-independent)
  //   omega_bar += J W z,   As z = psi_bar           (A^-T = -W As^-1, As symmetric)
  // the probes as coloured, batched launches of the frozen-switch stage (launch_stage mode 2).
  struct Adj {
    bool init = false;
    int nc1 = 0;
    DBuf<int32_t> col1, r1p, r1i, own_el;
    int ub = 1;                       // probe units (hoc_adj.hpp) of a batch
    bool seeds_kept = false;          // every unit fits one batch: its seeds are written once, by the setup
    DBuf<int8_t> own_f;
    DBuf<double> ws[4], Us[4], trus[4];  // recorded stages of one step
    DBuf<int8_t> sig[4];
    // probe batches (ub K^2 probes, at least 4K): seeds, products, velocities and their traces
    DBuf<double> seed, y, p, dU, dtru, lin_diff, lin_vj, pvel_seed;
    DBuf<double> zero_d, zero_e, lin_nvel, lin_vort, lin_adv;
    DBuf<double> lam, xbar, psibar, z, fake, wbar, kbar[4], pvbar;
    DBuf<double> Mv, Md, Ubar, diffbar, zero_u, zero_tu;  // assembled velocity map and its adjoints
    // adjoint solves: the previous solution z (in z) and the one before (zprev) with their stage
    // times, for a guess extrapolated in the reversed stage time
    DBuf<double> zprev;
    double ztau_a = 0., ztau_b = 0.;
    int zn = 0;
    DBuf<double> ckbuf, segbuf, segpsi, save_w, save_psi, save_vel;
    // schedule: 0 uniform segments, 1 every step recorded by the forward run, 2 binomial
    int sched = 0;
    DBuf<double> trajw, trajpsi;   // sched 1: omega_n and the four stage solutions of every step
    DBuf<double> snap;             // sched 2: omega snapshots
    int nsnap = 0;
    std::vector<int> snap_pos;     // sched 2: step held by each snapshot slot (-1: free)
    std::vector<int32_t> bsplit;   // sched 2: optimal first advance for (range, free slots)
    int bsplit_L = 0, bsplit_S = 0;
    int nsteps = 0, every = 0;
    double t0 = 0.;
    bool have_forward = false;
    BCDev Bz{}, Bl{};
    BCDev Bl_seed() const {  // homogeneous boundary values with the wall flux from the edge seeds
      BCDev b = Bl;
      b.diff = pvel_seed;
      return b;
    }
  } adj;

  void adjoint_check() const {
    if (!ready) throw StatusError(HOC_ESTATE, "call hoc_setup first");
    if (mixed) throw StatusError(HOC_EINVAL, "the adjoint needs precision HOC_FP64");
    if (n_inst > 1) throw StatusError(HOC_EINVAL, "the adjoint runs on one instance");
    if (cfg.problem_type != 1 || bch.time_dependent)
      throw StatusError(HOC_EINVAL, "the adjoint needs problem_type 1 (fixed walls, time-independent boundary values)");
    if (cfg.advection_type != 1) throw StatusError(HOC_EINVAL, "the adjoint needs advection_type 1");
    if (cfg.time_integration_type != 4) throw StatusError(HOC_EINVAL, "the adjoint needs time_integration_type 4");
    if (krylov != HOC_KRYLOV_PCG)
      throw StatusError(HOC_EINVAL, "the adjoint needs a symmetric Poisson operator (affine elements)");
    for (int e = 0; e < E; ++e)
      if (bch.sw_psi[e] != 0) throw StatusError(HOC_EINVAL, "the adjoint needs Dirichlet stream-function walls");
  }

  // Greedy colouring in which elements within face distance dist of each other differ.
  int color_within(int dist, std::vector<int32_t>& color) const {
    color.assign(N, -1);
    std::vector<int> mark(N, -1), used;
    std::vector<int> front, next, seen;
    int nc = 0;
    for (int e = 0; e < N; ++e) {
      seen.clear();
      front.assign(1, e);
      mark[e] = e;
      for (int d = 0; d < dist; ++d) {
        next.clear();
        for (int u : front)
          for (int f = 0; f < 4; ++f) {
            const int v = mesh.nb[(size_t)u * 4 + f];
            if (v >= 0 && mark[v] != e) { mark[v] = e; next.push_back(v); seen.push_back(v); }
          }
        front.swap(next);
      }
      for (int v : seen)
        if (color[v] >= 0) used[color[v]] = e;
      int c = 0;
      while (c < (int)used.size() && used[c] == e) ++c;
      if (c == (int)used.size()) used.push_back(-1);
      color[e] = c;
      nc = std::max(nc, c + 1);
    }
    return nc;
  }
  // Elements within face distance dist of each element (itself included), as CSR.
  void rings(int dist, std::vector<int32_t>& ptr, std::vector<int32_t>& idx) const {
    ptr.assign(1, 0);
    idx.clear();
    std::vector<int> mark(N, -1), front, next;
    for (int e = 0; e < N; ++e) {
      mark[e] = e;
      idx.push_back(e);
      front.assign(1, e);
      for (int d = 0; d < dist; ++d) {
        next.clear();
        for (int u : front)
          for (int f = 0; f < 4; ++f) {
            const int v = mesh.nb[(size_t)u * 4 + f];
            if (v >= 0 && mark[v] != e) { mark[v] = e; next.push_back(v); idx.push_back(v); }
          }
        front.swap(next);
      }
      ptr.push_back((int32_t)idx.size());
    }
  }

  void adjoint_setup() {
    adjoint_check();
    if (adj.init) return;
    std::vector<int32_t> c1, p1, i1;
    adj.nc1 = color_within(2, c1);
    rings(1, p1, i1);
    adj.col1.upload(c1);
    adj.r1p.upload(p1); adj.r1i.upload(i1);
    std::vector<int32_t> oe(std::max(E, 1), 0);
    std::vector<int8_t> of(std::max(E, 1), -1);
    for (int e = 0; e < E; ++e) { oe[e] = mesh.be_elem[e]; of[e] = mesh.be_ijp[e]; }
    adj.own_el.upload(oe); adj.own_f.upload(of);
    const size_t TU = (size_t)4 * N * K, EK = std::max<size_t>((size_t)E * K, 1);
    // Units per batch: as many as 256 MiB hold (one, whatever it takes, on meshes whose single units
    // fill the chip): batches of all 14 take 24 x 24 elements, K = 4, from 95 launches a stage to 14.
    const double unit = 8. * K2 * (4. * (double)D + (double)TU);
    adj.ub = (int)std::min(std::max(268435456. / unit, 1.), 2. * adj.nc1);
    adj.seeds_kept = adj.ub == 2 * adj.nc1;
    const size_t NB1 = std::max(K2, 4 * K), NB = std::max<size_t>((size_t)adj.ub * K2, NB1);
    const size_t NBw = std::max<size_t>((size_t)std::min(adj.ub, adj.nc1) * K2, NB1);  // vorticity units alone
    for (int s4 = 0; s4 < 4; ++s4) {
      adj.ws[s4].alloc(D); adj.Us[s4].alloc(2 * D); adj.trus[s4].alloc(TU);
      adj.sig[s4].alloc((size_t)4 * N * K); adj.kbar[s4].alloc(D);
    }
    for (DBuf<double>* b : {&adj.zero_d, &adj.lam, &adj.xbar, &adj.psibar, &adj.z, &adj.fake, &adj.wbar, &adj.save_w,
                            &adj.save_psi})
      b->alloc(D);
    adj.save_vel.alloc(2 * D);
    adj.seed.alloc(NBw * D); adj.y.alloc(NB * D);
    adj.dU.alloc(NB * 2 * D); adj.dtru.alloc(NB * TU);
    adj.p.alloc(NB * std::max(N, 1));
    adj.lin_diff.alloc(NB1 * EK); adj.lin_vj.alloc(NB1 * EK); adj.pvel_seed.alloc((size_t)4 * K * EK);
    // seeds of the wall-flux probes are edge arrays like the wall velocity's
    for (DBuf<double>* b : {&adj.zero_e, &adj.lin_vort, &adj.lin_adv, &adj.pvbar}) b->alloc(EK);
    adj.lin_nvel.alloc(EK);
    HIPCHK(hipMemcpy(adj.lin_nvel.p, b_nvel.p, EK * sizeof(double), hipMemcpyDeviceToDevice));
    // homogeneous boundary values: zero psi (null), zero wall velocity and flux; the walls' normal
    // velocity (a constant) multiplies the boundary vorticity's variation
    adj.Bl = B;
    adj.Bl.psi = nullptr;
    adj.Bl.diff = adj.lin_diff; adj.Bl.vjump = adj.lin_vj; adj.Bl.pvel = adj.zero_e;
    adj.Bl.nvel = adj.lin_nvel; adj.Bl.vort = adj.lin_vort; adj.Bl.adv = adj.lin_adv;
    adj.Bz = adj.Bl;
    adj.Bz.diff = adj.zero_e;
    adj.Mv.alloc((size_t)N * 5 * K2 * 2 * K2);
    adj.Md.alloc(EK * K2);
    adj.Ubar.alloc(2 * D); adj.zero_u.alloc(2 * D); adj.zero_tu.alloc(TU); adj.diffbar.alloc(EK);
    adj.zprev.alloc(D);
    // the velocity map psi -> (U, wall flux): K^2 probes per colour of the distance-2 colouring
    // (U of an element depends on psi of its face ring), velocity with homogeneous boundary values
    VelBatch vb;
    vb.psi = D; vb.U = 2 * D; vb.tru = TU; vb.vjump = EK; vb.diff = EK;
    for (int c = 0; c < adj.nc1; ++c) {
      HIPCHK(launch_adj_seed_batch(N, K, adj.col1, c, 1, adj.seed, stream));
      HIPCHK(launch_velocity(K, geo_kind, N, T, G, adj.Bl, adj.seed, nullptr, adj.dU, adj.dtru,
                             1. / (cfg.dt * re_inv), I, stream, K2, vb));
      HIPCHK(launch_adj_assemble_vel(N, E, K, adj.col1, c, d_nb, adj.own_el, adj.dU, adj.lin_diff, adj.Mv, adj.Md,
                                     stream));
    }
    if (adj.seeds_kept) {
      HIPCHK(launch_adj_seed_batch(N, K, adj.col1, 0, adj.nc1, adj.seed, stream));
      HIPCHK(launch_adj_seed_u_batch(N, K, adj.col1, 0, 2 * adj.nc1, T, adj.dU, adj.dtru, stream));
    }
    if (E > 0) HIPCHK(launch_adj_edge_seed_batch(E, K, adj.own_f, adj.pvel_seed, stream));
    HIPCHK(hipStreamSynchronize(stream));
    adj.init = true;
  }

  void dcopy(double* dst, const double* src, size_t n) {
    HIPCHK(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToDevice, stream));
  }

  // One RK4 step from w = omega_n recording every stage's input, velocity and upwind
  // switches (w itself is not advanced).  stage_psi: the stage solutions of the same step kept by
  // the segment's recompute (their inputs are recomputed here by the same kernels), or null to
  // solve.
  void adj_record_step(const double* stage_psi) {
    const double c[4] = {0., 0.5, 0.5, 1.};
    const double cn[3] = {0.5, 0.5, 1.};
    dcopy(adj.ws[0], w, D);
    for (int st = 0; st < 4; ++st) {
      update_bcs(c[st]);
      if (stage_psi) dcopy(psi, stage_psi + (size_t)st * D, D);
      else poisson(adj.ws[st]);
      HIPCHK(launch_velocity(K, geo_kind, N, T, G, B, psi, vel, adj.Us[st], adj.trus[st], 1. / (cfg.dt * re_inv), I,
                             stream));
      StageOut so;
      so.k = kscratch;
      so.sig = adj.sig[st];
      if (st < 3) { so.next = adj.ws[st + 1]; so.c = cn[st]; so.base = w; }
      HIPCHK(launch_stage(K, geo_kind, 1, N, T, G, B, adj.ws[st], adj.Us[st], adj.trus[st], re_inv, cfg.dt, I, so, stream,
                          1));
    }
  }

  // xbar = (dk_s/domega_s)^T lam for recorded stage st, adding (dk_s/dpvel)^T lam to adj.pvbar.
  // The probes of many colours (and the 4K wall-velocity probes) run as one batched launch each.
  void adj_stage(int st, const double* lam, double* xbar, double tau = std::nan("")) {
    const double idr = 1. / (cfg.dt * re_inv);
    const size_t TU = (size_t)4 * N * K, EK = std::max<size_t>((size_t)E * K, 1);
    StageOut so;
    so.k = adj.y;
    so.bs_k = D;
    so.sig = adj.sig[st];
    // (1) omega, with psi (so U and the wall flux) fixed
    so.bs_w = D;
    for (int u0 = 0; u0 < adj.nc1; u0 += adj.ub) {
      const int nu = std::min(adj.ub, adj.nc1 - u0);
      so.nbatch = nu * K2;
      if (!adj.seeds_kept) HIPCHK(launch_adj_seed_batch(N, K, adj.col1, u0, nu, adj.seed, stream));
      HIPCHK(launch_stage(K, geo_kind, 1, N, T, G, adj.Bz, adj.seed, adj.Us[st], adj.trus[st], re_inv, cfg.dt, I, so,
                          stream, 2));
      HIPCHK(launch_adj_dot_batch(N, K2, so.nbatch, lam, adj.y, adj.p, stream));
      HIPCHK(launch_adj_gather_batch(N, K2, 1, u0, nu, adj.col1, adj.r1p, adj.r1i, adj.p, xbar, stream));
    }
    // (2) velocity: a unit per colour and component (the stage depends on U over the face ring),
    //     the stage advecting the recorded vorticity with the seeded velocity
    so.bs_w = 0; so.bs_U = 2 * D; so.bs_tru = TU; so.bs_diff = 0;
    so.adv_only = 1;  // zero vorticity and wall flux for the diffusion term
    for (int u0 = 0; u0 < 2 * adj.nc1; u0 += adj.ub) {
      const int nu = std::min(adj.ub, 2 * adj.nc1 - u0);
      so.nbatch = nu * K2;
      if (!adj.seeds_kept) HIPCHK(launch_adj_seed_u_batch(N, K, adj.col1, u0, nu, T, adj.dU, adj.dtru, stream));
      HIPCHK(launch_stage(K, geo_kind, 1, N, T, G, adj.Bz, adj.ws[st], adj.dU, adj.dtru, re_inv, cfg.dt, I, so, stream,
                          2));
      HIPCHK(launch_adj_dot_batch(N, K2, so.nbatch, lam, adj.y, adj.p, stream));
      HIPCHK(launch_adj_gather_batch(N, K2, 2, u0, nu, adj.col1, adj.r1p, adj.r1i, adj.p, adj.Ubar, stream));
    }
    // (3) wall flux: probe f K + j seeds edge flux point j of the edges owned through face f, which
    //     reaches only the owner elements; then the wall velocity's share of it
    HIPCHK(hipMemsetAsync(adj.diffbar.p, 0, EK * sizeof(double), stream));
    if (E > 0) {
      so.bs_U = 0; so.bs_tru = 0; so.bs_diff = EK;
      so.adv_only = 0;
      so.nbatch = 4 * K;
      HIPCHK(launch_stage(K, geo_kind, 1, N, T, G, adj.Bl_seed(), adj.zero_d, adj.zero_u, adj.zero_tu, re_inv, cfg.dt, I,
                          so, stream, 2));
      HIPCHK(launch_adj_dot_batch(N, K2, 4 * K, lam, adj.y, adj.p, stream));
      HIPCHK(launch_adj_edge_gather_batch(N, E, K, adj.own_el, adj.own_f, adj.p, adj.diffbar, stream));
      HIPCHK(launch_adj_wall(E, K, d_noslip, d_esign, idr, adj.diffbar, adj.pvbar, stream));
    }
    // psi_bar through the assembled velocity map
    HIPCHK(launch_adj_vel_transpose(N, K, d_nb, d_nbf, adj.Mv, adj.Md, adj.Ubar, adj.diffbar, adj.psibar, stream));
    // (4) the Poisson solve: As z = psi_bar (a right-hand side -W b = psi_bar comes from the
    //     vorticity psi_bar / (W J) with zero boundary values), then omega_bar += W J z
    HIPCHK(launch_adj_wj(N, K, tab.wgt, d_jac, adj.psibar, adj.fake, 0, stream));
    if (std::isnan(tau)) {
      adj.zn = 0;
    } else if (adj.zn >= 1 && tau != adj.ztau_a) {
      const double d1 = tau - adj.ztau_a, d2 = adj.ztau_a - adj.ztau_b;
      const bool ok = adj.zn == 2 && d1 * d2 > 0. && std::fabs(d1) <= 1. && std::fabs(d2) <= 1.;
      psi_predict(stream, D, ok ? d1 / d2 : 0., ok ? 1 : 0, adj.z, adj.zprev);
    }
    rhs_bc = adj.zero_e;
    std::swap(psi.p, adj.z.p);
    proj_cur = &proj_adj;
    proj_force = true;
    try {
      poisson(adj.fake);
    } catch (...) {
      std::swap(psi.p, adj.z.p);
      rhs_bc = nullptr;
      proj_cur = &proj_fwd;
      proj_force = false;
      throw;
    }
    std::swap(psi.p, adj.z.p);
    rhs_bc = nullptr;
    proj_cur = &proj_fwd;
    proj_force = false;
    if (!std::isnan(tau) && !(adj.zn >= 1 && tau == adj.ztau_a)) {
      adj.ztau_b = adj.ztau_a;
      adj.ztau_a = tau;
      adj.zn = std::min(adj.zn + 1, 2);
    }
    HIPCHK(launch_adj_wj(N, K, tab.wgt, d_jac, adj.z, xbar, 1, stream));
  }

  // Binomial checkpointing: F(L, s) = the fewest step advances that reverse L steps from a
  // snapshot at the range's start with s free snapshot slots, each step then recorded once:
  // F(1, s) = 0, F(L, 0) = L (L - 1) / 2, F(L, s) = min_d [d + F(L - d, s - 1) + F(d, s)]
  // (advance d steps and snapshot, reverse the tail with one slot less, then the head).  The
  // table of optimal first advances d is built once per (L, s); above kBinoMaxL steps the range
  // is halved instead.
  static constexpr int kBinoMaxL = 2048;
  void binomial_table(int L, int S) {
    if (L <= adj.bsplit_L && S <= adj.bsplit_S) return;
    L = std::min(std::max(L, adj.bsplit_L), kBinoMaxL);
    S = std::max(S, adj.bsplit_S);
    std::vector<int64_t> F((size_t)(L + 1) * (S + 1), 0);
    adj.bsplit.assign((size_t)(L + 1) * (S + 1), 1);
    auto at = [&](int l, int sl) -> int64_t& { return F[(size_t)l * (S + 1) + sl]; };
    for (int l = 1; l <= L; ++l) at(l, 0) = (int64_t)l * (l - 1) / 2;
    for (int sl = 1; sl <= S; ++sl)
      for (int l = 2; l <= L; ++l) {
        int64_t best = INT64_MAX;
        int bd = 1;
        for (int d = 1; d < l; ++d) {
          const int64_t c = d + at(l - d, sl - 1) + at(d, sl);
          if (c < best) { best = c; bd = d; }
        }
        at(l, sl) = best;
        adj.bsplit[(size_t)l * (S + 1) + sl] = bd;
      }
    adj.bsplit_L = L;
    adj.bsplit_S = S;
  }
  int binomial_split(int L, int S) const {
    if (L > adj.bsplit_L || S > adj.bsplit_S) return std::max(1, L / 2);
    return adj.bsplit[(size_t)L * (adj.bsplit_S + 1) + S];
  }
  int snap_take(int pos) {
    for (int i = 0; i < adj.nsnap; ++i)
      if (adj.snap_pos[i] < 0) {
        adj.snap_pos[i] = pos;
        dcopy(adj.snap.p + (size_t)i * D, w, D);
        return i;
      }
    throw StatusError(HOC_EINVAL, "binomial schedule ran out of snapshot slots");
  }
  int snap_find(int pos) const {
    for (int i = 0; i < adj.nsnap; ++i)
      if (adj.snap_pos[i] == pos) return i;
    return -1;
  }

  // Forward run of nsteps RK4 steps recording what the reverse sweep needs (hoc_adjoint_forward):
  //  every >= 1: the vorticity every `every` steps (uniform segments, each recomputed once);
  //  every == 0: the vorticity and the four stage solutions of every step when they fit in half
  //              the free device memory (no recompute), otherwise binomial checkpointing with the
  //              snapshots that fit;
  //  every < 0:  binomial checkpointing with -every vorticity snapshots.
  void adjoint_forward(int nsteps, int every) {
    adjoint_setup();
    if (nsteps < 0) throw StatusError(HOC_EINVAL, "nsteps must be >= 0");
    adj.have_forward = false;
    adj.trajw.alloc(0); adj.trajpsi.alloc(0); adj.snap.alloc(0);
    adj.t0 = time;
    int sched = every >= 1 ? 0 : 2;
    int nsnap = every < 0 ? -every : 0;
    if (every == 0) {
      size_t fr = 0, tot = 0;
      HIPCHK(hipMemGetInfo(&fr, &tot));
      const double budget = 0.5 * (double)fr;
      const double per = (double)D * sizeof(double);
      if (5. * per * std::max(nsteps, 1) <= budget) sched = 1;
      else nsnap = (int)std::min<double>(budget / per, (double)std::max(nsteps, 1));
      if (sched == 2 && nsnap < 1) throw StatusError(HOC_EDEVICE, "no device memory for adjoint snapshots");
    }
    adj.sched = sched;
    if (sched == 0) {
      const int nck = std::max(1, (nsteps + every - 1) / every);
      adj.ckbuf.alloc((size_t)nck * D);
      adj.segbuf.alloc((size_t)std::min(every, std::max(nsteps, 1)) * D);
      adj.segpsi.alloc((size_t)std::min(every, std::max(nsteps, 1)) * 4 * D);
      for (int n = 0; n < nsteps; ++n) {
        if (n % every == 0) dcopy(adj.ckbuf.p + (size_t)(n / every) * D, w, D);
        rk_step();
      }
    } else if (sched == 1) {
      adj.trajw.alloc((size_t)std::max(nsteps, 1) * D);
      adj.trajpsi.alloc((size_t)std::max(nsteps, 1) * 4 * D);
      for (int n = 0; n < nsteps; ++n) {
        dcopy(adj.trajw.p + (size_t)n * D, w, D);
        capture_psi = adj.trajpsi.p + (size_t)n * 4 * D;
        rk_step();
        capture_psi = nullptr;
      }
    } else {
      // snapshot slots: the start and the first descent of the schedule, taken on the way
      nsnap = std::max(1, std::min(nsnap, std::max(nsteps, 1)));
      adj.nsnap = nsnap;
      adj.snap.alloc((size_t)nsnap * D);
      adj.snap_pos.assign(nsnap, -1);
      binomial_table(std::max(nsteps, 1), nsnap - 1);
      snap_take(0);
      int a = 0, free_slots = nsnap - 1;
      int next = (nsteps - a > 1 && free_slots > 0) ? a + binomial_split(nsteps - a, free_slots) : -1;
      for (int n = 0; n < nsteps; ++n) {
        rk_step();
        if (n + 1 == next) {
          snap_take(next);
          a = next;
          --free_slots;
          next = (nsteps - a > 1 && free_slots > 0) ? a + binomial_split(nsteps - a, free_slots) : -1;
        }
      }
    }
    HIPCHK(hipStreamSynchronize(stream));
    adj.nsteps = nsteps;
    adj.every = every;
    adj.have_forward = true;
  }

  // Reverse sweep over the recorded trajectory.  Each step is re-run from its vorticity recording
  // its stages (with the stage solutions kept by the forward run or a recompute, or solving them)
  // and transposed stage by stage:
  //   k4_bar = w_bar/6, k3_bar = k2_bar = w_bar/3, k1_bar = w_bar/6,
  //   for s = 4..1: x = (dk_s/domega_s)^T k_s_bar;  w_bar += x;  k_{s-1}_bar += c_s x
  // with omega_s = omega_n + c_s k_{s-1}, c = (1/2, 1/2, 1).  Uniform segments are recomputed from
  // their checkpoint keeping every step's vorticity and stage solutions; recorded trajectories
  // need no recompute; the binomial schedule advances from its snapshots as it goes.  The
  // handle's state (vorticity, stream function, velocity, time) is restored afterwards.
  void adjoint_backward(const double* wbar_h, double* w0bar_h, double* pvbar_h) {
    if (!adj.have_forward) throw StatusError(HOC_ESTATE, "call hoc_adjoint_forward first");
    adjoint_check();
    const double time_end_ = time;
    dcopy(adj.save_w, w, D);
    dcopy(adj.save_psi, psi, D);
    dcopy(adj.save_vel, vel, 2 * D);
    h2d(adj.wbar.p, wbar_h, D * sizeof(double));
    const size_t EK = std::max<size_t>((size_t)E * K, 1);
    HIPCHK(hipMemsetAsync(adj.pvbar.p, 0, EK * sizeof(double), stream));
    const double cn[3] = {0.5, 0.5, 1.};
    const double cst[4] = {0., 0.5, 0.5, 1.};
    const int every = adj.every, nsteps = adj.nsteps;
    adj.zn = 0;
    proj_adj.m = 0;
    auto restore = [&] {
      dcopy(w, adj.save_w, D);
      dcopy(psi, adj.save_psi, D);
      dcopy(vel, adj.save_vel, 2 * D);
      time = time_end_;
      invalidate_guess();   // the recompute left the histories of the trajectory's early steps
    };
    // w = omega_n on entry
    auto reverse_step = [&](int n, const double* stage_psi) {
      time = adj.t0 + n * cfg.dt;
      adj_record_step(stage_psi);
      HIPCHK(launch_adj_axpby(D, 1. / 6., adj.wbar, 0., adj.kbar[3], stream));
      HIPCHK(launch_adj_axpby(D, 1. / 3., adj.wbar, 0., adj.kbar[2], stream));
      HIPCHK(launch_adj_axpby(D, 1. / 3., adj.wbar, 0., adj.kbar[1], stream));
      HIPCHK(launch_adj_axpby(D, 1. / 6., adj.wbar, 0., adj.kbar[0], stream));
      for (int st = 3; st >= 0; --st) {
        adj_stage(st, adj.kbar[st], adj.xbar, n + cst[st]);
        HIPCHK(launch_adj_axpby(D, 1., adj.xbar, 1., adj.wbar, stream));
        if (st > 0) HIPCHK(launch_adj_axpby(D, cn[st - 1], adj.xbar, 1., adj.kbar[st - 1], stream));
      }
    };
    // binomial schedule: w = omega_{a+d}, advanced from the snapshot at a
    auto advance_from = [&](int a, int d) {
      const int sl = snap_find(a);
      if (sl < 0) throw StatusError(HOC_ESTATE, "binomial schedule lost a snapshot");
      dcopy(w, adj.snap.p + (size_t)sl * D, D);
      time = adj.t0 + a * cfg.dt;
      invalidate_guess();
      for (int i = 0; i < d; ++i) rk_step();
    };
    std::function<void(int, int, int)> rev = [&](int a, int b, int free_slots) {
      if (b <= a) return;
      if (b - a == 1) { advance_from(a, 0); reverse_step(a, nullptr); return; }
      if (free_slots == 0) {
        for (int n = b - 1; n >= a; --n) { advance_from(a, n - a); reverse_step(n, nullptr); }
        return;
      }
      const int d = binomial_split(b - a, free_slots);
      int sl = snap_find(a + d);
      if (sl < 0) { advance_from(a, d); sl = snap_take(a + d); }
      rev(a + d, b, free_slots - 1);
      adj.snap_pos[sl] = -1;
      rev(a, a + d, free_slots);
    };
    try {
      if (adj.sched == 0) {
        const int nseg = (nsteps + every - 1) / every;
        for (int sg = nseg - 1; sg >= 0; --sg) {
          const int n0 = sg * every, n1 = std::min(n0 + every, nsteps);
          dcopy(w, adj.ckbuf.p + (size_t)sg * D, D);
          time = adj.t0 + n0 * cfg.dt;
          invalidate_guess();
          for (int n = n0; n < n1; ++n) {
            dcopy(adj.segbuf.p + (size_t)(n - n0) * D, w, D);
            capture_psi = adj.segpsi.p + (size_t)(n - n0) * 4 * D;
            rk_step();
            capture_psi = nullptr;
          }
          for (int n = n1 - 1; n >= n0; --n) {
            dcopy(w, adj.segbuf.p + (size_t)(n - n0) * D, D);
            reverse_step(n, adj.segpsi.p + (size_t)(n - n0) * 4 * D);
          }
        }
      } else if (adj.sched == 1) {
        for (int n = nsteps - 1; n >= 0; --n) {
          dcopy(w, adj.trajw.p + (size_t)n * D, D);
          reverse_step(n, adj.trajpsi.p + (size_t)n * 4 * D);
        }
      } else {
        rev(0, nsteps, adj.nsnap - 1);
      }
      d2h(w0bar_h, adj.wbar.p, D * sizeof(double));
      if (pvbar_h && E > 0) d2h(pvbar_h, adj.pvbar.p, (size_t)E * K * sizeof(double));
    } catch (...) {
      capture_psi = nullptr;
      restore();
      throw;
    }
    restore();
    HIPCHK(hipStreamSynchronize(stream));
  }

  // (dk/domega)^T lam and (dk/dpvel)^T lam of one stage at time t (hoc_stage_residual's map).
  void stage_vjp(const double* omega_h, double t, const double* lam_h, double* out_h, double* pvbar_h) {
    adjoint_setup();
    proj_adj.m = 0;
    const size_t EK = std::max<size_t>((size_t)E * K, 1);
    h2d(adj.ws[0].p, omega_h, D * sizeof(double));
    h2d(adj.lam.p, lam_h, D * sizeof(double));
    update_bcs(0., t);
    poisson(adj.ws[0]);
    HIPCHK(launch_velocity(K, geo_kind, N, T, G, B, psi, vel, adj.Us[0], adj.trus[0], 1. / (cfg.dt * re_inv), I, stream));
    StageOut so;
    so.k = kscratch;
    so.sig = adj.sig[0];
    HIPCHK(launch_stage(K, geo_kind, 1, N, T, G, B, adj.ws[0], adj.Us[0], adj.trus[0], re_inv, cfg.dt, I, so, stream, 1));
    HIPCHK(hipMemsetAsync(adj.pvbar.p, 0, EK * sizeof(double), stream));
    adj_stage(0, adj.lam, adj.xbar);
    d2h(out_h, adj.xbar.p, D * sizeof(double));
    if (pvbar_h && E > 0) d2h(pvbar_h, adj.pvbar.p, (size_t)E * K * sizeof(double));
  }

  // Boundary flux points [E][K] (edge flux-point order of the boundary arrays), x and y.
  void boundary_points(double* xy) const {
    const int L = mesh.lnod;
    for (int e = 0; e < E; ++e) {
      const auto& nd = mesh.edges[e];
      for (int j = 0; j < K; ++j) {
        double x = 0., y = 0.;
        for (int l = 0; l < L; ++l) {
          x += tab.gsb[l][j] * mesh.xy[2 * (size_t)nd[l]];
          y += tab.gsb[l][j] * mesh.xy[2 * (size_t)nd[l] + 1];
        }
        xy[2 * ((size_t)e * K + j)] = x;
        xy[2 * ((size_t)e * K + j) + 1] = y;
      }
    }
  }

  // Ensemble tables (instance of every element and boundary edge, per-instance Re and dt).
  void setup_instances() {
    I = InstDev{};
    G.inst = nullptr;
    if (n_inst <= 1) return;
    if ((int)inst_off.size() != n_inst + 1 || inst_off[0] != 0 || inst_off[n_inst] != N)
      throw StatusError(HOC_EINVAL, "instance element offsets do not cover the mesh");
    std::vector<int32_t> ei(N), bi(std::max(E, 1), 0);
    for (int i = 0; i < n_inst; ++i) {
      if (inst_off[i + 1] <= inst_off[i]) throw StatusError(HOC_EINVAL, "instance element offsets must increase");
      for (int e = inst_off[i]; e < inst_off[i + 1]; ++e) ei[e] = i;
    }
    // instances must not share faces
    for (int e = 0; e < N; ++e)
      for (int f = 0; f < 4; ++f) {
        const int nb = mesh.nb[(size_t)e * 4 + f];
        if (nb >= 0 && ei[nb] != ei[e]) throw StatusError(HOC_EINVAL, "ensemble instances share a face");
      }
    for (int e = 0; e < E; ++e) bi[e] = ei[mesh.be_elem[e]];
    std::vector<double> ri(n_inst), idr(n_inst);
    for (int i = 0; i < n_inst; ++i) { ri[i] = 1. / inst_re[i]; idr[i] = 1. / (inst_dt[i] * ri[i]); }
    d_inst.upload(ei); d_einst.upload(bi); d_ioff.upload(inst_off);
    d_ireinv.upload(ri); d_idt.upload(inst_dt); d_iidr.upload(idr);
    d_iramp.alloc(n_inst); d_inorm.alloc(n_inst);
    inst_time.assign(n_inst, 0.);
    G.inst = d_inst;
    I = InstDev{d_ireinv, d_idt, d_iidr, d_iramp, d_einst};
  }
};

}  // namespace hoc

using hoc::Solver;

struct hoc_solver {
  Solver s;
};

static std::string g_err;

static int hoc_fail(hoc_t h, int code, const std::string& msg) {
  if (h) h->s.err = msg;
  g_err = msg;
  return code;
}

template <class Fn>
static int guarded(hoc_t h, Fn fn) {
  if (!h) return hoc_fail(nullptr, HOC_EINVAL, "null handle");
  try {
    fn();
  } catch (const hoc::StatusError& e) {
    return hoc_fail(h, e.code, e.what());
  } catch (const hoc::HipError& e) {
    return hoc_fail(h, HOC_EDEVICE, e.what());
  } catch (const std::bad_alloc&) {
    return hoc_fail(h, HOC_EDEVICE, "host allocation failed");
  } catch (const std::exception& e) {
    return hoc_fail(h, HOC_EMESH, e.what());
  }
  return HOC_OK;
}

extern "C" {

void hoc_default_config(hoc_config* c) {
  std::memset(c, 0, sizeof(*c));
  c->K = 3;                      // set_defaults (src/HO_2D.cpp:3699)
  c->problem_type = 11;             // :3702 (the hybrid driver's default)
  c->Re = 1.0;
  c->dt = 1.0;
  c->time_integration_type = 2;  // :3703
  c->advection_type = 2;         // :3704
  c->tol = 1e-15;                // :3067
  c->maxiter = 150;              // :3069
  c->precision = HOC_FP64;
  c->krylov = HOC_KRYLOV_AUTO;
  c->device = 0;
  c->fail_on_noconv = 0;
  c->mixed_inner_tol = 0.;
  c->cheb_degree = 0;
  c->cheb_lower = 0.;
  c->launch_mode = 0;
}

int hoc_create(hoc_t* out, const hoc_config* cfg) {
  if (!out || !cfg) return hoc_fail(nullptr, HOC_EINVAL, "null argument");
  *out = nullptr;
  if (cfg->K < 2 || cfg->K > 6) return hoc_fail(nullptr, HOC_EINVAL, "K must be in 2..6");
  if (cfg->time_integration_type != 1 && cfg->time_integration_type != 2 && cfg->time_integration_type != 4)
    return hoc_fail(nullptr, HOC_EINVAL, "time_integration_type must be 1, 2 or 4");
  if (cfg->advection_type != 1 && cfg->advection_type != 2) return hoc_fail(nullptr, HOC_EINVAL, "advection_type must be 1 or 2");
  if ((cfg->problem_type < 1 || cfg->problem_type > 3) && cfg->problem_type != 11)
    return hoc_fail(nullptr, HOC_EINVAL, "problem_type must be 1, 2, 3 or 11");
  if (cfg->precision != HOC_FP64 && cfg->precision != HOC_MIXED) return hoc_fail(nullptr, HOC_EINVAL, "bad precision");
  if (!(cfg->dt > 0.) || cfg->maxiter < 0 || !(cfg->tol >= 0.)) return hoc_fail(nullptr, HOC_EINVAL, "bad dt/tol/maxiter");
  if (!(cfg->mixed_inner_tol >= 0. && cfg->mixed_inner_tol < 1.)) return hoc_fail(nullptr, HOC_EINVAL, "mixed_inner_tol must be in [0, 1)");
  if (cfg->cheb_degree < 0 || cfg->cheb_degree > hoc::kMaxCheb) return hoc_fail(nullptr, HOC_EINVAL, "cheb_degree must be in 0..8");
  if (!(cfg->cheb_lower >= 0. && cfg->cheb_lower < 1.)) return hoc_fail(nullptr, HOC_EINVAL, "cheb_lower must be in [0, 1)");
  if (cfg->launch_mode < 0 || cfg->launch_mode > 2) return hoc_fail(nullptr, HOC_EINVAL, "launch_mode must be 0, 1 or 2");
  if (cfg->psi_guess < 0 || cfg->psi_guess > 5) return hoc_fail(nullptr, HOC_EINVAL, "psi_guess must be 0..5");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0) return hoc_fail(nullptr, HOC_EDEVICE, "no HIP device");
  if (cfg->device < 0 || cfg->device >= ndev) return hoc_fail(nullptr, HOC_EDEVICE, "device ordinal out of range");
  hoc_t h = new (std::nothrow) hoc_solver();
  if (!h) return hoc_fail(nullptr, HOC_EDEVICE, "allocation failed");
  h->s.cfg = *cfg;
  h->s.device = cfg->device;
  *out = h;
  return HOC_OK;
}

int hoc_load_mesh(hoc_t h, int32_t lnod, int32_t n_nodes, const double* xy, int32_t n_elem, const int32_t* elem_nodes,
                  int32_t n_bedges, const int32_t* bedge_nodes, const int32_t* bedge_bdry, int32_t n_bdry,
                  const char* bdry_names) {
  return guarded(h, [&] {
    Solver& s = h->s;
    if (lnod < 2 || lnod > 4) throw hoc::StatusError(HOC_EINVAL, "lnod must be 2, 3 or 4");
    if (n_nodes <= 0 || n_elem <= 0 || n_bedges < 0 || n_bdry < 0 || !xy || !elem_nodes)
      throw hoc::StatusError(HOC_EINVAL, "empty mesh");
    if (n_bedges > 0 && (!bedge_nodes || !bedge_bdry)) throw hoc::StatusError(HOC_EINVAL, "missing boundary arrays");
    hoc::Mesh m;
    m.lnod = lnod; m.n_nodes = n_nodes; m.n_elem = n_elem; m.n_bedges = n_bedges;
    m.xy.assign(xy, xy + 2 * (size_t)n_nodes);
    m.elem.assign(elem_nodes, elem_nodes + (size_t)n_elem * lnod * lnod);
    m.edges.resize(n_bedges);
    for (int e = 0; e < n_bedges; ++e) m.edges[e].assign(bedge_nodes + (size_t)e * lnod, bedge_nodes + (size_t)(e + 1) * lnod);
    m.bedge_bdry.assign(bedge_bdry, bedge_bdry + n_bedges);
    std::string names(bdry_names ? bdry_names : "");
    size_t p0 = 0;
    for (int b = 0; b < n_bdry; ++b) {
      size_t p1 = names.find('\n', p0);
      m.bnames.push_back(names.substr(p0, p1 == std::string::npos ? std::string::npos : p1 - p0));
      p0 = p1 == std::string::npos ? names.size() : p1 + 1;
    }
    s.accept_mesh(std::move(m));
  });
}

int hoc_load_gmsh(hoc_t h, const char* path, int32_t occ) {
  return guarded(h, [&] {
    if (!path) throw hoc::StatusError(HOC_EINVAL, "null path");
    hoc::Mesh m;
    try {
      hoc::read_gmsh41(path, occ, m);
    } catch (const std::runtime_error& e) {
      throw hoc::StatusError(HOC_EMESH, e.what());
    }
    h->s.accept_mesh(std::move(m));
  });
}

int hoc_set_instances(hoc_t h, int32_t n_inst, const int32_t* elem_offsets, const double* Re, const double* dt) {
  return guarded(h, [&] {
    Solver& s = h->s;
    if (!s.mesh_loaded) throw hoc::StatusError(HOC_ESTATE, "hoc_set_instances before hoc_load_mesh");
    if (n_inst < 1 || !elem_offsets || !Re || !dt) throw hoc::StatusError(HOC_EINVAL, "bad instance arrays");
    if (elem_offsets[0] != 0 || elem_offsets[n_inst] != s.mesh.n_elem)
      throw hoc::StatusError(HOC_EINVAL, "instance element offsets must run from 0 to n_elem");
    for (int i = 0; i < n_inst; ++i) {
      if (elem_offsets[i + 1] <= elem_offsets[i]) throw hoc::StatusError(HOC_EINVAL, "instance element offsets must increase");
      if (!(Re[i] > 1e-3) || !(dt[i] > 0.)) throw hoc::StatusError(HOC_EINVAL, "instance Re must exceed 1e-3 and dt be positive");
    }
    s.n_inst = n_inst;
    s.inst_off.assign(elem_offsets, elem_offsets + n_inst + 1);
    s.inst_re.assign(Re, Re + n_inst);
    s.inst_dt.assign(dt, dt + n_inst);
    s.ready = false;
  });
}

int hoc_setup(hoc_t h) {
  return guarded(h, [&] {
    if (!h->s.mesh_loaded) throw hoc::StatusError(HOC_ESTATE, "hoc_setup before hoc_load_mesh");
    h->s.setup();
  });
}

#define NEED_READY(h) if (!h->s.ready) throw hoc::StatusError(HOC_ESTATE, "call hoc_setup first")
#define NEED_LEN(len, want) if ((len) != (int64_t)(want)) throw hoc::StatusError(HOC_EINVAL, "length mismatch")

int hoc_set_boundary_values(hoc_t h, int32_t n_bedges, const int32_t* nval, const double* vals) {
  return guarded(h, [&] {
    Solver& s = h->s;
    if (!s.mesh_loaded) throw hoc::StatusError(HOC_ESTATE, "hoc_set_boundary_values before hoc_load_mesh");
    if (n_bedges != s.mesh.n_bedges || !nval || !vals) throw hoc::StatusError(HOC_EINVAL, "length mismatch");
    s.edge_nvel_in.assign(n_bedges, 0.);
    s.edge_has_nvel.assign(n_bedges, 0);
    for (int e = 0; e < n_bedges; ++e) {  // arrays_to_boundary (src/HO_2D.cpp:3779-3793, 3806-3814)
      if (nval[e] < 0 || nval[e] > 2) throw hoc::StatusError(HOC_EINVAL, "values per edge must be 0, 1 or 2");
      if (nval[e] == 1) s.edge_nvel_in[e] = vals[2 * (size_t)e];
      if (nval[e] == 2) s.edge_nvel_in[e] = vals[2 * (size_t)e + 1];
      s.edge_has_nvel[e] = nval[e] > 0;
    }
    s.ready = false;
  });
}

int64_t hoc_open_point_count(hoc_t h) {
  return (h && h->s.ready && h->s.cfg.problem_type == 11) ? (int64_t)h->s.open_edges.size() * h->s.K : 0;
}

int hoc_get_open_points(hoc_t h, int64_t len, double* xy) {
  return guarded(h, [&] {
    NEED_READY(h); h->s.need_hybrid(); NEED_LEN(len, 2 * hoc_open_point_count(h));
    h->s.open_points(xy);
  });
}

int hoc_set_open_velocities(hoc_t h, int64_t len, const double* uv) {
  return guarded(h, [&] {
    NEED_READY(h); h->s.need_hybrid(); NEED_LEN(len, 2 * hoc_open_point_count(h));
    h->s.set_open_velocities(uv);
  });
}

int hoc_set_open_vorticity(hoc_t h, int64_t len, const double* w) {
  return guarded(h, [&] {
    NEED_READY(h); h->s.need_hybrid(); NEED_LEN(len, hoc_open_point_count(h));
    h->s.set_open_vorticity(w);
  });
}

int hoc_set_vorticity_target(hoc_t h, int64_t len, const double* w) {
  return guarded(h, [&] {
    NEED_READY(h); h->s.need_hybrid(); NEED_LEN(len, h->s.D);
    h->s.set_vorticity_target(w);
  });
}

int hoc_set_p2g_weights(hoc_t h, int64_t len, const double* w) {
  return guarded(h, [&] {
    NEED_READY(h); h->s.need_hybrid(); NEED_LEN(len, h->s.D);
    h->s.h2d(h->s.d_hwgt.p, w, h->s.D * sizeof(double));
  });
}

int hoc_get_instance_times(hoc_t h, int32_t n_inst, double* t) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    if (n_inst != s.n_inst || !t) throw hoc::StatusError(HOC_EINVAL, "length mismatch");
    if (s.n_inst == 1) t[0] = s.time;
    else std::copy(s.inst_time.begin(), s.inst_time.end(), t);
  });
}


int hoc_set_vorticity(hoc_t h, int64_t len, const double* w) {
  return guarded(h, [&] {
    NEED_READY(h); NEED_LEN(len, h->s.D);
    h->s.h2d(h->s.w.p, w, h->s.D * sizeof(double));
    h->s.invalidate_guess();
  });
}
int hoc_get_vorticity(hoc_t h, int64_t len, double* w) {
  return guarded(h, [&] {
    NEED_READY(h); NEED_LEN(len, h->s.D);
    h->s.d2h(w, h->s.w.p, h->s.D * sizeof(double));
  });
}
int hoc_get_streamfunction(hoc_t h, int64_t len, double* p) {
  return guarded(h, [&] {
    NEED_READY(h); NEED_LEN(len, h->s.D);
    h->s.d2h(p, h->s.psi.p, h->s.D * sizeof(double));
  });
}
int hoc_set_streamfunction(hoc_t h, int64_t len, const double* p) {
  return guarded(h, [&] {
    NEED_READY(h); NEED_LEN(len, h->s.D);
    h->s.h2d(h->s.psi.p, p, h->s.D * sizeof(double));
    h->s.invalidate_guess();
  });
}
int hoc_get_velocity(hoc_t h, int64_t len, double* uv) {
  return guarded(h, [&] {
    NEED_READY(h); NEED_LEN(len, 2 * h->s.D);
    h->s.d2h(uv, h->s.vel.p, 2 * h->s.D * sizeof(double));
  });
}
int hoc_get_solution_points(hoc_t h, int64_t len, double* xy) {
  return guarded(h, [&] {
    NEED_READY(h); NEED_LEN(len, 2 * h->s.D);
    std::vector<double> pts;
    hoc::solution_points(h->s.mesh, h->s.tab, pts);
    std::memcpy(xy, pts.data(), pts.size() * sizeof(double));
  });
}
int hoc_get_solution_areas(hoc_t h, int64_t len, double* a) {
  return guarded(h, [&] {
    NEED_READY(h); NEED_LEN(len, h->s.D);
    Solver& s = h->s;
    for (int el = 0; el < s.N; ++el)
      for (int j = 0; j < s.K; ++j)
        for (int k = 0; k < s.K; ++k) {
          size_t v = (size_t)el * s.K2 + j * s.K + k;
          a[v] = s.tab.wgt[j] * s.tab.wgt[k] * s.geo.jac[v];  // src/HO_2D.cpp:3988
        }
  });
}
int hoc_get_node_fields(hoc_t h, int32_t refresh, int32_t n_nodes, double* out) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    if (n_nodes != s.mesh.n_nodes || !out) throw hoc::StatusError(HOC_EINVAL, "n_nodes must be the mesh's node count");
    s.node_fields(refresh != 0);
    s.d2h(out, s.d_nodeout.p, (size_t)n_nodes * 4 * sizeof(double));
  });
}

int hoc_write_smooth_vtk(hoc_t h, int32_t refresh, const char* path) {
  return guarded(h, [&] {
    NEED_READY(h);
    if (!path) throw hoc::StatusError(HOC_EINVAL, "null path");
    Solver& s = h->s;
    s.node_fields(refresh != 0);
    std::vector<double> nodes((size_t)s.mesh.n_nodes * 4);
    s.d2h(nodes.data(), s.d_nodeout.p, nodes.size() * sizeof(double));
    try {
      hoc::write_vtk_nodes(path, s.mesh, nodes.data());
    } catch (const std::runtime_error& e) {
      throw hoc::StatusError(HOC_EINVAL, e.what());
    }
  });
}

int hoc_set_sample_points(hoc_t h, int32_t n, const double* xy) {
  return guarded(h, [&] {
    NEED_READY(h);
    if (n < 0 || (n > 0 && !xy)) throw hoc::StatusError(HOC_EINVAL, "bad sample point array");
    for (int32_t i = 0; i < 2 * n; ++i)
      if (!std::isfinite(xy[i])) throw hoc::StatusError(HOC_EINVAL, "non-finite sample point coordinate");
    h->s.set_sample_points(n, xy);
  });
}

int hoc_get_sample_location(hoc_t h, int32_t n, int32_t* elem, double* local_xy) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    if (n != s.n_sp) throw hoc::StatusError(HOC_EINVAL, "n must be the number of sample points set");
    if (elem) std::copy(s.sp_elem.begin(), s.sp_elem.end(), elem);
    if (local_xy) std::copy(s.sp_loc.begin(), s.sp_loc.end(), local_xy);
  });
}

int hoc_get_sample_values(hoc_t h, int32_t refresh, int32_t n, double* out) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    if (n != s.n_sp || (n > 0 && !out)) throw hoc::StatusError(HOC_EINVAL, "n must be the number of sample points set");
    s.sample_values(refresh != 0, out);
  });
}

int hoc_write_samples(hoc_t h, int32_t refresh, const char* path) {
  return guarded(h, [&] {
    NEED_READY(h);
    if (!path) throw hoc::StatusError(HOC_EINVAL, "null path");
    Solver& s = h->s;
    std::vector<double> vals(3 * (size_t)s.n_sp);
    s.sample_values(refresh != 0, vals.data());
    try {
      hoc::write_samples(path, s.n_sp, s.sp_xy.data(), vals.data());
    } catch (const std::runtime_error& e) {
      throw hoc::StatusError(HOC_EINVAL, e.what());
    }
  });
}

int hoc_write_vtk(hoc_t h, const char* path) {
  return guarded(h, [&] {
    NEED_READY(h);
    if (!path) throw hoc::StatusError(HOC_EINVAL, "null path");
    Solver& s = h->s;
    std::vector<double> pts, w(s.D), p(s.D), uv(2 * s.D), u(s.D), v(s.D);
    hoc::solution_points(s.mesh, s.tab, pts);
    s.d2h(w.data(), s.w.p, s.D * sizeof(double));
    s.d2h(p.data(), s.psi.p, s.D * sizeof(double));
    s.d2h(uv.data(), s.vel.p, 2 * s.D * sizeof(double));
    for (size_t i = 0; i < s.D; ++i) { u[i] = uv[2 * i]; v[i] = uv[2 * i + 1]; }
    const char* names[4] = {"vorticity", "streamfunction", "u", "v"};
    const double* fields[4] = {w.data(), p.data(), u.data(), v.data()};
    try {
      hoc::write_vtk_sps(path, s.K, s.N, pts.data(), 4, names, fields);
    } catch (const std::runtime_error& e) {
      throw hoc::StatusError(HOC_EINVAL, e.what());
    }
  });
}

double hoc_get_time(hoc_t h) { return h ? h->s.time : 0.; }
int hoc_set_time(hoc_t h, double t) {
  return guarded(h, [&] {
    h->s.time = t;
    std::fill(h->s.inst_time.begin(), h->s.inst_time.end(), t);
  });
}

int hoc_step(hoc_t h, int32_t nsteps) {
  return guarded(h, [&] {
    NEED_READY(h);
    if (nsteps < 0) throw hoc::StatusError(HOC_EINVAL, "nsteps < 0");
    for (int i = 0; i < nsteps; ++i) h->s.rk_step();
    HIPCHK(hipStreamSynchronize(h->s.stream));
  });
}

int hoc_solveto(hoc_t h, double outer_dt, int32_t nsub, int32_t integ, double Re) {
  return guarded(h, [&] {
    NEED_READY(h);
    if (nsub <= 0 || !(outer_dt > 0.)) throw hoc::StatusError(HOC_EINVAL, "bad outer_dt/nsub");
    if (integ != 1 && integ != 2 && integ != 4) throw hoc::StatusError(HOC_EINVAL, "integ must be 1, 2 or 4");
    if (!(Re > 0.)) throw hoc::StatusError(HOC_EINVAL, "Re must be positive");
    Solver& s = h->s;
    if (s.n_inst > 1) throw hoc::StatusError(HOC_EINVAL, "hoc_solveto sets one dt and Re: not for an ensemble");
    s.cfg.dt = outer_dt / (double)nsub;   // src/HO_2D.cpp:4199
    s.cfg.time_integration_type = integ;  // :4203
    s.re_inv = 1.0 / Re;                  // :4204
    s.time_start = s.time_end;            // :4208-4211
    s.time = s.time_start;
    s.time_end += outer_dt;
    for (int i = 0; i < nsub; ++i) s.rk_step();
    HIPCHK(hipStreamSynchronize(s.stream));
  });
}

int hoc_poisson(hoc_t h, const double* omega, double t, double* psi_out) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    s.h2d(s.kscratch.p, omega, s.D * sizeof(double));
    s.update_bcs(0., t);
    s.poisson(s.kscratch);
    s.d2h(psi_out, s.psi.p, s.D * sizeof(double));
  });
}

int hoc_stage_residual(hoc_t h, const double* omega, double t, double* k) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    s.h2d(s.vort.p, omega, s.D * sizeof(double));
    hoc::StageOut so;
    so.k = s.kscratch;
    s.update_bcs(0., t);
    s.stage_body(s.vort, so);
    s.d2h(k, s.kscratch.p, s.D * sizeof(double));
  });
}

int64_t hoc_boundary_point_count(hoc_t h) { return h && h->s.mesh_loaded ? (int64_t)h->s.E * h->s.K : 0; }

int hoc_get_boundary_points(hoc_t h, int64_t len, double* xy) {
  return guarded(h, [&] {
    NEED_READY(h);
    NEED_LEN(len, 2 * (int64_t)h->s.E * h->s.K);
    h->s.boundary_points(xy);
  });
}

int hoc_get_wall_velocity(hoc_t h, int64_t len, double* v) {
  return guarded(h, [&] {
    NEED_READY(h);
    NEED_LEN(len, (int64_t)h->s.E * h->s.K);
    if (len) h->s.d2h(v, h->s.b_pvel0.p, len * sizeof(double));
  });
}

int hoc_set_wall_velocity(hoc_t h, int64_t len, const double* v) {
  return guarded(h, [&] {
    NEED_READY(h);
    NEED_LEN(len, (int64_t)h->s.E * h->s.K);
    for (int64_t i = 0; i < len; ++i)
      if (!std::isfinite(v[i])) throw hoc::StatusError(HOC_EINVAL, "wall velocity must be finite");
    if (len) h->s.h2d(h->s.b_pvel0.p, v, len * sizeof(double));
  });
}

int hoc_adjoint_forward(hoc_t h, int32_t nsteps, int32_t checkpoint_every) {
  return guarded(h, [&] {
    NEED_READY(h);
    h->s.adjoint_forward(nsteps, checkpoint_every);
  });
}

int hoc_adjoint_backward(hoc_t h, int64_t len, const double* wbar_final, double* wbar_initial, int64_t len_wall,
                         double* wall_velocity_bar) {
  return guarded(h, [&] {
    NEED_READY(h);
    NEED_LEN(len, h->s.D);
    if (wall_velocity_bar) NEED_LEN(len_wall, (int64_t)h->s.E * h->s.K);
    if (!wbar_final || !wbar_initial) throw hoc::StatusError(HOC_EINVAL, "null buffer");
    h->s.adjoint_backward(wbar_final, wbar_initial, wall_velocity_bar);
  });
}

int hoc_stage_residual_vjp(hoc_t h, const double* omega, double t, const double* lam, double* omega_bar,
                           double* wall_velocity_bar) {
  return guarded(h, [&] {
    NEED_READY(h);
    if (!omega || !lam || !omega_bar) throw hoc::StatusError(HOC_EINVAL, "null buffer");
    h->s.stage_vjp(omega, t, lam, omega_bar, wall_velocity_bar);
  });
}

// y = A x on device buffers (distinct) in one launch on a stream.
static void apply_plain(Solver& s, const double* x, double* y, hipStream_t st) {
  hoc::FineArgs<double> A;
  A.x = x;
  A.y = y;
  HIPCHK(hoc::launch_fine(s.K, s.geo_kind, hoc::IN_X, hoc::EPI_PLAIN, s.P64.T, s.P64.G, A, st));
}

int hoc_apply_laplacian(hoc_t h, const double* x, double* y) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    s.h2d(s.P64.z.p, x, s.D * sizeof(double));
    apply_plain(s, s.P64.z.p, s.P64.q.p, s.stream);
    s.d2h(y, s.P64.q.p, s.D * sizeof(double));
  });
}

int hoc_apply_laplacian_device(hoc_t h, const double* x, double* y, void* stream) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    if (!x || !y) throw hoc::StatusError(HOC_EINVAL, "null buffer");
    if (x == y) throw hoc::StatusError(HOC_EINVAL, "x and y must not alias");
    const size_t need = (size_t)s.N * 8 * s.K * sizeof(double);
    if (need > hoc::kNoAllocMaxTraceBytes)
      throw hoc::StatusError(HOC_EINVAL, "mesh too large for the no-allocation apply: its face traces would need " +
                                             std::to_string(need) + " bytes, the limit is " +
                                             std::to_string(hoc::kNoAllocMaxTraceBytes));
    HIPCHK(hipSetDevice(s.device));
    apply_plain(s, x, y, stream ? static_cast<hipStream_t>(stream) : s.stream);
  });
}

int hoc_stats_get(hoc_t h, hoc_stats* st) {
  return guarded(h, [&] {
    Solver& s = h->s;
    std::memset(st, 0, sizeof(*st));
    st->n_elem = s.N; st->n_dofs = (int64_t)s.D; st->n_bedges = s.E;
    st->n_levels = (int32_t)(s.mixed ? s.P32.lv.levels() : s.P64.lv.levels()) + 1;
    st->last_refinements = s.last_outer;
    st->precision = s.cfg.precision;
    st->n_nodes = s.mesh.n_nodes;
    st->launch_graphs = s.use_graphs ? 1 : 0;
    st->launch_tune_ratio = s.launch_tune_ratio;
    st->krylov = s.krylov;
    st->last_iters = s.last_iters;
    st->last_rel_residual = s.last_rel;
    st->total_iters = s.total_iters;
    st->n_solves = s.n_solves;
    st->setup_seconds = s.setup_seconds;
    st->fine_op_bytes = s.ready ? s.lap_bytes(hoc::IN_X, hoc::EPI_STORE) : 0.;
  });
}

int hoc_profile_enable(hoc_t h, int32_t on) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    s.prof_flush();
    if (on && s.prof.e0.empty()) {
      const int cap = 4096;
      s.prof.e0.resize(cap); s.prof.e1.resize(cap); s.prof.var.resize(cap); s.prof.nbytes.resize(cap);
      for (int i = 0; i < cap; ++i) { HIPCHK(hipEventCreate(&s.prof.e0[i])); HIPCHK(hipEventCreate(&s.prof.e1[i])); }
      s.prof.ran.alloc(cap);
    }
    if (on) {
      for (int v = 0; v < HOC_PROF_VARIANTS; ++v) { s.prof.ms[v] = 0.; s.prof.cnt[v] = 0; s.prof.bytes[v] = 0.; }
      s.prof.skipped = 0;
    }
    s.prof.on = on != 0;
    s.prof.every = on > 1 ? on : 1;
    s.prof.seen = 0;
  });
}

// Algorithmic bytes of a profile entry that has no launches yet.
static double prof_bytes(const Solver& s, int variant, double vb) {
  using namespace hoc;
  const int in[5] = {IN_X, IN_X, IN_X, IN_PROL, IN_X}, epi[5] = {EPI_STORE, EPI_RESID, EPI_SMOOTH, EPI_SMOOTH, EPI_RESTRICT};
  return s.lap_bytes(in[variant], epi[variant], vb, vb);
}
int hoc_profile_get(hoc_t h, hoc_kernel_profile* p) {
  return guarded(h, [&] {
    NEED_READY(h);
    Solver& s = h->s;
    s.prof_flush();
    static const char* names[HOC_PROF_VARIANTS] = {"lap_apply",     "lap_residual",     "lap_cheb",     "lap_cheb_first",
                                                   "lap_restrict",  "lap_apply_f32",    "lap_residual_f32", "lap_cheb_f32",
                                                   "lap_cheb_first_f32", "lap_restrict_f32"};
    std::memset(p, 0, sizeof(*p));
    for (int v = 0; v < HOC_PROF_VARIANTS; ++v) {
      p->launches[v] = s.prof.cnt[v];
      p->total_ms[v] = s.prof.ms[v];
      const int half = HOC_PROF_VARIANTS / 2;
      p->bytes_per_launch[v] = s.prof.cnt[v] > 0 ? s.prof.bytes[v] / (double)s.prof.cnt[v]
                                                 : prof_bytes(s, v < half ? v : v - half, v < half ? 8. : 4.);
      std::strncpy(p->names[v], names[v], sizeof(p->names[v]) - 1);
    }
    p->noop_launches = s.prof.skipped;
  });
}

const char* hoc_last_error(hoc_t h) { return h ? h->s.err.c_str() : g_err.c_str(); }

void hoc_destroy(hoc_t h) {
  if (!h) return;
  (void)hipSetDevice(h->s.device);
  if (h->s.stream) (void)hipStreamSynchronize(h->s.stream);
  delete h;
}

}  // extern "C"
