// hierarchy_check.cpp - CPU check of what the set-up makes for the Poisson V-cycle (hoc_host.cpp):
//   * build_vhierarchy on bilinear stiffness matrices (square and stretched cells): level shapes, column
//     indices, and the cycle replayed from the packed matrices with bounds-checked vectors laid out as the
//     device's ([f_l; u_{l+1}] per level): linear, symmetric and a contraction; and on random directed
//     patterns, where it must end at coarse_enough unknowns or at a level without coarse ones;
//   * sell_pack against the CSR product, for every number of lanes and rows around a slice's;
//   * dense_inverse with zeros on the diagonal (pivoting), and with a singular direction;
//   * fine_tables: S^T W S = 1 and the eigenvalues' signs for all pairs of end kinds.
// Prints "OK" and exits 0 on success.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <random>
#include <stdexcept>
#include <vector>

#include "hoc_host.hpp"

using namespace hoc;
using Vec = std::vector<double>;

static std::mt19937_64 rng(11);
static double uni() { return std::uniform_real_distribution<double>(-1., 1.)(rng); }
static void need(bool ok, const char* what) {
  if (!ok) throw std::runtime_error(what);
}

// kron(T, M) + r kron(M, T): T = tridiag(-1, 2, -1), M = tridiag(1, 4, 1) / 6, Dirichlet
static CSR stiffness(int g, double r) {
  const double T[3] = {-1., 2., -1.}, M[3] = {1. / 6., 4. / 6., 1. / 6.};
  CSR A;
  A.n = A.m = g * g;
  A.ptr.push_back(0);
  for (int y = 0; y < g; ++y)
    for (int x = 0; x < g; ++x) {
      for (int dy = -1; dy <= 1; ++dy)
        for (int dx = -1; dx <= 1; ++dx) {
          if (y + dy < 0 || y + dy >= g || x + dx < 0 || x + dx >= g) continue;
          A.col.push_back((y + dy) * g + x + dx);
          A.val.push_back(T[dy + 1] * M[dx + 1] + r * M[dy + 1] * T[dx + 1]);
        }
      A.ptr.push_back((int)A.col.size());
    }
  return A;
}

static Vec product(const CSR& A, const Vec& x) {
  Vec y(A.n, 0.);
  for (int i = 0; i < A.n; ++i)
    for (int j = A.ptr[i]; j < A.ptr[i + 1]; ++j) y[i] += A.val[j] * x.at(A.col[j]);
  return y;
}

// y = A x as k_sell reads the packing
struct Sell {
  int n, lanes;
  std::vector<int32_t> off, col;
  Vec val;
  Sell(const CSR& A, int l) : n(A.n), lanes(l) {
    csr_check(A);
    sell_pack(A, l, off, col, val);
    for (int32_t c : col) need(c >= 0 && c < A.m, "packed column");
  }
  void apply(const double* x, size_t nx, double* y) const {
    const int R = 64 / lanes;
    for (int i = 0; i < n; ++i) {
      double s = 0.;
      for (int lane = (i % R) * lanes; lane < (i % R + 1) * lanes; ++lane)
        for (int q = off.at(i / R) + lane; q < off.at(i / R + 1); q += 64) {
          need((size_t)col.at(q) < nx, "read past the vector");
          s += val.at(q) * x[col[q]];
        }
      y[i] = s;
    }
  }
};

struct Cycle {
  std::vector<Sell> Rt, U;
  std::vector<Vec> fu;
  Vec inv, fc;
  explicit Cycle(const VHierarchy& H) {
    for (const VLevel& l : H.levels) {
      Rt.emplace_back(l.Rt, sell_lanes(l.Rt));
      U.emplace_back(l.U, sell_lanes(l.U));
      fu.emplace_back(l.U.m, 0.);
    }
    dense_inverse(H.coarse, inv);
    fc.assign(H.coarse.n, 0.);
  }
  Vec operator()(const Vec& f) {
    const size_t n = Rt.size();
    std::copy(f.begin(), f.end(), n ? fu[0].begin() : fc.begin());
    for (size_t l = 0; l < n; ++l) Rt[l].apply(fu[l].data(), fu[l].size(), l + 1 < n ? fu[l + 1].data() : fc.data());
    const size_t nc = fc.size();
    Vec u(f.size()), uc(nc, 0.);
    for (size_t i = 0; i < nc; ++i)
      for (size_t j = 0; j < nc; ++j) uc[i] += inv[i * nc + j] * fc[j];
    if (n == 0) return uc;
    std::copy(uc.begin(), uc.end(), fu[n - 1].begin() + U[n - 1].n);
    for (size_t l = n; l-- > 0;)
      U[l].apply(fu[l].data(), fu[l].size(), l ? fu[l - 1].data() + U[l - 1].n : u.data());
    return u;
  }
};

static void shapes(const CSR& A, const VHierarchy& H, int enough) {
  int n = A.n;
  for (const VLevel& l : H.levels) {
    const int nc = l.Rt.n;
    need(l.U.n == n && l.Rt.m == n && l.U.m == n + nc && nc < n, "level shapes");
    csr_check(l.Rt);
    csr_check(l.U);
    n = nc;
  }
  need(H.coarse.n == n && n <= enough, "coarsest size");
}

static void check_hierarchy(int g, double r, double rho_max) {
  const CSR A = stiffness(g, r);
  VHierarchy H;
  build_vhierarchy(A, 60, H);
  shapes(A, H, 60);
  Cycle B(H);
  const size_t n = A.n;
  Vec f1(n), f2(n), f3(n);
  for (size_t i = 0; i < n; ++i) { f1[i] = uni(); f2[i] = uni(); f3[i] = 0.3 * f1[i] - 1.7 * f2[i]; }
  const Vec u1 = B(f1), u2 = B(f2), u3 = B(f3);
  double lin = 0., nrm = 0., a = 0., b = 0., sa = 0.;
  for (size_t i = 0; i < n; ++i) {
    const double e = u3[i] - (0.3 * u1[i] - 1.7 * u2[i]);
    lin += e * e; nrm += u3[i] * u3[i];
    a += f2[i] * u1[i]; b += f1[i] * u2[i]; sa += std::fabs(f2[i] * u1[i]);
  }
  need(lin <= 1e-24 * nrm, "cycle is not linear");
  need(std::fabs(a - b) <= 1e-11 * sa, "cycle is not symmetric");
  Vec e = f1;  // error of x <- x + B (0 - A x)
  double rho = 0., last = 1.;
  for (int it = 0; it < 20; ++it) {
    const Vec z = B(product(A, e));
    double s = 0.;
    for (size_t i = 0; i < n; ++i) { e[i] -= z[i]; s += e[i] * e[i]; }
    rho = std::sqrt(s) / last;
    for (double& v : e) v /= std::sqrt(s);
    last = 1.;
  }
  std::printf("%d x %d, ratio %g: %zu levels, coarsest %d, contraction %.3f\n", g, g, r, H.levels.size(), H.coarse.n, rho);
  need(rho <= rho_max, "cycle does not contract");
}

static void check_patterns() {
  for (int t = 0; t < 200; ++t) {
    const int n = 30 + (int)(rng() % 200), deg = (int)(rng() % 6);
    CSR A;
    A.n = A.m = n;
    A.ptr.push_back(0);
    for (int i = 0; i < n; ++i) {
      A.col.push_back(i);
      A.val.push_back(1. + deg);
      for (int d = 0; d < deg; ++d) {  // directed, of widely varying size, some positive
        const int c = t % 2 ? (int)(rng() % n) : std::max(0, i - 1 - (int)(rng() % 9));
        if (std::find(A.col.begin() + A.ptr[i], A.col.end(), c) != A.col.end()) continue;
        A.col.push_back(c);
        A.val.push_back(-std::pow(10., 2. * uni() - 1.) * (rng() % 8 ? 1. : -1.));
      }
      A.ptr.push_back((int)A.col.size());
    }
    VHierarchy H;
    build_vhierarchy(A, 10, H);
    shapes(A, H, 10);
  }
}

static void check_sell() {
  for (int lanes : {4, 8, 16})
    for (int n : {1, 64 / lanes - 1, 64 / lanes, 64 / lanes + 1, 131}) {
      CSR A;
      A.n = n;
      A.m = 97;
      A.ptr.push_back(0);
      for (int i = 0; i < n; ++i) {
        const int len = i % 7 == 3 ? 0 : i == n / 2 ? 90 : (int)(rng() % 20);
        for (int c = 0; c < len; ++c) { A.col.push_back((c * 31 + i) % 97); A.val.push_back(uni()); }
        A.ptr.push_back((int)A.col.size());
      }
      Vec x(A.m), y(n);
      for (double& v : x) v = uni();
      Sell(A, lanes).apply(x.data(), x.size(), y.data());
      const Vec want = product(A, x);
      for (int i = 0; i < n; ++i) need(std::fabs(y[i] - want[i]) <= 90 * 2.3e-16 * 90, "packed product");
    }
}

static void check_dense() {
  for (int n : {1, 2, 33}) {
    CSR A;
    A.n = A.m = n + 1;  // the last row and column are zero
    A.ptr.push_back(0);
    for (int i = 0; i < n; ++i) {
      for (int j = 0; j < n; ++j) {
        if (n > 1 && i == j) continue;
        A.col.push_back(j);
        A.val.push_back(n == 1 ? 2. : j == (i + 1) % n ? 4. : uni() / n);
      }
      A.ptr.push_back((int)A.col.size());
    }
    A.ptr.push_back(A.ptr.back());
    Vec inv;
    dense_inverse(A, inv);
    Vec x(n + 1, 0.);
    for (int i = 0; i < n; ++i) x[i] = uni();
    const Vec b = product(A, x);
    for (int i = 0; i < n; ++i) {
      double s = 0.;
      for (int j = 0; j < n; ++j) s += inv[(size_t)i * (n + 1) + j] * b[j];
      need(std::fabs(s - x[i]) <= 1e-12, "dense inverse");
    }
  }
}

static void check_tables() {
  for (int K = 2; K <= 6; ++K) {
    Tables t;
    build_tables(K, 2, t);
    FineTables f;
    fine_tables(t, f);
    for (int code = 0; code < 9; ++code) {
      const double *lam = &f.fdm[(size_t)code * (K + K * K)], *S = lam + K;
      double lmax = 0., lmin = 1e300;
      for (int a = 0; a < K; ++a) {
        lmax = std::max(lmax, lam[a]);
        lmin = std::min(lmin, lam[a]);
        for (int b = 0; b < K; ++b) {
          double s = 0.;
          for (int i = 0; i < K; ++i) s += S[i * K + a] * t.wgt[i] * S[i * K + b];
          need(std::fabs(s - (a == b)) <= 1e-13, "eigenvectors");
        }
      }
      // the only line block with a null space (constants) is the one between two Neumann ends
      need(code == 8 ? std::fabs(lmin) <= 1e-13 * lmax : lmin > 1e-3, "eigenvalues");
    }
  }
}

int main() {
  try {
    check_tables();
    check_dense();
    check_sell();
    check_patterns();
    check_hierarchy(7, 1., 1e-12);  // solved directly
    check_hierarchy(40, 1., 0.5);
    check_hierarchy(60, 1., 0.5);
    check_hierarchy(50, 25., 0.7);
    std::printf("OK\n");
    return 0;
  } catch (const std::exception& e) {
    std::printf("ERROR %s\n", e.what());
    return 1;
  }
}
