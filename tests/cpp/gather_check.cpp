// gather_check.cpp - CPU check of gather_pack (hoc_host.cpp): every vertex finds its corners and otherwise
// padding, and the table stays in proportion to the corners when one vertex has many.  Prints "OK", exits 0.
#include <cstdio>
#include <vector>

#include "hoc_host.hpp"

using namespace hoc;

// valence(v) corners at vertex v; returns entries per corner, or -1 on a wrong table
template <class Fn>
static double check(int nv, bool want_off, Fn valence) {
  std::vector<int32_t> ptr(1, 0), vinc, off, inc;
  for (int v = 0; v < nv; ++v) {
    for (int c = 0; c < valence(v); ++c) vinc.push_back(7 * v + c);
    ptr.push_back((int)vinc.size());
  }
  const int pad = -5;
  int w = -1;
  gather_pack(ptr, vinc, pad, w, off, inc);
  if (off.empty() == want_off) return -1.;
  for (int v = 0; v < nv; ++v) {
    const size_t q = off.empty() ? (size_t)(v / 64) * 64 * w : (size_t)off[v / 64];
    const int n = off.empty() ? w : (off[v / 64 + 1] - off[v / 64]) / 64;
    if (n < valence(v)) return -1.;
    for (int c = 0; c < n; ++c) {
      const size_t i = q + (size_t)64 * c + v % 64;
      if (i >= inc.size() || inc[i] != (c < valence(v) ? 7 * v + c : pad)) return -1.;
    }
  }
  return vinc.empty() ? 0. : (double)inc.size() / (double)vinc.size();
}

int main() {
  const double r[] = {
      check(1, false, [](int) { return 1; }),
      check(64, false, [](int) { return 4; }),
      check(65, false, [](int v) { return 1 + v % 4; }),
      check(100000, false, [](int v) { return v % 300 == 0 ? 2 : 4; }),
      check(129, true, [](int v) { return v == 128 ? 128 : 2; }),
      check(100000, true, [](int v) { return v == 4711 ? 2000 : 4; }),
  };
  int bad = 0;
  for (double x : r) bad += x < 0.;
  std::printf("entries per corner: uniform %.2f, one vertex of 2000 %.2f\n", r[3], r[5]);
  bad += !(r[3] <= 1.1) || !(r[5] <= 1.5);  // 2000 entries for the 63 other vertices of one slice: 0.32 on top
  std::printf(bad ? "%d failures\n" : "OK\n", bad);
  return bad != 0;
}
