// hoc_rowlane.hpp - device helpers of the kernels that give K lanes of a wavefront to an element: lane
// k holds row k (the xi line) and column k (the eta line) of the element and face point k of each of
// its four faces.
#pragma once

#include "hoc_poisson.hpp"

namespace hoc {

namespace {

// Blocks are dealt to the 8 XCDs in turn: block b works on part b % 8 of the elements, so the
// elements an XCD works on at one time are neighbours and share its L2.
__device__ __forceinline__ int xcd_block(int b, int nb) {
  const int q = nb >> 3, r = nb & 7, x = b & 7, i = b >> 3;
  return x * q + min(x, r) + i;
}

// Orders this wavefront's LDS writes before its reads (LDS serves one wavefront in order).
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <int K>
struct Lay {
  static constexpr int EPW = fine_epw(K);
  static constexpr int RS = (K & 1) ? K : K + 1;  // row stride in LDS (odd: rows on distinct banks)
  static constexpr int ES = K * RS;
  static constexpr int TILE = EPW * ES;
};

// Two values at any address aligned to one of them (one 16- or 8-byte load).
template <class R> struct Two;
template <> struct Two<double> { typedef double t __attribute__((ext_vector_type(2), aligned(8))); };
template <> struct Two<float> { typedef float t __attribute__((ext_vector_type(2), aligned(4))); };

template <int K, class V, class R>
__device__ __forceinline__ void load_row(const V* __restrict__ g, R (&v)[K]) {
#pragma unroll
  for (int i = 0; i + 1 < K; i += 2) {
    const typename Two<V>::t t = *reinterpret_cast<const typename Two<V>::t*>(g + i);
    v[i] = (R)t.x;
    v[i + 1] = (R)t.y;
  }
  if (K & 1) v[K - 1] = (R)g[K - 1];
}
template <int K, class V, class R>
__device__ __forceinline__ void store_row(V* __restrict__ g, const R (&v)[K]) {
#pragma unroll
  for (int i = 0; i + 1 < K; i += 2) {
    typename Two<V>::t t;
    t.x = (V)v[i];
    t.y = (V)v[i + 1];
    *reinterpret_cast<typename Two<V>::t*>(g + i) = t;
  }
  if (K & 1) g[K - 1] = (V)v[K - 1];
}

// rows -> columns (and columns -> rows) of the wavefront's elements through its LDS tile
template <int K, class R>
__device__ __forceinline__ void rows_to_cols(R* t, int k, const R (&row)[K], R (&col)[K]) {
  constexpr int RS = Lay<K>::RS;
  wave_fence();
#pragma unroll
  for (int i = 0; i < K; ++i) t[k * RS + i] = row[i];
  wave_fence();
#pragma unroll
  for (int j = 0; j < K; ++j) col[j] = t[j * RS + k];
}
template <int K, class R>
__device__ __forceinline__ void cols_to_rows(R* t, int k, const R (&col)[K], R (&row)[K]) {
  constexpr int RS = Lay<K>::RS;
  wave_fence();
#pragma unroll
  for (int j = 0; j < K; ++j) t[j * RS + k] = col[j];
  wave_fence();
#pragma unroll
  for (int i = 0; i < K; ++i) row[i] = t[k * RS + i];
}

// The neighbour's point on its face fn that meets this element's point k of face f.
template <int K>
__device__ __forceinline__ int face_point(int f, int fn, int k) {
  return ((f + fn - f / 2 - fn / 2 + 1) & 1) ? K - 1 - k : k;
}

// The line of neighbour nb through its point kk of its face fn, from that face inward (f: the face of
// this element, k: the lane).  opp: every lane of the wavefront meets the neighbour with its opposite
// face (meshes numbered and oriented alike); the line's stride is a constant then.
template <int K, class V, class R>
__device__ __forceinline__ void nbr_line(const V* __restrict__ g, int nb, int f, int fn, int kk, int k, bool opp,
                                         R (&v)[K]) {
  const size_t o = (size_t)nb * (K * K);
  if (opp) {
    if (f < 2) {
      R w[K];
      load_row<K>(g + o + k * K, w);
#pragma unroll
      for (int m = 0; m < K; ++m) v[m] = f == 0 ? w[K - 1 - m] : w[m];
    } else {
#pragma unroll
      for (int m = 0; m < K; ++m) v[m] = (R)g[o + k + (f == 2 ? (K - 1 - m) * K : m * K)];
    }
  } else {
    const int up = fn & 1, step = fn < 2 ? (up ? -1 : 1) : (up ? -K : K);
    const V* q = g + o + (fn < 2 ? kk * K + (up ? K - 1 : 0) : (up ? (K - 1) * K : 0) + kk);
#pragma unroll
    for (int m = 0; m < K; ++m) v[m] = (R)q[m * step];
  }
}

}  // namespace

}  // namespace hoc
