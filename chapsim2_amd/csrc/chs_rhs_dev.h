// Device-side pieces of the fused line operators (chs_rhs.h).
#pragma once

#include "chs_rhs.h"

namespace chs {

// Explicit rows of a chunk from its window g[t] = element (row s0 - 2 + sh + t):
// y[i] = c1 (g[i+2] + s g[i+1]) + c2 (g[i+3] + s g[i]), the one form of all
// four staggered operators.  Chunks at a wall take rows 0, 1 and n-2, n-1
// from dense window weights (`first` / `last`; len rows in the chunk).
template <typename T, int CH>
__device__ __forceinline__ void fuse_rows(const FusePlan<T>& p, bool first, bool last, int len,
                                          const T (&g)[CH + 3], const T (&fb4)[4], T (&y)[CH]) {
  constexpr int W = CH + 3;
  auto edge = [&](int r) -> T {
    const T* w = p.edge + r * (W + 4);
    T v = T(0);
#pragma unroll
    for (int t = 0; t < W; ++t) v = v + w[t] * g[t];
#pragma unroll
    for (int m = 0; m < 4; ++m) v = v + w[W + m] * fb4[m];
    return v;
  };
  T v0 = T(0), v1 = T(0), v2 = T(0), v3 = T(0);
  if (first) {
    v0 = edge(0);
    v1 = edge(1);
  }
  if (last) {
    v2 = edge(2);
    v3 = edge(3);
  }
#pragma unroll
  for (int i = 0; i < CH; ++i)
    y[i] = p.c1 * (g[i + 2] + p.sgn * g[i + 1]) + p.c2 * (g[i + 3] + p.sgn * g[i]);
  if (first) {
    y[0] = v0;
    y[1] = v1;
  }
  if (last) {
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      y[i] = i == len - 2 ? v2 : y[i];
      y[i] = i == len - 1 ? v3 : y[i];
    }
  }
}

// Chunk-local Thomas sweeps.  Rows past the chunk's length copy the row before
// them, so the chunk's last value always ends in y[CH - 1].
template <typename T, int CH>
__device__ __forceinline__ void fuse_solve(const T* c, T (&y)[CH]) {
  y[0] = y[0] * c[FC_LD];
#pragma unroll
  for (int i = 1; i < CH; ++i) y[i] = y[i] * c[i * kFuseCo + FC_LD] - c[i * kFuseCo + FC_AL] * y[i - 1];
#pragma unroll
  for (int i = CH - 2; i >= 0; --i) y[i] = y[i] - c[i * kFuseCo + FC_LC] * y[i + 1];
}

// Spike correction from the published chunk ends ex(k) (k: 2 * chunk + 0 first,
// 1 last): the previous chunk's last and the next chunk's first value, each a
// sum over the fuse_band ends around chunk q with the plan's weights cp.
template <typename T, int CH, class EX>
__device__ __forceinline__ void fuse_couple(const FusePlan<T>& p, int q, const T* cp, const T* c, EX&& ex,
                                            T (&y)[CH]) {
  constexpr int NB = fuse_band<T>(CH);
  const int M = 2 * p.P;
  int k = 2 * q - (NB / 2 - 1);
  T uL = T(0), uF = T(0);
  if (p.wrap) {
    // (the weights of ends met twice on short lines are zero)
    while (k < 0) k += M;
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const T v = ex(k);
      uL = uL + cp[j] * v;
      uF = uF + cp[NB + j] * v;
      ++k;
      if (k >= M) k -= M;
    }
  } else {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int kk = k + j;
      const T v = ex(kk < 0 ? 0 : (kk > M - 1 ? M - 1 : kk));
      uL = uL + cp[j] * v;
      uF = uF + cp[NB + j] * v;
    }
  }
#pragma unroll
  for (int i = 0; i < CH; ++i) y[i] = y[i] - c[i * kFuseCo + FC_SV] * uL - c[i * kFuseCo + FC_SW] * uF;
}

// Offsets of a plan's tables after `tab`: coupling weights, metric.
__host__ __device__ __forceinline__ int fuse_cp_at(int rows) { return 3 * rows * kFuseCo; }
template <typename T>
__host__ __device__ __forceinline__ int fuse_met_at(int rows, int P) {
  return 3 * rows * kFuseCo + P * 2 * fuse_band<T>(rows);
}

// A plan's table on its way to LDS in 16-byte pieces: the loads are issued
// first thing (NS pieces per thread; more only for lines of few chunks), the
// stores once the window's loads are in flight behind them.  dst is 16-byte
// aligned and ntab a multiple of 4.
template <typename T, int NS>
struct TableLoad {
  uint4 v[NS];
  __device__ __forceinline__ void issue(const FusePlan<T>& p, int tid, int nthr) {
    const uint4* src = reinterpret_cast<const uint4*>(p.tab);
    const int n = p.ntab * (int)sizeof(T) / 16;
#pragma unroll
    for (int u = 0; u < NS; ++u) v[u] = src[tid + u * nthr < n ? tid + u * nthr : 0];
  }
  __device__ __forceinline__ void store(T* dst, const FusePlan<T>& p, int tid, int nthr) const {
    const uint4* src = reinterpret_cast<const uint4*>(p.tab);
    uint4* d = reinterpret_cast<uint4*>(dst);
    const int n = p.ntab * (int)sizeof(T) / 16;
#pragma unroll
    for (int u = 0; u < NS; ++u)
      if (tid + u * nthr < n) d[tid + u * nthr] = v[u];
    for (int e = tid + NS * nthr; e < n; e += nthr) d[e] = src[e];
  }
};

}  // namespace chs
