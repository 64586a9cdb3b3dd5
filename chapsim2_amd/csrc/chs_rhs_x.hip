// Fused x line operators (chs_rhs.h): periodic lines, contiguous in memory.
//
// A wave owns 64 / P whole lines and one lane one chunk of CH rows (the last
// one of a line may be shorter).  The lines (one contiguous piece of memory of
// at most 64 x CH values) pass through the wave's own part of the LDS:
// coalesced 16-byte loads in, each lane's window out, the chunk ends
// exchanged, the results back and out with coalesced stores.  No step needs
// another wave, so there is no workgroup barrier after the coefficient tables
// are in place, and the waves of a CU load, solve and store independently (the
// workgroup-wide tiles of k_line_xu do each of these as a phase of the whole
// workgroup).  Chunks lie CH + 1 values apart, so the lanes' window reads
// spread over the banks.
#include "chs_rhs_dev.h"

namespace chs {

constexpr int kXWaves = 4;  // most waves per workgroup (they share the coefficient tables)

// LDS operations of one wave complete in order; this only keeps the compiler
// from moving them across the point where other lanes' values are read.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

typedef unsigned xu32x4 __attribute__((ext_vector_type(4)));
typedef unsigned xu32x2 __attribute__((ext_vector_type(2)));
template <typename T, int G>
struct alignas(sizeof(T) * G) XGrp {
  T v[G];
};
template <typename T, int G>
__device__ __forceinline__ XGrp<T, G> ld_grp_x(const T* p) {
  return *reinterpret_cast<const XGrp<T, G>*>(p);
}
template <typename T, int G>
__device__ __forceinline__ void st_grp_x(T* p, const XGrp<T, G>& g) {
  if constexpr (sizeof(T) * G == 16) {
    xu32x4 v;
    __builtin_memcpy(&v, &g, 16);
    __builtin_nontemporal_store(v, reinterpret_cast<xu32x4*>(p));
  } else if constexpr (sizeof(T) * G == 8) {
    xu32x2 v;
    __builtin_memcpy(&v, &g, 8);
    __builtin_nontemporal_store(v, reinterpret_cast<xu32x2*>(p));
  } else {
    static_assert(sizeof(T) * G == 32, "groups of 8, 16 or 32 bytes");
    XGrp<T, G / 2> a, b;
#pragma unroll
    for (int c = 0; c < G / 2; ++c) {
      a.v[c] = g.v[c];
      b.v[c] = g.v[G / 2 + c];
    }
    st_grp_x<T, G / 2>(p, a);
    st_grp_x<T, G / 2>(p + G / 2, b);
  }
}

// Tile values a wave needs: its lines, or two sets of chunk ends.
__host__ __device__ __forceinline__ int x_piece(int P, int ch) {
  const int lines = (64 / P) * P * (ch + 1);
  return lines > 256 ? lines : 256;
}

// G values (a divisor of the line length, at most 16 bytes) per access.
template <typename T, int KIND, int CH, int G>
__global__ void __launch_bounds__(64 * kXWaves) __attribute__((amdgpu_waves_per_eu(4))) k_rhs_x(RhsGroup<T> Gr) {
  constexpr bool kTwo = KIND == RK_PAIR || KIND == RK_FINAL;
  constexpr bool kWin2 = KIND == RK_FINAL;
  constexpr int UB = CH / G;   // groups per lane
  constexpr int CS = CH + 1;   // chunk stride in the tile
  static_assert(CH % G == 0, "a group lies in one chunk");
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int jb = 0;
#pragma unroll
  for (int t = 1; t < kGroupJobs; ++t)
    if (t < Gr.n && (int)blockIdx.x >= Gr.first[t]) jb = t;
  const RhsJob<T>& J = Gr.job[jb];
  const FusePlan<T>& p1 = J.p1;
  const FusePlan<T>& p2 = J.p2;
  const int tid = threadIdx.x, lane = tid & 63, nthr = blockDim.x;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int P = p1.P, n = p1.n_in, lpw = 64 / P, LS = P * CS;
  // (a wave without lines, nl = 0, runs along and stores nothing)
  const long Lw = ((long)((int)blockIdx.x - Gr.first[jb]) * (nthr >> 6) + wv) * lpw;
  const long left = J.nlines - Lw;
  const int nl = left < 0 ? 0 : (left < lpw ? (int)left : lpw);
  const int tot = nl * n;
  const long base = (nl > 0 ? Lw : 0) * n;
  T* const s1 = reinterpret_cast<T*>(smem_raw);
  T* const s2 = s1 + p1.ntab;
  T* const tile = s1 + p1.ntab + (kTwo ? p2.ntab : 0) + wv * x_piece(P, CH);
  // the tables' loads, the first field's behind them
  TableLoad<T, 3> t1, t2;
  t1.issue(p1, tid, nthr);
  if constexpr (kTwo) t2.issue(p2, tid, nthr);
  XGrp<T, G> v[UB];
  auto fetch = [&](const T* src) {
#pragma unroll
    for (int u = 0; u < UB; ++u) {
      const int e = (lane + 64 * u) * G;
      v[u] = ld_grp_x<T, G>(src + base + (e < tot ? e : 0));
    }
  };
  fetch(J.A);
  // tile position of each group: line e / n (2^20 / n rounded up: exact for e < 64 CH)
  const unsigned mn = ((1u << 20) + n - 1) / n;
  int at[UB];
#pragma unroll
  for (int u = 0; u < UB; ++u) {
    const int e = (lane + 64 * u) * G;
    const int line = (int)(((unsigned)e * mn) >> 20), k = e - line * n;
    at[u] = e < tot ? line * LS + k + k / CH : -1;
  }
  auto each = [&](auto&& f) {
#pragma unroll
    for (int u = 0; u < UB; ++u)
      if (at[u] >= 0) f(u, base + (lane + 64 * u) * G);
  };
  auto to_lines = [&]() {
    if constexpr (KIND == RK_CORRECT) {
      if (J.add) {  // the pressure takes its increment on the way
        each([&](int u, long o) {
          XGrp<double, G> p = ld_grp_x<double, G>(J.add + o);
          XGrp<float, G> w;
#pragma unroll
          for (int c = 0; c < G; ++c) {
            p.v[c] = p.v[c] + v[u].v[c];
            w.v[c] = (float)p.v[c];
          }
          st_grp_x<double, G>(J.add + o, p);
          if (J.add32) *reinterpret_cast<XGrp<float, G>*>(J.add32 + o) = w;
        });
      }
    }
    each([&](int u, long) {
#pragma unroll
      for (int c = 0; c < G; ++c) tile[at[u] + c] = v[u].v[c];
    });
    wave_sync();
  };
  t1.store(s1, p1, tid, nthr);
  if constexpr (kTwo) t2.store(s2, p2, tid, nthr);
  __syncthreads();
  // this lane's chunk
  const int line = lane / P, q = lane - line * P;
  const bool live = line < nl;
  const int lb = (live ? line : 0) * LS, s0 = q * CH, own = lb + q * CS;
  const int len = n - s0 < CH ? n - s0 : CH;
  auto window = [&](T(&g)[CH + 3]) {
    const int sh = p1.sh;
#pragma unroll
    for (int t = 0; t < CH + 3; ++t) {
      const int i = t - 2 + sh;  // row of the chunk
      int a = own + i + (i >= CH ? 1 : 0);
      if (t < 2 && i < 0) {  // the previous chunk's end, or the line's
        const int k = q == 0 ? n + i : s0 + i;
        a = lb + k + k / CH;
      }
      // past the line's end: its first two rows (what lies beyond is not used)
      if (t > 2 && i >= len && q == P - 1) a = lb + (i - len > 1 ? 1 : i - len);
      g[t] = tile[a];
    }
  };
  const T zero4[4] = {T(0), T(0), T(0), T(0)};
  const int cls = (q == 0 ? 0 : (q == P - 1 ? 2 : 1)) * CH * kFuseCo;
  T y1[CH];
  T y2[kTwo ? CH : 1];
  {
    T g[CH + 3];
    to_lines();
    if constexpr (kWin2) fetch(J.A2);
    window(g);
    fuse_rows<T, CH>(p1, false, false, len, g, zero4, y1);
    if constexpr (kTwo && !kWin2) fuse_rows<T, CH>(p2, false, false, len, g, zero4, y2);
    wave_sync();
  }
  if constexpr (kWin2) {
    T g[CH + 3];
    to_lines();
    window(g);
    fuse_rows<T, CH>(p2, false, false, len, g, zero4, y2);
    wave_sync();
  }
  // chunk ends through the tile's start (every window has been read)
  if (p1.solve) {
    fuse_solve<T, CH>(s1 + cls, y1);
    tile[2 * lane] = y1[0];
    tile[2 * lane + 1] = y1[CH - 1];
  }
  if constexpr (kTwo) {
    if (p2.solve) {
      fuse_solve<T, CH>(s2 + cls, y2);
      tile[128 + 2 * lane] = y2[0];
      tile[128 + 2 * lane + 1] = y2[CH - 1];
    }
  }
  wave_sync();
  const T* const ends = tile + 2 * (lane - q);  // this line's chunk ends
  if (p1.solve) fuse_couple<T, CH>(p1, q, s1 + fuse_cp_at(CH) + q * 2 * fuse_band<T>(CH), s1 + cls, [&](int e) { return ends[e]; }, y1);
  if constexpr (kTwo) {
    if (p2.solve)
      fuse_couple<T, CH>(p2, q, s2 + fuse_cp_at(CH) + q * 2 * fuse_band<T>(CH), s2 + cls, [&](int e) { return ends[128 + e]; }, y2);
  }
  wave_sync();
  auto rows_out = [&](const T(&y)[CH]) {
    if (live)
#pragma unroll
      for (int i = 0; i < CH; ++i)
        if (i < len) tile[own + i] = y[i];
    wave_sync();
  };
  auto from_tile = [&](int u) {
    XGrp<T, G> r;
#pragma unroll
    for (int c = 0; c < G; ++c) r.v[c] = tile[at[u] + c];
    return r;
  };
  rows_out(y1);
  if constexpr (KIND == RK_SINGLE) {
    each([&](int u, long o) { st_grp_x<T, G>(J.out + o, from_tile(u)); });
  } else if constexpr (KIND == RK_PAIR) {
    each([&](int u, long o) { st_grp_x<T, G>(J.out + o, from_tile(u)); });
    wave_sync();
    rows_out(y2);
    each([&](int u, long o) { st_grp_x<T, G>(J.out2 + o, from_tile(u)); });
  } else if constexpr (KIND == RK_CORRECT) {
    const T bulk = J.bulk ? T(J.bulk[0]) : T(0);
    each([&](int u, long o) {
      XGrp<T, G> r = from_tile(u);
      const XGrp<T, G> prev = ld_grp_x<T, G>(J.out + o);
      XGrp<float, G> w;
#pragma unroll
      for (int c = 0; c < G; ++c) {
        r.v[c] = (prev.v[c] - bulk) + r.v[c] * J.sOut;
        w.v[c] = (float)r.v[c];
      }
      st_grp_x<T, G>(J.out + o, r);
      if (J.out32) *reinterpret_cast<XGrp<float, G>*>(J.out32 + o) = w;
    });
  } else {
    // RK_FINAL: own operator and pressure gradient back in memory order, then
    // the fractional step
    each([&](int u, long) { v[u] = from_tile(u); });
    wave_sync();
    rows_out(y2);
    double sum = 0.0;
    each([&](int u, long o) {
      const XGrp<T, G> f2 = from_tile(u);
      const XGrp<T, G> a = ld_grp_x<T, G>(J.o1 + o), b = ld_grp_x<T, G>(J.o2 + o);
      XGrp<T, G> c;
#pragma unroll
      for (int x = 0; x < G; ++x) c.v[x] = T(0);
      if (J.tz != T(0)) c = ld_grp_x<T, G>(J.r0 + o);
      XGrp<double, G> qv;
      if (J.q) qv = ld_grp_x<double, G>(J.q + o);
      XGrp<T, G> rv;
#pragma unroll
      for (int x = 0; x < G; ++x) {
        const T cur = (a.v[x] + b.v[x]) + v[u].v[x];
        T tt = J.tg * cur + J.tz * c.v[x];
        tt = tt - J.ta * f2.v[x];
        c.v[x] = cur;
        rv.v[x] = J.dt * tt;
      }
      st_grp_x<T, G>(J.r0 + o, c);
      if (J.q) {
#pragma unroll
        for (int x = 0; x < G; ++x) qv.v[x] = qv.v[x] + (double)rv.v[x];
        st_grp_x<double, G>(J.q + o, qv);
      } else {
        st_grp_x<T, G>(J.out + o, rv);
      }
      if (J.partial) {
        // (a group lies in one line: G divides n)
        const double w = J.dyw[(int)((Lw + (((unsigned)((lane + 64 * u) * G) * mn) >> 20)) % J.n2)] * J.dxdz;
#pragma unroll
        for (int x = 0; x < G; ++x) sum += (double)rv.v[x] * w;
      }
    });
    if (J.partial) {
      __shared__ double red[kXWaves];
#pragma unroll
      for (int k = 32; k > 0; k >>= 1) sum = sum + __shfl_xor(sum, k);
      if (lane == 0) red[wv] = sum;
      __syncthreads();
      if (tid == 0) {
        double t = red[0];
        for (int k = 1; k < (nthr >> 6); ++k) t = t + red[k];
        J.partial[blockIdx.x - Gr.first[jb]] = t;
      }
    }
  }
}

// Waves per workgroup: as many as share the tables, but no fewer workgroups
// than the CUs have room for.  FP64 sub-steps with 1, 2 and 4 waves: 64^3 (512
// waves of x lines) 177, 175, 174 us, 128x96x96 (1152) 344, 335, 341, 192x96x160
// (3072) 705, 676, 675, 256x128x256 (8192) 1685, 1642, 1589; below 1024 waves
// the choice is worth 2 % at most.
static int x_waves(long waves) { return waves >= 2048 ? kXWaves : waves >= 1024 ? 2 : 1; }

template <typename T>
static long job_waves(const RhsJob<T>& J) {
  const int lpw = 64 / J.p1.P;
  return (J.nlines + lpw - 1) / lpw;
}

template <typename T>
int rhs_x_blocks(const RhsJob<T>& J) {
  const int nw = x_waves(job_waves(J));
  return (int)((job_waves(J) + nw - 1) / nw);
}

template <typename T, int CH, int G>
static void x_kind(int kind, dim3 g, dim3 b, size_t shm, hipStream_t s, const RhsGroup<T>& Gr) {
  switch (kind) {
    case RK_SINGLE: hipLaunchKernelGGL((k_rhs_x<T, RK_SINGLE, CH, G>), g, b, shm, s, Gr); break;
    case RK_PAIR: hipLaunchKernelGGL((k_rhs_x<T, RK_PAIR, CH, G>), g, b, shm, s, Gr); break;
    case RK_CORRECT:
      if constexpr (sizeof(T) == 8) hipLaunchKernelGGL((k_rhs_x<T, RK_CORRECT, CH, G>), g, b, shm, s, Gr);
      break;
    default: hipLaunchKernelGGL((k_rhs_x<T, RK_FINAL, CH, G>), g, b, shm, s, Gr); break;
  }
}

template <typename T>
std::string launch_rhs_x(int kind, int rows, RhsGroup<T>& G, hipStream_t s) {
  if (G.n < 1 || G.n > kGroupJobs || (rows != 16 && rows != 8) ||
      (kind != RK_SINGLE && kind != RK_PAIR && kind != RK_FINAL && !(kind == RK_CORRECT && sizeof(T) == 8)))
    return "fused x: bad group";
  const bool two = kind == RK_PAIR || kind == RK_FINAL;
  long waves = 0;
  for (int j = 0; j < G.n; ++j) {
    if (G.job[j].p1.P < 1 || G.job[j].p1.P > kFuseChunks || G.job[j].nlines < 1) return "fused x: bad job";
    waves += job_waves(G.job[j]);
  }
  const int nw = x_waves(waves);
  size_t shm = 0;
  bool quad = sizeof(T) == 4;  // FP32 lines of a multiple of four: 16-byte groups
  G.first[0] = 0;
  for (int j = 0; j < G.n; ++j) {
    const RhsJob<T>& J = G.job[j];
    const FusePlan<T>& p = J.p1;
    if (p.ell != rows || !p.wrap || p.n_in != p.n_out || p.n_in % 2 || p.n_in > 64 * rows) return "fused x: not such a line";
    if (two && (J.p2.P != p.P || J.p2.ell != p.ell || J.p2.n_in != p.n_in || J.p2.sh != p.sh || !J.p2.wrap))
      return "fused x: a job's two plans differ in geometry";
    auto al = [](const void* q) { return ((size_t)q % 16) == 0; };
    if (!al(J.A) || !al(J.A2) || !al(J.out) || !al(J.out2) || !al(J.o1) || !al(J.o2) || !al(J.r0) || !al(J.q) ||
        !al(J.add) || !al(J.add32) || !al(J.out32))
      return "fused x: unaligned array";
    if (p.n_in % 4) quad = false;
    G.first[j + 1] = G.first[j] + (int)((job_waves(J) + nw - 1) / nw);
    shm = std::max(shm, sizeof(T) * ((size_t)p.ntab + (two ? J.p2.ntab : 0) + (size_t)nw * x_piece(p.P, rows)));
  }
  const dim3 g((unsigned)G.first[G.n]), b((unsigned)(64 * nw));
  if constexpr (sizeof(T) == 4) {
    if (rows == 16) quad ? x_kind<T, 16, 4>(kind, g, b, shm, s, G) : x_kind<T, 16, 2>(kind, g, b, shm, s, G);
    else quad ? x_kind<T, 8, 4>(kind, g, b, shm, s, G) : x_kind<T, 8, 2>(kind, g, b, shm, s, G);
  } else {
    if (rows == 16) x_kind<T, 16, 2>(kind, g, b, shm, s, G);
    else x_kind<T, 8, 2>(kind, g, b, shm, s, G);
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? "" : std::string("fused x launch: ") + hipGetErrorString(e);
}

template int rhs_x_blocks<double>(const RhsJob<double>&);
template int rhs_x_blocks<float>(const RhsJob<float>&);
template std::string launch_rhs_x<double>(int, int, RhsGroup<double>&, hipStream_t);
template std::string launch_rhs_x<float>(int, int, RhsGroup<float>&, hipStream_t);

}  // namespace chs
