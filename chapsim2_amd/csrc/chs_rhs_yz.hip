// Fused y and z line operators (chs_rhs.h).
//
// A workgroup is NLW neighbouring lines x P chunks as in k_line_yz: with 64
// lines wave q holds chunk q, with 32 a wave holds two consecutive chunks (so
// that smaller workgroups share a CU, and lines of up to 32 chunks fit 1024
// threads).  The window of a chunk is loaded once into registers; both
// operators of a pair run from it, publish their chunk ends together (one
// barrier for two solves) and finish in the epilogue of the job's kind.  The
// coefficient tables take 3 to 7 KB of LDS per plan (one set for all inner
// chunks, twelve coupling weights per chunk) where the single operators'
// rows and full inverse take up to 40 KB.
#include "chs_lineop_dev.h"
#include "chs_rhs_dev.h"

namespace chs {

// Rows per epilogue batch: a batch's loads are issued together (in FP32 the
// first ones before the solves; in FP64 that spills), and the next batch's
// before this one's stores, so that a small grid, whose few waves cannot hide
// a memory round trip, waits for as few of them as the registers allow.
template <typename T, int KIND>
constexpr int kEpi = KIND == RK_SHEAR || KIND == RK_CORRECT ? (sizeof(T) == 8 ? 6 : 9) : KIND == RK_DIV ? (sizeof(T) == 8 ? 3 : 6) : (sizeof(T) == 8 ? 4 : 6);

template <typename T, int KIND, int CH, int NLW>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) k_rhs_yz(RhsGroup<T> G) {
  constexpr bool kTwo = KIND != RK_SINGLE && KIND != RK_CORRECT;  // two operators
  constexpr bool kWin2 = KIND == RK_FINAL;   // the second on a field of its own
  extern __shared__ __align__(16) unsigned char smem_raw[];
  int jb = 0;
#pragma unroll
  for (int t = 1; t < kGroupJobs; ++t)
    if (t < G.n && (int)blockIdx.x >= G.first[t]) jb = t;
  const RhsJob<T>& J = G.job[jb];
  const FusePlan<T>& p1 = J.p1;
  const FusePlan<T>& p2 = J.p2;
  // (the workgroup has lanes for G.P chunks; those past this job's repeat its last one and store nothing)
  const int Pn = p1.P, nthr = NLW * G.P, tid = threadIdx.x;
  T* ex1 = reinterpret_cast<T*>(smem_raw);
  T* ex2 = ex1 + (kTwo ? 2 * NLW * G.P : 0);
  T* s1 = ex2 + 2 * NLW * G.P;
  T* s2 = s1 + p1.ntab;
  TableLoad<T, 2> t1, t2;
  t1.issue(p1, tid, nthr);
  if constexpr (kTwo) t2.issue(p2, tid, nthr);
  const int lane = tid & (NLW - 1);
  const int qw = NLW == 64 ? __builtin_amdgcn_readfirstlane(tid >> 6) : tid / NLW;
  const int q = qw < Pn ? qw : Pn - 1;
  const int L0 = ((int)blockIdx.x - G.first[jb]) * NLW;
  const int Lr = L0 + lane;
  const bool live = Lr < J.nlines;
  const int L = live ? Lr : J.nlines - 1;
  const int e1 = J.e1;
  const int i0 = L0 % e1, k0 = L0 / e1, i = L % e1, k = L / e1;
  // wave-uniform base + per-lane 32-bit byte offsets (checked at launch)
  const long ib0 = i0 + J.ips * k0, ob0 = i0 + J.ops * k0;
  const unsigned ri = (unsigned)((i - i0 + J.ips * (k - k0)) * (long)sizeof(T));
  const unsigned ro = (unsigned)((i - i0 + J.ops * (k - k0)) * (long)sizeof(T));
  const int n_in = p1.n_in, n_out = p1.n_out;
  const int s0 = q * p1.ell, len = (q == Pn - 1) ? n_out - s0 : p1.ell;
  const bool first = q == 0 && p1.ends, last = q == Pn - 1 && p1.ends;
  T g[CH + 3];
  T h[kWin2 ? CH + 3 : 1];
  {
    long off[CH + 3];
#pragma unroll
    for (int t = 0; t < CH + 3; ++t) {
      int e = s0 - 2 + p1.sh + t;
      if (p1.wrap) e = e < 0 ? e + n_in : (e >= n_in ? e - n_in : e);
      // (rows past a shorter last chunk: any valid element)
      e = e < 0 ? 0 : (e > n_in - 1 ? n_in - 1 : e);
      off[t] = ib0 + J.is * e;
    }
#pragma unroll
    for (int t = 0; t < CH + 3; ++t) g[t] = ld_at(J.A + off[t], ri);
    if constexpr (kWin2) {
#pragma unroll
      for (int t = 0; t < CH + 3; ++t) h[t] = ld_at(J.A2 + off[t], ri);
    }
  }
  T fb1[4] = {T(0), T(0), T(0), T(0)}, fb2[4] = {T(0), T(0), T(0), T(0)};
  if ((q == 0 || q == Pn - 1) && p1.ends) {
    const long fb = i + (long)e1 * 4 * k;
    if (J.fbc)
#pragma unroll
      for (int m = 0; m < 4; ++m) fb1[m] = J.fbc[fb + (long)e1 * m];
    if (kTwo && J.fbc2)
#pragma unroll
      for (int m = 0; m < 4; ++m) fb2[m] = J.fbc2[fb + (long)e1 * m];
  }
  t1.store(s1, p1, tid, nthr);
  if constexpr (kTwo) t2.store(s2, p2, tid, nthr);
  __syncthreads();  // tables
  const int cls = (q == 0 ? 0 : (q == Pn - 1 ? 2 : 1)) * CH * kFuseCo;
  T y1[CH];
  T y2[kTwo ? CH : 1];
  fuse_rows<T, CH>(p1, first, last, len, g, fb1, y1);
  if constexpr (kTwo) {
    if constexpr (kWin2) fuse_rows<T, CH>(p2, first, last, len, h, fb2, y2);
    else fuse_rows<T, CH>(p2, first, last, len, g, fb2, y2);
  }
  // the epilogue's operands, a batch of rows at a time
  constexpr bool kEpil = KIND != RK_SINGLE && KIND != RK_PAIR;
  constexpr int H = kEpi<T, KIND>;
  const long os = J.os;
  const long rb = ob0 + os * s0;
  const unsigned ro8 = ro * (unsigned)(sizeof(double) / sizeof(T));
  T ea[kEpil ? H : 1], eb[kEpil ? H : 1], ec[KIND == RK_DIV || KIND == RK_FINAL ? H : 1], ed[KIND == RK_DIV ? H : 1];
  double eq[KIND == RK_FINAL ? H : 1];
  auto fetch = [&](int r0) {
    if constexpr (kEpil) {
#pragma unroll
      for (int u = 0; u < H; ++u) {
        if (r0 + u >= CH) break;
        const int r = r0 + u < len ? r0 + u : len - 1;
        const long o = rb + os * r;
        if constexpr (KIND == RK_CORRECT) {
          ea[u] = ld_at((const T*)J.out + o, ro);
          continue;
        }
        ea[u] = ld_at(J.o1 + o, ro);
        eb[u] = ld_at(J.o2 + o, ro);
        if constexpr (KIND == RK_DIV) {
          ec[u] = ld_at((const T*)J.o3 + o, ro);
          ed[u] = ld_at((const T*)J.o4 + o, ro);
        }
        if constexpr (KIND == RK_FINAL) {
          ec[u] = J.tz != T(0) ? ld_at((const T*)J.r0 + o, ro) : T(0);
          eq[u] = J.q ? ld_at((const double*)J.q + o, ro8) : 0.0;
        }
      }
    }
  };
  if constexpr (sizeof(T) == 4) fetch(0);
  if (p1.solve) {
    fuse_solve<T, CH>(s1 + cls, y1);
    ex1[lane + NLW * (2 * q)] = y1[0];
    ex1[lane + NLW * (2 * q + 1)] = y1[CH - 1];
  }
  if constexpr (kTwo) {
    if (p2.solve) {
      fuse_solve<T, CH>(s2 + cls, y2);
      ex2[lane + NLW * (2 * q)] = y2[0];
      ex2[lane + NLW * (2 * q + 1)] = y2[CH - 1];
    }
  }
  if (p1.solve || (kTwo && p2.solve)) __syncthreads();
  if (!live || qw >= Pn) return;
  if (p1.solve)
    fuse_couple<T, CH>(p1, q, s1 + fuse_cp_at(CH) + q * 2 * fuse_band<T>(CH), s1 + cls,
                       [&](int e) { return ex1[lane + NLW * e]; }, y1);
  if constexpr (kTwo) {
    if (p2.solve)
      fuse_couple<T, CH>(p2, q, s2 + fuse_cp_at(CH) + q * 2 * fuse_band<T>(CH), s2 + cls,
                         [&](int e) { return ex2[lane + NLW * e]; }, y2);
  }
  // metric and Neumann rows
  auto post = [&](const FusePlan<T>& p, const T* sm, const T(&fb)[4], T(&y)[CH]) {
    if (p.met) {
      const T* m = sm + fuse_met_at<T>(CH, Pn) + s0;
#pragma unroll
      for (int r = 0; r < CH; ++r)
        y[r] = r < len ? y[r] * m[r] : y[r];
    }
    if (p.neu_lo && q == 0) y[0] = fb[0];
    if (p.neu_hi && q == Pn - 1) {
#pragma unroll
      for (int r = 0; r < CH; ++r)
        y[r] = r == len - 1 ? fb[1] : y[r];
    }
  };
  post(p1, s1, fb1, y1);
  if constexpr (kTwo) post(p2, s2, fb2, y2);
  if constexpr (sizeof(T) == 8) fetch(0);
  if constexpr (!kEpil) {
#pragma unroll
    for (int r = 0; r < CH; ++r)
      if (r < len) {
        st_at<T>(J.out + rb + os * r, ro, y1[r]);
        if constexpr (kTwo) st_at<T>(J.out2 + rb + os * r, ro, y2[r]);
      }
  } else {
#pragma unroll
    for (int r0 = 0; r0 < CH; r0 += H) {
      // results of the batch over y1, y2 (and ec, eq), which frees the operands
      // for the next batch's loads
#pragma unroll
      for (int u = 0; u < H; ++u) {
        const int r = r0 + u;
        if (r >= CH) break;
        if constexpr (KIND == RK_CORRECT) {
          y1[r] = ea[u] + y1[r] * J.sOut;
          if (J.fbw) {
            const long fb = i + (long)e1 * 4 * k;
            if (s0 + r == 0) y1[r] = J.fbw[fb];
            else if (s0 + r == n_out - 1) y1[r] = J.fbw[fb + e1];
          }
        } else if constexpr (KIND == RK_SHEAR) {
          const T v = (T(-1) * y1[r]) * ea[u];
          y1[r] = v + J.r * y2[r] + J.r * eb[u];
        } else if constexpr (KIND == RK_DIV) {
          const T r2 = J.r * T(2), r3 = r2 * T(-1.0 / 3.0);
          const T dv = (ea[u] + eb[u]) + y2[r];
          y1[r] = (T(-1) * y1[r]) * y1[r] + r2 * y2[r] + r3 * dv;
          ea[u] = (T(-1) * ec[u]) * ec[u] + r2 * ea[u] + r3 * dv;
          eb[u] = (T(-1) * ed[u]) * ed[u] + r2 * eb[u] + r3 * dv;
        } else {
          const T cur = (ea[u] + eb[u]) + y1[r];
          T tot = J.tg * cur + J.tz * ec[u];
          tot = tot - J.ta * y2[r];
          y1[r] = cur;
          y2[r] = J.dt * tot;
          if (J.q) {
            eq[u] = eq[u] + (double)y2[r];
            if (J.fbw) {
              const long fb = i + (long)e1 * 4 * k;
              if (s0 + r == 0) eq[u] = J.fbw[fb];
              else if (s0 + r == n_out - 1) eq[u] = J.fbw[fb + e1];
            }
          }
        }
      }
      T sa[KIND == RK_DIV ? H : 1], sb[KIND == RK_DIV ? H : 1];
      double sq[KIND == RK_FINAL ? H : 1];
      if constexpr (KIND == RK_DIV)
#pragma unroll
        for (int u = 0; u < H; ++u) {
          sa[u] = ea[u];
          sb[u] = eb[u];
        }
      if constexpr (KIND == RK_FINAL)
#pragma unroll
        for (int u = 0; u < H; ++u) sq[u] = eq[u];
      if (r0 + H < CH) fetch(r0 + H);
#pragma unroll
      for (int u = 0; u < H; ++u) {
        const int r = r0 + u;
        if (r >= CH) break;
        if (r < len) {
          const long o = rb + os * r;
          if constexpr (KIND == RK_SHEAR || KIND == RK_CORRECT) st_at<T>(J.out + o, ro, y1[r]);
          if constexpr (KIND == RK_CORRECT)
            if (J.out32) st_at<float>(J.out32 + o, ro / (unsigned)(sizeof(T) / sizeof(float)), (float)y1[r]);
          if constexpr (KIND == RK_DIV) {
            st_at<T>(J.out + o, ro, y1[r]);
            st_at<T>(J.o3 + o, ro, sa[u]);
            st_at<T>(J.o4 + o, ro, sb[u]);
          }
          if constexpr (KIND == RK_FINAL) {
            st_at<T>(J.r0 + o, ro, y1[r]);
            if (J.q) st_at<double>(J.q + o, ro8, sq[u]);
            else st_at<T>(J.out + o, ro, y2[r]);
          }
        }
      }
    }
  }
}

template <typename T, int KIND, int CH>
static void yz_width(int nlw, dim3 g, int P, size_t ex, size_t tab, hipStream_t s, const RhsGroup<T>& G) {
  const size_t shm = sizeof(T) * (ex + tab);
  if (nlw == 64)
    hipLaunchKernelGGL((k_rhs_yz<T, KIND, CH, 64>), g, dim3(64 * P), shm, s, G);
  else
    hipLaunchKernelGGL((k_rhs_yz<T, KIND, CH, 32>), g, dim3(32 * P), shm, s, G);
}

template <typename T, int CH>
static void yz_kind(int kind, int nlw, dim3 g, int P, size_t ex, size_t tab, hipStream_t s, const RhsGroup<T>& G) {
  switch (kind) {
    case RK_SINGLE: yz_width<T, RK_SINGLE, CH>(nlw, g, P, ex, tab, s, G); break;
    case RK_PAIR: yz_width<T, RK_PAIR, CH>(nlw, g, P, ex, tab, s, G); break;
    case RK_SHEAR: yz_width<T, RK_SHEAR, CH>(nlw, g, P, ex, tab, s, G); break;
    case RK_CORRECT:
      if constexpr (sizeof(T) == 8) yz_width<T, RK_CORRECT, CH>(nlw, g, P, ex, tab, s, G);
      break;
    case RK_DIV: yz_width<T, RK_DIV, CH>(nlw, g, P, ex, tab, s, G); break;
    default: yz_width<T, RK_FINAL, CH>(nlw, g, P, ex, tab, s, G); break;
  }
}

template <typename T>
std::string launch_rhs_yz(int kind, int rows, RhsGroup<T>& G, hipStream_t s) {
  if (G.n < 1 || G.n > kGroupJobs || (rows != 16 && rows != 17 && rows != 8 && rows != 9) || kind < RK_SINGLE || kind > RK_CORRECT ||
      (kind == RK_CORRECT && sizeof(T) != 8))
    return "fused yz: bad group";
  const bool two = kind != RK_SINGLE && kind != RK_CORRECT;
  int P = 0;
  for (int j = 0; j < G.n; ++j) P = std::max(P, G.job[j].p1.P);
  if (P < 1 || P > kFuseChunks) return "fused yz: bad chunks";
  G.P = P;
  // 64 lines per workgroup up to 16 chunks of 8 or 9 rows (8 of 16 or 17): at
  // 256x128x256, where only lines of up to 8 chunks take them, a sub-step is as
  // fast with 32 lines throughout (1591 us FP64, 1124 mixed) and slower with 64
  // for 16 chunks too (1609, 1148).  On small grids the two are within 3 %: 129 us
  // against 132 at 32x24x16, 177 against 172 at 64^3, 200 against 195 at 96x64x64.
  const bool wide = rows < 16 ? P <= 16 : P <= 8;
  const int nlw = wide ? 64 : 32;
  size_t tab = 0;
  G.first[0] = 0;
  for (int j = 0; j < G.n; ++j) {
    const RhsJob<T>& J = G.job[j];
    if (J.p1.P < 1 || J.rows != rows || J.p1.ell > rows) return "fused yz: a plan of another chunk length";
    if (two && (J.p2.P != J.p1.P || J.p2.ell != J.p1.ell || J.p2.n_in != J.p1.n_in || J.p2.n_out != J.p1.n_out ||
                              J.p2.sh != J.p1.sh || J.p2.wrap != J.p1.wrap))
      return "fused yz: a job's two plans differ in geometry";
    if (J.nlines < 1 || J.e1 < 1) return "fused yz: no lines";
    // per-lane byte offsets from the workgroup's first line stay below 2^31
    const long span = (long)nlw + (nlw / J.e1 + 2) * std::max(J.ips, J.ops);
    if (span * (long)sizeof(double) >= (1L << 31)) return "fused yz: lines too far apart for 32-bit offsets";
    G.first[j + 1] = G.first[j] + (J.nlines + nlw - 1) / nlw;
    tab = std::max(tab, (size_t)J.p1.ntab + (two ? J.p2.ntab : 0));
  }
  const size_t ex = (size_t)2 * nlw * P * (two ? 2 : 1);
  const dim3 g((unsigned)G.first[G.n]);
  switch (rows) {
    case 8: yz_kind<T, 8>(kind, nlw, g, P, ex, tab, s, G); break;
    case 9: yz_kind<T, 9>(kind, nlw, g, P, ex, tab, s, G); break;
    case 16: yz_kind<T, 16>(kind, nlw, g, P, ex, tab, s, G); break;
    default: yz_kind<T, 17>(kind, nlw, g, P, ex, tab, s, G); break;
  }
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? "" : std::string("fused yz launch: ") + hipGetErrorString(e);
}

template std::string launch_rhs_yz<double>(int, int, RhsGroup<double>&, hipStream_t);
template std::string launch_rhs_yz<float>(int, int, RhsGroup<float>&, hipStream_t);

}  // namespace chs
