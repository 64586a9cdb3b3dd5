// Thermal properties from the tabulated equation of state, per cell.
//
// Host: the table build of buildup_property_relations_from_table
// (src/input_thermo.f90:617-693): selection sort by T (:512-556), reference
// state by bisection in T (:121-154), non-dimensionalisation, rho*h and its
// range.  Device: one thread per cell runs ftp_refresh_thermal_properties_from_DH
// (:393-446) -- clamp, bisection on rho*h, h, properties from h (:345-374),
// h = rho*h / d, properties from h -- with the searched columns (rho*h, h, d,
// m) staged in LDS when they fit, and with searches that start near their
// result and end in the bisection's interval.  Floating-point contraction is off in the
// kernel so every product and sum rounds as in the reference's expressions.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "chs_props.h"

namespace chs {
void set_error(const std::string& msg);
}


namespace {

enum { CT = 0, CD, CM, CK, CB, CCP, CH, CRH };
constexpr double kMinP = 1.0e-20;  // src/modules.f90:141
constexpr double kNodeGap = 1.001e-10;  // sqrt(kMinP), with room for its square's rounding
constexpr int kNoBin = 65535;       // entry of bins that are not used
constexpr int kPropsLds = 2048;    // rows of the one column k_props_from_h stages (x3, 48 KB)
constexpr int kPropsBlock = 1024;  // threads of the persistent from-rho*h kernel

int fail(int code, const std::string& msg) {
  chs::set_error(msg);
  return code;
}

void bisect_host(const std::vector<double>& c, double v, int* i1o, int* i2o) {
  int i1 = 0, i2 = (int)c.size() - 1;
  while (i2 - i1 > 1) {
    const int im = i1 + (i2 - i1) / 2;
    const double d1 = c[i1] - v, dm = c[im] - v;
    if (d1 * dm > kMinP) i1 = im;
    else i2 = im;
  }
  *i1o = i1;
  *i2o = i2;
}

// Bins of the rho*h search (find_rhoh): nbins + 1 edges of equal spacing over
// [dhmin, dhmax].  A value v has its interval k (the bisection's result,
// whatever rows it probes) where every row up to k lies on one side of v and
// every later row on the other; an entry is the k of its edge, so the
// intervals of a bin lie between its two edges' entries.  Columns need not be
// monotone: an interval some other row also falls into (the tail of rho*h of
// a supercritical table) is not searched by bins, and both entries of every
// bin that meets one are kNoBin.  Twice as many bins as rows and at most
// 16384 (32 KB of LDS); none for columns that are not finite or beyond 16-bit
// row numbers.
std::vector<uint16_t> rhoh_bins(chs_props* p) {
  const int n = p->n;
  const double range = p->dhmax - p->dhmin;
  int nb = 16;
  while (nb < 2 * n && nb < 16384) nb *= 2;
  const double scale = nb / range;
  if (n >= kNoBin || !(range > 0.0) || !std::isfinite(range) || !std::isfinite(scale)) return {};
  const int sg = p->col[CRH][n - 1] > p->col[CRH][0] ? 1 : -1;
  std::vector<double> c(p->col[CRH]), before(n), after(n);  // rising from here on
  for (double& x : c) {
    if (!std::isfinite(x)) return {};
    x *= sg;
  }
  for (int i = 0; i < n; ++i) before[i] = i && before[i - 1] > c[i] ? before[i - 1] : c[i];
  for (int i = n - 1; i >= 0; --i) after[i] = i < n - 1 && after[i + 1] < c[i] ? after[i + 1] : c[i];
  auto clean = [&](int k) { return before[k] == c[k] && after[k + 1] == c[k + 1] && c[k] < c[k + 1]; };
  std::vector<uint16_t> e((size_t)nb + 1);
  for (int b = 0; b <= nb; ++b) {
    const double edge = sg * (p->dhmin + range * ((double)b / nb));
    const int k = (int)(std::upper_bound(before.begin(), before.end(), edge) - before.begin()) - 1;
    e[b] = (uint16_t)(k < 0 ? 0 : k < n - 1 ? k : n - 2);
  }
  std::vector<char> bad((size_t)nb + 1, 0);
  for (int b = 0; b < nb; ++b)
    for (int k = std::min(e[b], e[b + 1]); k <= std::max(e[b], e[b + 1]); ++k)
      if (!clean(k)) bad[b] = bad[b + 1] = 1;
  for (int b = 0; b <= nb; ++b)
    if (bad[b]) e[b] = kNoBin;
  p->rh_sign = sg;
  p->nbins = nb;
  p->bscale = scale;
  return e;
}

#pragma clang fp contract(off)

__device__ __forceinline__ void bisect_dev(const double* c, int n, double v, int* i1o, int* i2o) {
  int i1 = 0, i2 = n - 1;
  while (i2 - i1 > 1) {
    const int im = i1 + (i2 - i1) / 2;
    const double d1 = c[i1] - v, dm = c[im] - v;
    if (d1 * dm > kMinP) i1 = im;
    else i2 = im;
  }
  *i1o = i1;
  *i2o = i2;
}

// What a kernel sees of the table: the three columns it searches and m (in
// LDS or in global memory), one 64-byte record per interval with both ends'
// k, t, b and cp, and the bins of the rho*h search.
struct TabView {
  const double *crh, *ch, *cd, *cm;
  const double* __restrict__ rec;
  const uint16_t* bins;
  int n, nbins, hrise, rhsign;  // nbins 0: bisection only
  double dhmin, dhmax, bscale;
};

// Whether v lies inside interval k of a rising or falling column.  On a
// strictly monotone column the bisection for v then ends in (k, k + 1): every
// sign product it tests left of the interval is at least the square of the
// distance from node k, above kMinP, and none right of it is positive.
__device__ __forceinline__ bool inside(const double* c, int k, double v) { return c[k] + kNodeGap < v && v < c[k + 1]; }
__device__ __forceinline__ bool inside_falling(const double* c, int k, double v) {
  return v + kNodeGap < c[k] && c[k + 1] < v;
}

// The interval of bisect_dev(crh, n, v).  The bin of v (nbins of equal width
// over the column's range) bounds it to the few intervals that meet the bin,
// 1.3 halvings on average for 4096 rows and 8192 bins instead of 12; values
// at or within kNodeGap of a node, where the bisection's result hangs on its
// product test, and values of several intervals take the bisection itself.
__device__ __forceinline__ void find_rhoh(const TabView& t, double v, int* i1o, int* i2o) {
  if (t.nbins) {
    int b = (int)((v - t.dhmin) * t.bscale);
    b = b < 0 ? 0 : b > t.nbins - 1 ? t.nbins - 1 : b;
    const int e0 = t.bins[b], e1 = t.bins[b + 1];
    if (e0 != kNoBin && e1 != kNoBin) {
      int lo = e0 < e1 ? e0 : e1, hi = (e0 < e1 ? e1 : e0) + 1;
      while (hi - lo > 1) {
        const int im = (lo + hi) / 2;
        const double cm = t.crh[im];
        if (t.rhsign > 0 ? cm < v : cm > v) lo = im;
        else hi = im;
      }
      if (t.rhsign > 0 ? inside(t.crh, lo, v) : inside_falling(t.crh, lo, v)) {
        *i1o = lo;
        *i2o = lo + 1;
        return;
      }
    }
  }
  bisect_dev(t.crh, t.n, v, i1o, i2o);
}

// The interval of bisect_dev(ch, n, h), from a guess: the interval of rho*h
// or one of its neighbours on a strictly rising column.
__device__ __forceinline__ void find_h(const TabView& t, double h, int* i1, int* i2) {
  int k = *i1;
  if (t.hrise) {
    if (inside(t.ch, k, h)) return;
    k = h < t.ch[k] ? k - 1 : k + 1;
    if (k >= 0 && k < t.n - 1 && inside(t.ch, k, h)) {
      *i1 = k;
      *i2 = k + 1;
      return;
    }
  }
  bisect_dev(t.ch, t.n, h, i1, i2);
}

// x of lane S of this lane's group of four
template <int S>
__device__ __forceinline__ int quad(int x) {
  return __builtin_amdgcn_mov_dpp(x, 0x55 * S, 0xF, 0xF, true);
}
template <int S>
__device__ __forceinline__ double quad(double x) {
  const int lo = quad<S>(__double2loint(x)), hi = quad<S>(__double2hiint(x));
  return __hiloint2double(hi, lo);
}

// One cell of ftp_refresh_thermal_properties_from_DH: clamp rho*h to the
// table, h from the rho*h column, d from h, h = rho*h / d, then every
// property from that h (src/thermo_info.f90 ftp_refresh_thermal_properties_
// from_DH).  All lanes of a wave take part; those of cells from N on store
// nothing.
//
// Each group of four lanes reads the 64-byte records of its four cells
// together, one record per load and 16 bytes per lane: lane j interpolates
// property j of all four, and the values change lanes within the group.  A
// gather costs the texture unit a clock per cache line, 16 here against 64
// when every lane reads its own record, which then also stalls on the lines
// its first 16 bytes have in flight (58 % of that kernel's time).
struct DhOut {
  double *h, *d, *m, *k, *t, *b, *cp;
  float *fh, *fm, *fk, *ft;
};

__device__ __forceinline__ void props_dh_cell(const TabView& tv, double v, long c, long N, const DhOut& o,
                                              int* __restrict__ flag) {
  const bool live = c < N;
  if (v < tv.dhmin) {
    v = tv.dhmin;
    if (live) atomicAdd(flag, 1);
  } else if (v > tv.dhmax) {
    v = tv.dhmax;
    if (live) atomicAdd(flag, 1);
  }
  const double *crh = tv.crh, *ch = tv.ch, *cd = tv.cd;
  int i1, i2;
  find_rhoh(tv, v, &i1, &i2);
  double w1 = (crh[i2] - v) / (crh[i2] - crh[i1]);
  double w2 = 1.0 - w1;
  double h = w1 * ch[i1] + w2 * ch[i2];
  // properties from h (first pass needs only d)
  find_h(tv, h, &i1, &i2);
  w1 = (ch[i2] - h) / (ch[i2] - ch[i1]);
  w2 = 1.0 - w1;
  const double d1 = w1 * cd[i1] + w2 * cd[i2];
  h = v / d1;
  find_h(tv, h, &i1, &i2);
  const int j = threadIdx.x & 3;
  const double2* rec = reinterpret_cast<const double2*>(tv.rec) + j;  // (i2 is i1 + 1)
  const double2 r0 = rec[4 * (long)quad<0>(i1)], r1 = rec[4 * (long)quad<1>(i1)], r2 = rec[4 * (long)quad<2>(i1)],
                r3 = rec[4 * (long)quad<3>(i1)];
  w1 = (ch[i2] - h) / (ch[i2] - ch[i1]);
  w2 = 1.0 - w1;
  auto put = [&](double* p, float* f, double x) {
    if (p && live) __builtin_nontemporal_store(x, p + c);
    if (f && live) f[c] = (float)x;
  };
  put(o.h, o.fh, h);
  if (o.d) put(o.d, nullptr, w1 * cd[i1] + w2 * cd[i2]);
  if (o.m || o.fm) put(o.m, o.fm, w1 * tv.cm[i1] + w2 * tv.cm[i2]);
  const double x0 = quad<0>(w1) * r0.x + quad<0>(w2) * r0.y, x1 = quad<1>(w1) * r1.x + quad<1>(w2) * r1.y,
               x2 = quad<2>(w1) * r2.x + quad<2>(w2) * r2.y, x3 = quad<3>(w1) * r3.x + quad<3>(w2) * r3.y;
  // property P of this lane's cell: value j of lane P
  auto mine = [&](auto lane) {
    constexpr int P = decltype(lane)::value;
    const double y0 = quad<P>(x0), y1 = quad<P>(x1), y2 = quad<P>(x2), y3 = quad<P>(x3);
    return j < 2 ? (j == 0 ? y0 : y1) : (j == 2 ? y2 : y3);
  };
  if (o.k || o.fk) put(o.k, o.fk, mine(std::integral_constant<int, 0>()));
  if (o.t || o.ft) put(o.t, o.ft, mine(std::integral_constant<int, 1>()));
  if (o.b) put(o.b, nullptr, mine(std::integral_constant<int, 2>()));
  if (o.cp) put(o.cp, nullptr, mine(std::integral_constant<int, 3>()));
}

// Table in global memory (any size): one thread per cell.
__global__ void __launch_bounds__(256) k_props_from_dh(TabView tv, const double* __restrict__ rhoh_in, long N, DhOut o,
                                                       int* __restrict__ flag) {
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  props_dh_cell(tv, c < N ? rhoh_in[c] : tv.dhmin, c, N, o, flag);
}

// The searched columns (rho*h, h, then d and m as far as NC reaches) and the
// bins staged in LDS once per workgroup; a grid of the one or two
// workgroups that fit a CU then walks the cells with a grid stride, so the table crosses L2 once
// per workgroup instead of once per few hundred cells, the next cell's rho*h
// in flight meanwhile.  With full bisections (12 dependent LDS reads) and a
// gather per column and end, 8.4 M cells with seven outputs took 306 us at
// 4096 rows; with the bins, the neighbours and per-lane records 213, with the
// records read by four lanes 185, and with stores that do not displace what
// the L2 holds 106, the rate of a large copy.  Two cells per thread were
// slower (229 against 213).  Every thread reaches the barrier: the staging
// loops run before any thread leaves.
template <int NC>
__global__ void __launch_bounds__(kPropsBlock) k_props_from_dh_lds(TabView tv, const double* __restrict__ rhoh_in,
                                                                   long N, DhOut o, int* __restrict__ flag) {
  extern __shared__ double sh[];
  const int n = tv.n;
  for (int i = threadIdx.x; i < n; i += blockDim.x) {
    sh[i] = tv.crh[i];
    sh[n + i] = tv.ch[i];
    if (NC > 2) sh[2 * n + i] = tv.cd[i];
    if (NC > 3) sh[3 * n + i] = tv.cm[i];
  }
  uint16_t* sb = reinterpret_cast<uint16_t*>(sh + NC * n);
  if (tv.nbins)
    for (int i = threadIdx.x; i <= tv.nbins; i += blockDim.x) sb[i] = tv.bins[i];
  __syncthreads();
  tv.crh = sh;
  tv.ch = sh + n;
  if (NC > 2) tv.cd = sh + 2 * n;
  if (NC > 3) tv.cm = sh + 3 * n;
  tv.bins = sb;
  const long stride = (long)gridDim.x * blockDim.x;
  long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const long lane = threadIdx.x & 63;
  double v = c < N ? rhoh_in[c] : tv.dhmin;
  while (c - lane < N) {  // whole waves
    const long cn = c + stride;
    const double vn = cn < N ? rhoh_in[cn] : tv.dhmin;
    props_dh_cell(tv, v, c, N, o, flag);
    c = cn;
    v = vn;
  }
}

// ftp_refresh_thermal_properties_from_H per cell (no clamping, as the
// reference: outside the table the end segment extrapolates)
template <bool LDS>
__global__ void __launch_bounds__(256) k_props_from_h(const double* __restrict__ tab, int n,
                                                      const double* __restrict__ h_in, long N,
                                                      double* __restrict__ od, double* __restrict__ om,
                                                      double* __restrict__ ok, double* __restrict__ ot,
                                                      double* __restrict__ ob, double* __restrict__ ocp) {
  extern __shared__ double sh[];
  const double* ch = tab + (long)CH * n;
  if (LDS) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) sh[i] = ch[i];
    __syncthreads();
    ch = sh;
  }
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  const double h = h_in[c];
  int i1, i2;
  bisect_dev(ch, n, h, &i1, &i2);
  const double w1 = (ch[i2] - h) / (ch[i2] - ch[i1]);
  const double w2 = 1.0 - w1;
  auto interp = [&](int col) { return w1 * tab[(long)col * n + i1] + w2 * tab[(long)col * n + i2]; };
  if (od) od[c] = interp(CD);
  if (om) om[c] = interp(CM);
  if (ok) ok[c] = interp(CK);
  if (ot) ot[c] = interp(CT);
  if (ob) ob[c] = interp(CB);
  if (ocp) ocp[c] = interp(CCP);
}

#pragma clang fp contract(on)

// Launches the from-rho*h kernel for n cells: the persistent LDS form with
// the bins and as many columns as fit a workgroup's LDS (four to two; four
// columns and the bins of 4096 rows are 144 of its 160 KB), else the global
// form.
// o holds the seven outputs (h, d, m, k, t, b, cp), each possibly null; f
// the FP32 roundings of h, m, k, t (or null).
hipError_t launch_from_dh(const chs_props* p, const double* rhoh, long n, double* const o[7], int* flag,
                          hipStream_t s, float* const* f = nullptr) {
  float* const fz[4] = {nullptr, nullptr, nullptr, nullptr};
  if (!f) f = fz;
  const size_t N = (size_t)p->n, col = sizeof(double) * N;
  const TabView tv{p->dev + CRH * N, p->dev + CH * N, p->dev + CD * N, p->dev + CM * N, p->rec, p->bins, p->n,
                   p->nbins, p->h_rising ? 1 : 0, p->rh_sign, p->dhmin, p->dhmax, p->bscale};
  const DhOut out{o[0], o[1], o[2], o[3], o[4], o[5], o[6], f[0], f[1], f[2], f[3]};
  const size_t extra = p->bins ? sizeof(uint16_t) * ((size_t)p->nbins + 1) : 0;
  int nc = 4;
  while (nc > 1 && nc * col + extra > p->lds_block) --nc;
  if (nc > 1) {
    const long want = (n + kPropsBlock - 1) / kPropsBlock;
    // (a workgroup that waits for another's LDS would stage the table again)
    const long cap = (2 * (nc * col + extra) <= p->lds_block ? 2L : 1L) * (p->cus > 0 ? p->cus : 256);
    const unsigned grid = (unsigned)(want < cap ? want : cap);
    auto* k = nc == 4 ? k_props_from_dh_lds<4> : nc == 3 ? k_props_from_dh_lds<3> : k_props_from_dh_lds<2>;
    hipLaunchKernelGGL(k, dim3(grid), dim3(kPropsBlock), nc * col + extra, s, tv, rhoh, n, out, flag);
  } else {
    hipLaunchKernelGGL(k_props_from_dh, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, tv, rhoh, n, out, flag);
  }
  return hipGetLastError();
}

}  // namespace

namespace chs {
std::string props_refresh_dh(const chs_props* p, int mode, const double* rhoh, long n, double* h, double* d,
                             double* m, double* k, double* t, int* flag, hipStream_t s, float* const* r32) {
  if (n <= 0) return "";
  if (mode == CHS_PROPS_MLP) {
    if (!p->surrogate) return "properties: no surrogate attached to the table";
    return mlp_refresh_dh(p->surrogate, p, rhoh, n, h, d, m, k, t, flag, s, r32);
  }
  if (mode != CHS_PROPS_TABLE) return "properties: unknown mode";
  double* const o[7] = {h, d, m, k, t, nullptr, nullptr};
  const hipError_t e = launch_from_dh(p, rhoh, n, o, flag, s, r32);
  if (e != hipSuccess) return std::string("property kernel: ") + hipGetErrorString(e);
  return "";
}
}  // namespace chs

extern "C" {

int chs_props_set_surrogate(chs_props_t* p, chs_mlp_t* m) {
  if (!p) return fail(CHS_EINVAL, "null handle");
  p->surrogate = m;
  return CHS_OK;
}

int chs_props_create(const double* table, int nrows, double ref_t0, chs_props_t** out) {
  if (!table || !out || nrows < 2) return fail(CHS_EINVAL, "invalid argument");
  *out = nullptr;
  chs_props* p = new chs_props();
  p->n = nrows;
  for (auto& c : p->col) c.resize(nrows);
  for (int i = 0; i < nrows; ++i) {
    const double* r = table + 8 * (size_t)i;
    p->col[CH][i] = r[1];
    p->col[CT][i] = r[2];
    p->col[CD][i] = r[3];
    p->col[CM][i] = r[4];
    p->col[CK][i] = r[5];
    p->col[CCP][i] = r[6];
    p->col[CB][i] = r[7];
    p->col[CRH][i] = r[3] * r[1];
  }
  // selection sort by T (the first minimum wins, as minloc does)
  for (int i = 0; i < nrows; ++i) {
    int kmin = i;
    for (int j = i + 1; j < nrows; ++j)
      if (p->col[CT][j] < p->col[CT][kmin]) kmin = j;
    if (kmin != i)
      for (auto& c : p->col) std::swap(c[i], c[kmin]);
  }
  if (ref_t0 > 0.0) {
    int i1, i2;
    bisect_host(p->col[CT], ref_t0, &i1, &i2);
    const double w1 = (p->col[CT][i2] - ref_t0) / (p->col[CT][i2] - p->col[CT][i1]), w2 = 1.0 - w1;
    auto in = [&](int c) {
      const double a = w1 * p->col[c][i1];
      const double b = w2 * p->col[c][i2];
      return a + b;
    };
    p->ref[0] = ref_t0;
    p->ref[1] = in(CD);
    p->ref[2] = in(CM);
    p->ref[3] = in(CK);
    p->ref[4] = in(CH);
    p->ref[5] = in(CB);
    p->ref[6] = in(CCP);
    for (int i = 0; i < nrows; ++i) {
      p->col[CT][i] = p->col[CT][i] / p->ref[0];
      p->col[CD][i] = p->col[CD][i] / p->ref[1];
      p->col[CM][i] = p->col[CM][i] / p->ref[2];
      p->col[CK][i] = p->col[CK][i] / p->ref[3];
      p->col[CB][i] = p->col[CB][i] / p->ref[5];
      p->col[CCP][i] = p->col[CCP][i] / p->ref[6];
      p->col[CH][i] = (p->col[CH][i] - p->ref[4]) / p->ref[0] / p->ref[6];
      p->col[CRH][i] = p->col[CD][i] * p->col[CH][i];
    }
  }
  // ref_t0 <= 0: the rows are already non-dimensional (ref stays zero)
  int imin = 0, imax = 0;
  for (int i = 1; i < nrows; ++i) {
    if (p->col[CRH][i] < p->col[CRH][imin]) imin = i;
    if (p->col[CRH][i] > p->col[CRH][imax]) imax = i;
  }
  p->dhmin = p->col[CRH][imin];
  p->dhmax = p->col[CRH][imax];
  p->h_rising = true;
  for (int i = 1; i < nrows; ++i)
    if (!(p->col[CH][i] > p->col[CH][i - 1])) p->h_rising = false;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
    delete p;
    return fail(CHS_EHIP, "no HIP device");
  }
  int dev = 0, v = 0;
  if (hipGetDevice(&dev) == hipSuccess) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess && v > 0)
      p->lds_block = (size_t)v;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0) p->cus = v;
  }
  std::vector<double> flat(8 * (size_t)nrows);
  for (int c = 0; c < 8; ++c) std::memcpy(flat.data() + (size_t)c * nrows, p->col[c].data(), sizeof(double) * nrows);
  if (hipStreamCreate(&p->stream) != hipSuccess || hipMalloc(&p->dev, sizeof(double) * flat.size()) != hipSuccess ||
      hipMalloc(&p->flag, sizeof(int)) != hipSuccess ||
      hipMemcpy(p->dev, flat.data(), sizeof(double) * flat.size(), hipMemcpyHostToDevice) != hipSuccess) {
    delete p;
    return fail(CHS_ENOMEM, "device allocation failed");
  }
  std::vector<double> rec(8 * (size_t)nrows, 0.0);
  const int rc[4] = {CK, CT, CB, CCP};
  for (int i = 0; i + 1 < nrows; ++i)
    for (int q = 0; q < 4; ++q) {
      rec[8 * (size_t)i + 2 * q] = p->col[rc[q]][i];
      rec[8 * (size_t)i + 2 * q + 1] = p->col[rc[q]][i + 1];
    }
  const std::vector<uint16_t> bins = rhoh_bins(p);
  if (hipMalloc(&p->rec, sizeof(double) * rec.size()) != hipSuccess ||
      hipMemcpy(p->rec, rec.data(), sizeof(double) * rec.size(), hipMemcpyHostToDevice) != hipSuccess ||
      (!bins.empty() &&
       (hipMalloc(&p->bins, sizeof(uint16_t) * bins.size()) != hipSuccess ||
        hipMemcpy(p->bins, bins.data(), sizeof(uint16_t) * bins.size(), hipMemcpyHostToDevice) != hipSuccess))) {
    delete p;
    return fail(CHS_ENOMEM, "device allocation failed");
  }
  *out = p;
  return CHS_OK;
}

int chs_props_destroy(chs_props_t* p) {
  if (!p) return CHS_OK;
  if (p->stream) (void)hipStreamSynchronize(p->stream);
  delete p;
  return CHS_OK;
}

int chs_props_info(const chs_props_t* p, double* dhmin, double* dhmax, double ref[7]) {
  if (!p) return fail(CHS_EINVAL, "null handle");
  if (dhmin) *dhmin = p->dhmin;
  if (dhmax) *dhmax = p->dhmax;
  if (ref)
    for (int i = 0; i < 7; ++i) ref[i] = p->ref[i];
  return CHS_OK;
}

int chs_props_from_rhoh(chs_props_t* p, const double* rhoh, long n, double* h, double* d, double* m, double* k,
                        double* t, double* b, double* cp, int mode, int mem) {
  if (!p || !rhoh || n < 0) return fail(CHS_EINVAL, "invalid argument");
  if (mode != CHS_PROPS_TABLE && mode != CHS_PROPS_MLP) return fail(CHS_EUNSUP, "unknown property mode");
  if (mode == CHS_PROPS_MLP && !p->surrogate) return fail(CHS_EINVAL, "no surrogate attached to the table");
  if (mode == CHS_PROPS_MLP && (b || cp)) return fail(CHS_EUNSUP, "the surrogate gives h, d, m, k and t only");
  if (mem != CHS_MEM_HOST && mem != CHS_MEM_DEVICE) return fail(CHS_EINVAL, "invalid mem kind");
  if (n == 0) return CHS_OK;
  double* outs[7] = {h, d, m, k, t, b, cp};
  const double* din = rhoh;
  double* dout[7] = {h, d, m, k, t, b, cp};
  if (mem == CHS_MEM_HOST) {
    int nout = 0;
    for (double* o : outs) nout += o != nullptr;
    const size_t need = sizeof(double) * (size_t)n * (1 + nout);
    if (need > p->io_bytes) {
      if (p->io) (void)hipFree(p->io);
      p->io = nullptr;
      p->io_bytes = 0;
      if (hipMalloc(&p->io, need) != hipSuccess) return fail(CHS_ENOMEM, "staging allocation failed");
      p->io_bytes = need;
    }
    double* base = static_cast<double*>(p->io);
    if (hipMemcpyAsync(base, rhoh, sizeof(double) * n, hipMemcpyHostToDevice, p->stream) != hipSuccess)
      return fail(CHS_EHIP, "copy in");
    din = base;
    int slot = 1;
    for (int q = 0; q < 7; ++q) dout[q] = outs[q] ? base + (size_t)n * slot++ : nullptr;
  }
  if (hipMemsetAsync(p->flag, 0, sizeof(int), p->stream) != hipSuccess) return fail(CHS_EHIP, "flag reset");
  const unsigned grid = (unsigned)((n + 255) / 256);
  if (mode == CHS_PROPS_MLP) {
    const std::string e = chs::mlp_refresh_dh(p->surrogate, p, din, n, dout[0], dout[1], dout[2], dout[3], dout[4],
                                              p->flag, p->stream);
    if (!e.empty()) return fail(CHS_EHIP, e);
  } else if (launch_from_dh(p, din, n, dout, p->flag, p->stream) != hipSuccess) {
    return fail(CHS_EHIP, "property kernel launch");
  }
  if (mem == CHS_MEM_HOST)
    for (int q = 0; q < 7; ++q)
      if (outs[q] && hipMemcpyAsync(outs[q], dout[q], sizeof(double) * n, hipMemcpyDeviceToHost, p->stream) !=
                         hipSuccess)
        return fail(CHS_EHIP, "copy out");
  int nbad = 0;
  if (hipMemcpyAsync(&nbad, p->flag, sizeof(int), hipMemcpyDeviceToHost, p->stream) != hipSuccess ||
      hipStreamSynchronize(p->stream) != hipSuccess)
    return fail(CHS_EHIP, "synchronise");
  if (nbad) return fail(CHS_ERANGE, "rho*h is out of range (" + std::to_string(nbad) + " cells clamped)");
  return CHS_OK;
}

int chs_props_from_h(chs_props_t* p, const double* h, long n, double* d, double* m, double* k, double* t,
                     double* b, double* cp, int mem) {
  if (!p || !h || n < 0) return fail(CHS_EINVAL, "invalid argument");
  if (mem != CHS_MEM_HOST && mem != CHS_MEM_DEVICE) return fail(CHS_EINVAL, "invalid mem kind");
  if (n == 0) return CHS_OK;
  double* outs[6] = {d, m, k, t, b, cp};
  const double* din = h;
  double* dout[6] = {d, m, k, t, b, cp};
  if (mem == CHS_MEM_HOST) {
    int nout = 0;
    for (double* o : outs) nout += o != nullptr;
    const size_t need = sizeof(double) * (size_t)n * (1 + nout);
    if (need > p->io_bytes) {
      if (p->io) (void)hipFree(p->io);
      p->io = nullptr;
      p->io_bytes = 0;
      if (hipMalloc(&p->io, need) != hipSuccess) return fail(CHS_ENOMEM, "staging allocation failed");
      p->io_bytes = need;
    }
    double* base = static_cast<double*>(p->io);
    if (hipMemcpyAsync(base, h, sizeof(double) * n, hipMemcpyHostToDevice, p->stream) != hipSuccess)
      return fail(CHS_EHIP, "copy in");
    din = base;
    int slot = 1;
    for (int q = 0; q < 6; ++q) dout[q] = outs[q] ? base + (size_t)n * slot++ : nullptr;
  }
  const unsigned grid = (unsigned)((n + 255) / 256);
  if (p->n <= 3 * kPropsLds)
    hipLaunchKernelGGL(k_props_from_h<true>, dim3(grid), dim3(256), sizeof(double) * (size_t)p->n, p->stream, p->dev,
                       p->n, din, n, dout[0], dout[1], dout[2], dout[3], dout[4], dout[5]);
  else
    hipLaunchKernelGGL(k_props_from_h<false>, dim3(grid), dim3(256), 0, p->stream, p->dev, p->n, din, n, dout[0],
                       dout[1], dout[2], dout[3], dout[4], dout[5]);
  if (hipGetLastError() != hipSuccess) return fail(CHS_EHIP, "property kernel launch");
  if (mem == CHS_MEM_HOST)
    for (int q = 0; q < 6; ++q)
      if (outs[q] && hipMemcpyAsync(outs[q], dout[q], sizeof(double) * n, hipMemcpyDeviceToHost, p->stream) !=
                         hipSuccess)
        return fail(CHS_EHIP, "copy out");
  if (hipStreamSynchronize(p->stream) != hipSuccess) return fail(CHS_EHIP, "synchronise");
  return CHS_OK;
}

}  // extern "C"
