// Plans of the fused line operators (chs_rhs.h) and the wall flux.
#include "chs_rhs_dev.h"

#include <cmath>
#include <cstring>
#include <vector>

namespace chs {

#define RCHK(x)                                                             \
  do {                                                                      \
    hipError_t e_ = (x);                                                    \
    if (e_ != hipSuccess) return std::string(#x ": ") + hipGetErrorString(e_); \
  } while (0)

bool fuse_chunks(int dir, int n, bool short_form, int* P, int* ell, int* rows) {
  const int ch = short_form ? 8 : 16;
  if (n < 8) return false;
  const int whole = (n + ch - 1) / ch;
  if (dir == 0 || (n % ch == 0 && whole <= kFuseChunks)) {
    *P = whole;
    *ell = *rows = ch;
    return whole <= kFuseChunks && n - ch * (whole - 1) >= 2;
  }
  for (int p = (n + ch) / (ch + 1); p <= kFuseChunks; ++p) {
    const int l = (n + p - 1) / p;
    if (n - l * (p - 1) >= 2 && (p == 1 || 2 * l >= ch)) {
      *P = p;
      *ell = l;
      *rows = l <= ch ? ch : ch + 1;
      return true;
    }
  }
  return false;
}

template <typename T>
DevFusePlan<T>::~DevFusePlan() {
  if (mem) (void)hipFree(mem);
}

template <typename T>
std::string upload_fuse_plan(const LinePlan& p, int rows, DevFusePlan<T>* out) {
  const int NB = fuse_band<T>(rows);
  out->ok = false;
  out->rows = rows;
  const bool to_node = p.op == MIDP_C2P || p.op == D1_C2P;
  if (!to_node && p.op != MIDP_P2C && p.op != D1_P2C) return "";
  const int P = p.part_P, ell = p.part_ch, W = rows + 3, M = 2 * P;
  if (P < 1 || P > kFuseChunks || ell > rows || (p.dir == 0 && ell != rows) || (int)p.part_start.size() != P + 1) return "";
  const bool wrap = p.ibc[0] == BC_PERIODIC;
  if (wrap && (p.has_fbc || p.n_in < 10)) return "";
  FusePlan<T>& k = out->k;
  k = FusePlan<T>{};
  k.n_in = p.n_in; k.n_out = p.n_out; k.P = P; k.ell = ell;
  k.solve = p.solve != 0; k.wrap = wrap ? 1 : 0;
  k.sh = to_node ? 0 : 1;
  k.sgn = T(p.sgn);
  k.c1 = T(p.c1 * p.dd); k.c2 = T(p.c2 * p.dd);
  k.neu_lo = p.neu_lo; k.neu_hi = p.neu_hi;
  // boundary rows: the bulk stencil on the wrapped line, or weights of their own
  std::vector<double> edge((size_t)4 * (W + 4), 0.0);
  if (wrap) {
    const int at[4] = {0, 1, p.n_out - 2, p.n_out - 1};
    for (int q = 0; q < 4; ++q) {
      std::vector<double> a(p.n_in, 0.0), b(p.n_in, 0.0);
      for (int t = 0; t < p.rows[q].nterm; ++t) a[p.rows[q].idx[t]] += p.rows[q].w[t];
      auto wi = [&](int e) { return ((e % p.n_in) + p.n_in) % p.n_in; };
      b[wi(at[q] + p.p1)] += p.c1;
      b[wi(at[q] + p.p2)] += p.sgn * p.c1;
      b[wi(at[q] + p.p3)] += p.c2;
      b[wi(at[q] + p.p4)] += p.sgn * p.c2;
      double mag = 0.0;
      for (double v : b) mag = std::max(mag, std::fabs(v));
      for (int e = 0; e < p.n_in; ++e)
        if (std::fabs(a[e] - b[e]) > 1e-14 * mag) return "";
    }
  } else {
    k.ends = 1;
    for (int q = 0; q < 4; ++q) {
      const int s0 = q < 2 ? 0 : p.part_start[P - 1];
      // (rows n-2 and n-1 belong to the last chunk, rows 0 and 1 to the first)
      for (int t = 0; t < p.rows[q].nterm; ++t) {
        int slot = -1;
        for (int u = 0; u < W && slot < 0; ++u) {
          const int e = s0 - 2 + k.sh + u;
          if (e == p.rows[q].idx[t] && e >= 0 && e < p.n_in) slot = u;
        }
        if (slot < 0) return "";
        edge[(size_t)q * (W + 4) + slot] += p.rows[q].w[t] * p.dd;
      }
      for (int m = 0; m < 4; ++m) edge[(size_t)q * (W + 4) + W + m] = p.has_fbc ? p.rows[q].u[m] * p.dd : 0.0;
    }
    if (P > 1 && (p.part_start[1] < 2 || p.n_out - p.part_start[P - 1] < 2)) return "";
    if (P == 1 && p.n_out < 4) return "";
  }

  // coefficient rows of the first, the inner and the last chunk; every inner
  // chunk must have those of chunk 1
  auto chunk_rows_of = [&](int q, std::vector<double>* c) {
    c->assign((size_t)rows * kFuseCo, 0.0);
    const int s0 = p.part_start[q], len = p.part_start[q + 1] - s0;
    for (int i = 0; i < rows; ++i) {
      double* r = c->data() + (size_t)i * kFuseCo;
      if (p.ld.empty()) continue;
      if (i >= len) {  // y[i] = y[i - 1]
        r[FC_AL] = -1.0;
        continue;
      }
      r[FC_LD] = p.ld[s0 + i];
      r[FC_AL] = i > 0 ? p.a_raw[s0 + i] * p.ld[s0 + i] : 0.0;
      r[FC_LC] = i < len - 1 ? p.lc[s0 + i] : 0.0;
      r[FC_SV] = p.sv[s0 + i];
      r[FC_SW] = p.sw[s0 + i];
    }
  };
  std::vector<double> tab, c;
  for (int cls = 0; cls < 3; ++cls) {
    const int q = cls == 0 ? 0 : cls == 1 ? std::min(1, P - 1) : P - 1;
    chunk_rows_of(q, &c);
    tab.insert(tab.end(), c.begin(), c.end());
  }
  for (int q = 1; q < P - 1; ++q) {
    chunk_rows_of(q, &c);
    if (std::memcmp(c.data(), tab.data() + (size_t)rows * kFuseCo, sizeof(double) * c.size()) != 0) return "";
  }
  // coupling weights: the rows of the inverse for the previous chunk's last
  // and the next chunk's first value, over the ends around the chunk
  std::vector<double> cp((size_t)P * 2 * NB, 0.0);
  if (p.solve) {
    const double drop = sizeof(T) == 8 ? std::ldexp(1.0, -59) : std::ldexp(1.0, -36);
    for (int q = 0; q < P; ++q)
      for (int side = 0; side < 2; ++side) {
        if (!wrap && (side == 0 ? q == 0 : q == P - 1)) continue;
        const int row = side == 0 ? 2 * ((q + P - 1) % P) + 1 : 2 * ((q + 1) % P);
        const double* R = &p.rinv[(size_t)row * M];
        double mag = 0.0;
        for (int j = 0; j < M; ++j) mag = std::max(mag, std::fabs(R[j]));
        std::vector<char> seen(M, 0);
        for (int j = 0; j < NB; ++j) {
          int e = 2 * q - (NB / 2 - 1) + j;
          if (wrap) e = ((e % M) + M) % M;
          if (e < 0 || e >= M || seen[e]) continue;
          seen[e] = 1;
          cp[((size_t)q * 2 + side) * NB + j] = R[e];
        }
        for (int e = 0; e < M; ++e)
          if (!seen[e] && std::fabs(R[e]) > drop * mag) return "";
      }
  }
  tab.insert(tab.end(), cp.begin(), cp.end());
  std::vector<double> met((size_t)P * ell, 1.0);
  for (int r = 0; r < p.n_out && !p.metric.empty(); ++r) {
    met[r] = p.metric[r];
    if (p.metric[r] != 1.0) k.met = 1;
  }
  if (k.met) tab.insert(tab.end(), met.begin(), met.end());
  while (tab.size() % 4) tab.push_back(0.0);  // (16-byte copies into LDS)
  k.ntab = (int)tab.size();
  tab.insert(tab.end(), edge.begin(), edge.end());
  std::vector<T> t(tab.begin(), tab.end());
  RCHK(hipMalloc(&out->mem, sizeof(T) * t.size()));
  RCHK(hipMemcpy(out->mem, t.data(), sizeof(T) * t.size(), hipMemcpyHostToDevice));
  k.tab = out->mem;
  k.edge = out->mem + k.ntab;
  out->ok = true;
  return "";
}

// One thread per (x, z) line: both walls' dv/dy from the end-row recipes, then
// the wall flux into rows s and s + 2 (what the boundary rows read).
template <typename T>
__global__ void __launch_bounds__(64) k_wall_flux(const DevRow<T>* rows, const T* __restrict__ v, const T* __restrict__ fbc,
                                                  int e1, int e2, int e3, int n_out, T dd, T b0, int solve,
                                                  const T* __restrict__ d, const T* __restrict__ metric, T r,
                                                  T* __restrict__ flux) {
  const long L = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (L >= (long)e1 * e3) return;
  const long i = L % e1, k = L / e1;
  const long fb = i + (long)e1 * 4 * k;
  T fb4[4];
  for (int m = 0; m < 4; ++m) fb4[m] = fbc[fb + (long)e1 * m];
  for (int s = 0; s < 2; ++s) {
    const DevRow<T>& R = rows[s ? 3 : 0];
    const int row = s ? n_out - 1 : 0;
    T dy = T(0);
    for (int t = 0; t < R.nterm; ++t) dy = dy + R.w[t] * v[i + (long)e1 * (R.idx[t] + (long)e2 * k)];
    for (int m = 0; m < 4; ++m) dy = dy + R.u[m] * fb4[m];
    dy = dy * dd;
    if (solve) dy = s ? dy * d[row] : dy / b0;
    if (metric) dy = dy * metric[row];
    const T vs = (dy - T(1.0 / 3.0) * dy) * T(2);
    const T f = -fb4[s] * fb4[s] + r * vs;
    flux[fb + (long)e1 * s] = f;
    flux[fb + (long)e1 * (s + 2)] = f;
  }
}

template <typename T>
std::string launch_wall_flux(const DevPlan<T>& D, const Ext3& ein, const T* qyiy, const T* fbc, T r, T* flux,
                             hipStream_t s) {
  const LinePlan& p = D.host;
  if (p.dir != 1 || !fbc || !p.has_fbc || ein.n[1] != p.n_in || p.solve == 2) return "wall flux: not a wall-bounded y plan";
  if (p.solve == 1) {
    const int n = p.n_out;
    if (!(p.b0 == 1.0 && p.c[0] == 0.0 && p.a[n - 1] == 0.0 && p.d[n - 1] == 1.0))
      return "wall flux: end rows are coupled to the line";
  }
  const long n = (long)ein.n[0] * ein.n[2];
  if (n <= 0) return "";
  hipLaunchKernelGGL(k_wall_flux<T>, dim3((unsigned)((n + 63) / 64)), dim3(64), 0, s, D.rows, qyiy, fbc, ein.n[0], ein.n[1],
                     ein.n[2], p.n_out, T(p.dd), T(p.b0), p.solve, D.d, D.metric, r, flux);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? "" : std::string("wall flux launch: ") + hipGetErrorString(e);
}

template struct DevFusePlan<double>;
template struct DevFusePlan<float>;
template std::string upload_fuse_plan<double>(const LinePlan&, int, DevFusePlan<double>*);
template std::string upload_fuse_plan<float>(const LinePlan&, int, DevFusePlan<float>*);
template std::string launch_wall_flux<double>(const DevPlan<double>&, const Ext3&, const double*, const double*, double,
                                              double*, hipStream_t);
template std::string launch_wall_flux<float>(const DevPlan<float>&, const Ext3&, const float*, const float*, float, float*,
                                             hipStream_t);

}  // namespace chs
