// Batched transforms (chs_fft.h): two-pass register kernels for the usual
// lengths, LDS-resident Stockham kernels (radix 4/2/3/5, a workgroup per tile
// of lines) for any other 2,3,5-smooth one.  Included by chs_fft64.hip and
// chs_fft32.hip, which instantiate it.
#include "chs_fft.h"

#include <string>

#include "chs_tune.h"

namespace chs {

constexpr int kThreads = 256;

template <typename T, int R>
__device__ inline void small_dft(cx<T>* v, T s) {
  if constexpr (R == 2) {
    cx<T> a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 4) {
    cx<T> t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    cx<T> t2 = cadd(v[1], v[3]), t3 = cmuli(csub(v[1], v[3]), s);
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
  } else if constexpr (R == 3) {
    const T h = T(0.5), q = T(0.86602540378443864676);
    cx<T> t = cadd(v[1], v[2]), u = cmuli(csub(v[1], v[2]), s * q);
    cx<T> m = csub(v[0], cscale(t, h));
    v[0] = cadd(v[0], t);
    v[1] = cadd(m, u);
    v[2] = csub(m, u);
  } else {  // R == 5
    const T c1 = T(0.30901699437494742410), c2 = T(-0.80901699437494742410);
    const T s1 = T(0.95105651629515357212), s2 = T(0.58778525229247312917);
    cx<T> a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]);
    cx<T> a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
    cx<T> m1 = cadd(v[0], cadd(cscale(a1, c1), cscale(a2, c2)));
    cx<T> m2 = cadd(v[0], cadd(cscale(a1, c2), cscale(a2, c1)));
    cx<T> n1 = cmuli(cadd(cscale(b1, s1), cscale(b2, s2)), s);
    cx<T> n2 = cmuli(csub(cscale(b1, s2), cscale(b2, s1)), s);
    v[0] = cadd(v[0], cadd(a1, a2));
    v[1] = cadd(m1, n1);
    v[4] = csub(m1, n1);
    v[2] = cadd(m2, n2);
    v[3] = csub(m2, n2);
  }
}

// One Stockham stage over `nl` lines of Nc points held in LDS (in place: all
// inputs are read into registers before the barrier, outputs written after).
template <typename T, int R>
__device__ void stage(cx<T>* buf, int Nc, int nl, int Ns, const cx<T>* tw, T s) {
  constexpr int QMAX = (16 + R - 1) / R;
  const int nb = Nc / R;
  const int total = nl * nb;
  const int tstep = Nc / (Ns * R);
  cx<T> v[QMAX][R];
  int bidx[QMAX];
#pragma unroll
  for (int q = 0; q < QMAX; ++q) {
    int b = threadIdx.x + q * kThreads;
    bidx[q] = b;
    if (b < total) {
      int line = b / nb, j = b % nb;
      int k = j % Ns;
      const cx<T>* src = buf + line * Nc + j;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        cx<T> x = src[r * nb];
        if (r > 0 && k > 0) {
          cx<T> w = tw[r * k * tstep];
          w.im = s < T(0) ? w.im : -w.im;
          x = cmul(x, w);
        }
        v[q][r] = x;
      }
      small_dft<T, R>(v[q], s);
    }
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < QMAX; ++q) {
    int b = bidx[q];
    if (b < total) {
      int line = b / nb, j = b % nb;
      int k = j % Ns;
      cx<T>* dst = buf + line * Nc + (j / Ns) * Ns * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) dst[r * Ns] = v[q][r];
    }
  }
  __syncthreads();
}

template <typename T>
__device__ void fft_tile(cx<T>* buf, int Nc, int nl, const Radices& rp, const cx<T>* tw, T s) {
  int Ns = 1;
  for (int q = 0; q < rp.n; ++q) {
    switch (rp.r[q]) {
      case 2: stage<T, 2>(buf, Nc, nl, Ns, tw, s); break;
      case 3: stage<T, 3>(buf, Nc, nl, Ns, tw, s); break;
      case 4: stage<T, 4>(buf, Nc, nl, Ns, tw, s); break;
      default: stage<T, 5>(buf, Nc, nl, Ns, tw, s); break;
    }
    Ns *= rp.r[q];
  }
}

// x forward: real lines (nx) -> complex spectrum kx = 0..nx/2 into W.
template <typename T>
__global__ void __launch_bounds__(kThreads) k_fft_x_fwd(const T* __restrict__ in, cx<T>* __restrict__ W, int nx,
                                                       long nlines, Radices rp, const cx<T>* tw, const cx<T>* rot,
                                                       T in_scale) {
  extern __shared__ unsigned char smem[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
  const int N = nx / 2, nxh = N + 1;
  const int lpb = kTileC / N;
  const long L0 = (long)blockIdx.x * lpb;
  const int nl = (int)((nlines - L0) < lpb ? (nlines - L0) : lpb);
  for (int t = threadIdx.x; t < nl * N; t += kThreads) {
    int line = t / N, n = t % N;
    const T* src = in + (L0 + line) * nx;
    buf[t] = {src[2 * n] * in_scale, src[2 * n + 1] * in_scale};
  }
  __syncthreads();
  fft_tile<T>(buf, N, nl, rp, tw, T(-1));
  for (int t = threadIdx.x; t < nl * nxh; t += kThreads) {
    int line = t / nxh, k = t % nxh;
    cx<T> zk = buf[line * N + (k % N)];
    cx<T> zn = buf[line * N + ((N - k) % N)];
    zn.im = -zn.im;  // conj(Z[N-k])
    cx<T> e = cscale(cadd(zk, zn), T(0.5));
    cx<T> d = csub(zk, zn);
    cx<T> o = {d.im * T(0.5), -d.re * T(0.5)};  // (Z - conj)/(2i)
    cx<T> x = cadd(e, cmul(rot[k], o));
    W[(L0 + line) * nxh + k] = x;
  }
}

// x inverse: complex spectrum kx = 0..nx/2 -> real lines, times `scale`.
template <typename T>
__global__ void __launch_bounds__(kThreads) k_fft_x_inv(const cx<T>* __restrict__ W, T* __restrict__ out, int nx,
                                                       long nlines, Radices rp, const cx<T>* tw, const cx<T>* rot,
                                                       T scale) {
  extern __shared__ unsigned char smem[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
  const int N = nx / 2, nxh = N + 1;
  const int lpb = kTileC / N;
  const long L0 = (long)blockIdx.x * lpb;
  const int nl = (int)((nlines - L0) < lpb ? (nlines - L0) : lpb);
  for (int t = threadIdx.x; t < nl * N; t += kThreads) {
    int line = t / N, k = t % N;
    const cx<T>* src = W + (L0 + line) * nxh;
    cx<T> xk = src[k], xn = src[N - k];
    xn.im = -xn.im;  // conj(X[N-k])
    cx<T> e = cadd(xk, xn);
    cx<T> r = rot[k];
    r.im = -r.im;  // exp(+2 pi i k / nx)
    cx<T> o = cmul(csub(xk, xn), r);
    buf[t] = {e.re - o.im, e.im + o.re};  // e + i*o
  }
  __syncthreads();
  fft_tile<T>(buf, N, nl, rp, tw, T(1));
  for (int t = threadIdx.x; t < nl * N; t += kThreads) {
    int line = t / N, n = t % N;
    T* dst = out + (L0 + line) * nx;
    cx<T> z = buf[t];
    dst[2 * n] = z.re * scale;
    dst[2 * n + 1] = z.im * scale;
  }
}

// Complex transform (either sign) in place along one strided dimension of the
// spectrum W(nxh, ny, nz): lines of n points at stride ls, for every kx (tiles
// of consecutive kx, so loads and stores are contiguous along kx) and every
// value of the remaining index (count no, stride os).  z: n = nz,
// ls = nxh*ny, os = nxh; y: n = ny, ls = nxh, os = nxh*ny.
template <typename T>
__global__ void __launch_bounds__(kThreads) k_fft_s(cx<T>* __restrict__ W, int nxh, int n, long ls, int no, long os,
                                                   Radices rp, const cx<T>* tw, T s) {
  extern __shared__ unsigned char smem[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
  const int lpb = kTileC / n;
  const int ntile = (nxh + lpb - 1) / lpb;
  const int tile = blockIdx.x % ntile, o = blockIdx.x / ntile;
  if (o >= no) return;
  const int kx0 = tile * lpb;
  const int nl = (nxh - kx0) < lpb ? (nxh - kx0) : lpb;
  const long base = kx0 + os * o;
  for (int t = threadIdx.x; t < nl * n; t += kThreads) {
    int m = t / nl, line = t % nl;
    buf[line * n + m] = W[base + line + ls * m];
  }
  __syncthreads();
  fft_tile<T>(buf, n, nl, rp, tw, s);
  for (int t = threadIdx.x; t < nl * n; t += kThreads) {
    int m = t / nl, line = t % nl;
    W[base + line + ls * m] = buf[line * n + m];
  }
}

// ---------------------------------------------------------------------------
// Two-pass transforms for N = A * B (A, B <= 32).  With n = a + A b
// and k = k2 + B k1 (a, k1 < A; b, k2 < B):
//   X[k2 + B k1] = sum_a W_A^(a k1) [ W_N^(a k2) sum_b x[a + A b] W_B^(b k2) ].
// A threads per line: thread a loads x[a + A b] for all b and does the
// B-point DFT in registers, applies W_N^(a k2) (table, index a k2 < N), and
// writes to LDS (rows of A + 1 entries, so the A-point reads of pass 2 hit
// distinct banks); after one barrier, thread a does the A-point DFTs for
// k2 = a, a + A, ... < B in registers.  The register DFTs of power-of-two
// length are radix-2 with compile-time twiddles W_32^m = (-i)^(m/8)
// W_32^(m%8) from the first octant below, exactly symmetric; other lengths go
// by their factors 2 to 5.
__device__ constexpr double kOctC[8] = {1.0, 0.9807852804032304, 0.9238795325112867, 0.8314696123025452,
                                        0.7071067811865476, 0.5555702330196022, 0.3826834323650898,
                                        0.19509032201612825};
__device__ constexpr double kOctS[8] = {0.0, 0.19509032201612825, 0.3826834323650898, 0.5555702330196022,
                                        0.7071067811865476, 0.8314696123025452, 0.9238795325112867,
                                        0.9807852804032304};

// v * W_32^m, W = exp(-2 pi i / 32) (forward) or its conjugate (inverse)
template <typename T, bool FWD>
__device__ __forceinline__ cx<T> tw32(cx<T> v, int m) {
  m &= 31;
  const int q = m >> 3, r = m & 7;
  cx<T> t = v;
  if (r != 0) {
    const T c = T(kOctC[r]), sn = FWD ? T(-kOctS[r]) : T(kOctS[r]);
    t = {v.re * c - v.im * sn, v.re * sn + v.im * c};
  }
  // times (-i)^q (forward) or (+i)^q (inverse)
  if (q == 1) t = FWD ? cx<T>{t.im, -t.re} : cx<T>{-t.im, t.re};
  if (q == 2) t = {-t.re, -t.im};
  if (q == 3) t = FWD ? cx<T>{-t.im, t.re} : cx<T>{t.im, -t.re};
  return t;
}

__host__ __device__ constexpr int bitrev_c(int i, int R) {
  int r = 0;
  for (int b = 1; b < R; b <<= 1) {
    r = (r << 1) | (i & 1);
    i >>= 1;
  }
  return r;
}

// In-register DFT of R = 2^p <= 32 points (radix-2, decimation in time).
template <typename T, int R, bool FWD>
__device__ __forceinline__ void dft_reg(cx<T> (&v)[R]) {
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int j = bitrev_c(i, R);
    if (j > i) {
      const cx<T> t = v[i];
      v[i] = v[j];
      v[j] = t;
    }
  }
#pragma unroll
  for (int len = 2; len <= R; len <<= 1) {
#pragma unroll
    for (int i = 0; i < R; i += len) {
#pragma unroll
      for (int k = 0; k < len / 2; ++k) {
        const cx<T> u = v[i + k];
        const cx<T> t = tw32<T, FWD>(v[i + k + len / 2], k * (32 / len));
        v[i + k] = cadd(u, t);
        v[i + k + len / 2] = csub(u, t);
      }
    }
  }
}

// cos and sin of 2 pi m / R at compile time, from the first octant (Taylor
// series on [0, pi / 4]), so that symmetric twiddles are exactly symmetric.
struct CosSin {
  double c, s;
};
constexpr CosSin octant(double x) {  // 0 <= x <= pi / 4
  double c = 1.0, s = x, t = 1.0;
  for (int k = 2; k <= 22; k += 2) {
    t = -t * x * x / (k * (k - 1.0));
    c += t;
    s += t * x / (k + 1.0);
  }
  return {c, s};
}
constexpr CosSin turn(int m, int R) {
  const double q = 0.78539816339744830962;  // pi / 4
  m %= R;
  const int o = 8 * m / R, r = 8 * m - o * R;
  const CosSin a = octant(q * r / R), b = octant(q * (R - r) / R);  // past the octant, short of the next
  switch (o) {
    case 0: return {a.c, a.s};
    case 1: return {b.s, b.c};
    case 2: return {-a.s, a.c};
    case 3: return {-b.c, b.s};
    case 4: return {-a.c, -a.s};
    case 5: return {-b.s, -b.c};
    case 6: return {a.s, -a.c};
    default: return {b.c, -b.s};
  }
}
template <int R>
struct Turns {
  double c[R], s[R];
  constexpr Turns() : c{}, s{} {
    for (int m = 0; m < R; ++m) {
      const CosSin t = turn(m, R);
      c[m] = t.c;
      s[m] = t.s;
    }
  }
};

// First factor of a composite length that is not a power of two.
constexpr int first_factor(int R) { return R % 4 == 0 ? 4 : R % 3 == 0 ? 3 : R % 2 == 0 ? 2 : 5; }

// In-register DFT of R points: radix-2 for powers of two, else by factors with
// compile-time twiddles (n = n1 + R1 n2, k = k2 + R2 k1).
template <typename T, int R, bool FWD>
__device__ __forceinline__ void dft_any(cx<T> (&v)[R]) {
  if constexpr ((R & (R - 1)) == 0) {
    dft_reg<T, R, FWD>(v);
  } else if constexpr (R == 3 || R == 5) {
    small_dft<T, R>(v, FWD ? T(-1) : T(1));
  } else {
    constexpr int R1 = first_factor(R), R2 = R / R1;
    constexpr Turns<R> tw;
    cx<T> a[R1][R2];
#pragma unroll
    for (int n1 = 0; n1 < R1; ++n1) {
#pragma unroll
      for (int n2 = 0; n2 < R2; ++n2) a[n1][n2] = v[n1 + R1 * n2];
      dft_any<T, R2, FWD>(a[n1]);
    }
#pragma unroll
    for (int k2 = 0; k2 < R2; ++k2) {
      cx<T> b[R1];
#pragma unroll
      for (int n1 = 0; n1 < R1; ++n1) {
        const cx<T> w = {T(tw.c[n1 * k2]), FWD ? T(-tw.s[n1 * k2]) : T(tw.s[n1 * k2])};
        b[n1] = n1 * k2 == 0 ? a[n1][k2] : cmul(a[n1][k2], w);
      }
      dft_any<T, R1, FWD>(b);
#pragma unroll
      for (int k1 = 0; k1 < R1; ++k1) v[k2 + R2 * k1] = b[k1];
    }
  }
}

// Pass-1 twiddle v[k2] *= W_N^(a k2) (table of exp(-2 pi i q / N)).
template <typename T, int B, bool FWD>
__device__ __forceinline__ void twiddle_rows(cx<T> (&v)[B], int a, const cx<T>* __restrict__ twN) {
#pragma unroll
  for (int k2 = 1; k2 < B; ++k2) {
    cx<T> w = twN[a * k2];
    if (!FWD) w.im = -w.im;
    v[k2] = cmul(v[k2], w);
  }
}

template <int A, int B>
struct Fft2 {
  static constexpr int N = A * B;
  static constexpr int LSL = B * (A + 1) + 1;  // LDS entries per line
  static constexpr int G = (B + A - 1) / A;    // pass-2 columns per thread
};

// Strided complex transform (as k_fft_s) in two passes; LPW consecutive kx
// lines per workgroup, thread = l + LPW * a.
template <typename T, int A, int B, int LPW, bool FWD>
__global__ void __launch_bounds__(LPW * A) k_fft2_s(cx<T>* __restrict__ W, int nxh, long ls, long os,
                                                   const cx<T>* __restrict__ twN) {
  using F = Fft2<A, B>;
  extern __shared__ unsigned char smem[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
  const int ntile = (nxh + LPW - 1) / LPW;
  const int tile = blockIdx.x % ntile, o = blockIdx.x / ntile;
  const int l = threadIdx.x % LPW, a = threadIdx.x / LPW;
  const int kx = tile * LPW + l;
  const bool ok = kx < nxh;
  const long base = (long)(ok ? kx : nxh - 1) + os * o;
  cx<T> v[B];
#pragma unroll
  for (int b = 0; b < B; ++b) v[b] = W[base + ls * (a + A * b)];
  dft_any<T, B, FWD>(v);
  twiddle_rows<T, B, FWD>(v, a, twN);
  cx<T>* lb = buf + l * F::LSL;
#pragma unroll
  for (int k2 = 0; k2 < B; ++k2) lb[k2 * (A + 1) + a] = v[k2];
  __syncthreads();
#pragma unroll
  for (int g = 0; g < F::G; ++g) {
    const int k2 = a + A * g;
    if (F::G * A != B && k2 >= B) break;
    cx<T> u[A];
#pragma unroll
    for (int j = 0; j < A; ++j) u[j] = lb[k2 * (A + 1) + j];
    dft_any<T, A, FWD>(u);
    if (ok) {
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) W[base + ls * (k2 + B * k1)] = u[k1];
    }
  }
}

// Barrier of the threads that share x lines: A threads of one wave where A
// divides 64, so that waves load, transform and store on their own.  With
// that, the real lines read and written past the L2's replacement and the
// spectrum's rows (N + 1 entries, which start anywhere) written in whole cache
// lines, 131072 x lines of 512 take 294 us forward and 253 inverse (330 and
// 284); streaming stores of the spectrum itself were slower (326; strided
// lines 275 against 259).
template <int A>
__device__ __forceinline__ void lines_sync() {
  if constexpr (64 % A == 0) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  } else {
    __syncthreads();
  }
}

// x forward (real lines of 2N -> spectrum kx = 0..N) in two passes; LPW
// lines per workgroup, thread = a + A * l (lanes along the line).
template <typename T, int A, int B, int LPW>
__global__ void __launch_bounds__(LPW * A) k_fft2_x_fwd(const T* __restrict__ in, cx<T>* __restrict__ W,
                                                       long nlines, const cx<T>* __restrict__ twN,
                                                       const cx<T>* __restrict__ rot, T in_scale) {
  using F = Fft2<A, B>;
  constexpr int N = F::N, nxh = N + 1;
  extern __shared__ unsigned char smem[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
  const int a = threadIdx.x % A, l = threadIdx.x / A;
  const long L = (long)blockIdx.x * LPW + l;
  const bool ok = L < nlines;
  const T* src = in + (ok ? L : nlines - 1) * (2L * N);
  cx<T> v[B];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const int n = a + A * b;
    v[b] = cscale(ld_stream(src + 2 * n), in_scale);
  }
  dft_any<T, B, true>(v);
  twiddle_rows<T, B, true>(v, a, twN);
  cx<T>* lb = buf + l * F::LSL;
#pragma unroll
  for (int k2 = 0; k2 < B; ++k2) lb[k2 * (A + 1) + a] = v[k2];
  lines_sync<A>();
  cx<T> z[F::G * A];  // z[g * A + k1] = Z[(a + A g) + B k1]
#pragma unroll
  for (int g = 0; g < F::G; ++g) {
    const int k2 = a + A * g;
    cx<T> u[A];
#pragma unroll
    for (int j = 0; j < A; ++j) u[j] = (k2 < B) ? lb[k2 * (A + 1) + j] : cx<T>{T(0), T(0)};
    dft_any<T, A, true>(u);
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) z[g * A + k1] = u[k1];
  }
  lines_sync<A>();  // pass-2 reads done: the line buffer takes Z in natural order
#pragma unroll
  for (int g = 0; g < F::G; ++g)
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1)
      if (a + A * g < B) lb[(a + A * g) + B * k1] = z[g * A + k1];
  lines_sync<A>();
  if (!ok) return;
  cx<T>* dst = W + L * nxh;
  // (stores of whole cache lines; W is 256-byte aligned)
  const int skew = A % 8 == 0 ? (int)((L * nxh) % A) : 0;
#pragma unroll 4
  for (int k = a - skew; k < nxh; k += A) {
    if (k < 0) continue;
    const cx<T> zk = lb[k % N];
    cx<T> zn = lb[(N - k) % N];
    zn.im = -zn.im;  // conj(Z[N-k])
    const cx<T> e = cscale(cadd(zk, zn), T(0.5));
    const cx<T> d = csub(zk, zn);
    const cx<T> od = {d.im * T(0.5), -d.re * T(0.5)};  // (Z - conj)/(2i)
    dst[k] = cadd(e, cmul(rot[k], od));
  }
}

// x inverse (spectrum kx = 0..N -> real lines of 2N, times `scale`) in two
// passes; LPW lines per workgroup, thread = a + A * l.
template <typename T, int A, int B, int LPW>
__global__ void __launch_bounds__(LPW * A) k_fft2_x_inv(const cx<T>* __restrict__ W, T* __restrict__ out,
                                                       long nlines, const cx<T>* __restrict__ twN,
                                                       const cx<T>* __restrict__ rot, T scale) {
  using F = Fft2<A, B>;
  constexpr int N = F::N, nxh = N + 1;
  extern __shared__ unsigned char smem[];
  cx<T>* buf = reinterpret_cast<cx<T>*>(smem);
  const int a = threadIdx.x % A, l = threadIdx.x / A;
  const long L = (long)blockIdx.x * LPW + l;
  const bool ok = L < nlines;
  const cx<T>* src = W + (ok ? L : nlines - 1) * nxh;
  cx<T>* lb = buf + l * F::LSL;
  for (int k = a; k < N; k += A) {
    const cx<T> xk = src[k];
    cx<T> xn = src[N - k];
    xn.im = -xn.im;  // conj(X[N-k])
    const cx<T> e = cadd(xk, xn);
    cx<T> r = rot[k];
    r.im = -r.im;  // exp(+2 pi i k / nx)
    const cx<T> od = cmul(csub(xk, xn), r);
    lb[k] = {e.re - od.im, e.im + od.re};  // e + i*o
  }
  lines_sync<A>();
  cx<T> v[B];
#pragma unroll
  for (int b = 0; b < B; ++b) v[b] = lb[a + A * b];
  dft_any<T, B, false>(v);
  twiddle_rows<T, B, false>(v, a, twN);
  lines_sync<A>();  // every thread has read its pass-1 input
#pragma unroll
  for (int k2 = 0; k2 < B; ++k2) lb[k2 * (A + 1) + a] = v[k2];
  lines_sync<A>();
  T* dst = out + L * (2L * N);
#pragma unroll
  for (int g = 0; g < F::G; ++g) {
    const int k2 = a + A * g;
    if (F::G * A != B && k2 >= B) break;
    cx<T> u[A];
#pragma unroll
    for (int j = 0; j < A; ++j) u[j] = lb[k2 * (A + 1) + j];
    dft_any<T, A, false>(u);
    if (ok) {
#pragma unroll
      for (int k1 = 0; k1 < A; ++k1) {
        const int n = k2 + B * k1;
        st_stream(dst + 2 * n, cscale(u[k1], scale));
      }
    }
  }
}

// Launchers: the two-pass kernels for the lengths below (all 2,3,5-smooth ones
// from 16 to 512 but 18, 125, 243, 250, 324, 375, 405, 450, 486 and 500, which
// were not timed in two passes), the general Stockham kernels
// otherwise: those pass every element through LDS once per prime factor, and
// at FP64 took 51 us where the two-pass kernel takes 17 (z lines of 160 on
// 97 x 96), 19 against 6.3 (x lines of 64, 4096 of them), 45 against 13 (x
// lines of 192, 15360) and 211 against 58 (z lines of 480, 257 x 64).
// Lines per workgroup 8 or 16 (v = 1, 2), by timing both once per shape
// (chs_tune.h; 24 against 17 us at 160, 54 against 57 at x lines of 512);
// untuned shapes use 16 (8 for N = 512).  v = 3, on request only, is the
// general kernel: it never was the fastest on a length of the list.  The
// numbers stand in saved reports; 0, which was 4 lines per workgroup, takes 8.
#define CHS_FFT2_LENGTHS(X)                                                                                     \
  X(4, 4) X(4, 5) X(4, 6) X(5, 5) X(3, 9) X(5, 6) X(4, 8) X(6, 6) X(5, 8) X(5, 9) X(6, 8) X(5, 10) X(6, 9)        \
  X(6, 10) X(8, 8) X(8, 9) X(5, 15) X(8, 10) X(9, 9) X(9, 10) X(8, 12) X(10, 10) X(9, 12) X(10, 12) X(8, 16)      \
  X(9, 15) X(12, 12) X(10, 15) X(10, 16) X(9, 18) X(12, 15) X(12, 16) X(10, 20) X(12, 18) X(15, 15) X(15, 16)     \
  X(16, 16) X(15, 18) X(16, 18) X(15, 20) X(16, 20) X(18, 20) X(16, 24) X(20, 20) X(18, 24) X(20, 24) X(16, 32)
constexpr int kFft2Variants = 3, kFftVariants = 4;

template <typename T, int A, int B>
static size_t fft2_lds(int lpw) { return sizeof(cx<T>) * (size_t)lpw * Fft2<A, B>::LSL; }

// the launch shape of a key: forced or tuned, else by the length
static int fft2_shape(const std::string& key, int n) {
  const int v = forced_or_tuned(key, kFftVariants);
  return v < 0 ? (n >= 512 ? 1 : 2) : v == 0 ? 1 : v;
}

static std::string fft_key(const char* what, size_t tsize, int n, long nl, long no) {
  return std::string(what) + (tsize == 8 ? "/f64/" : "/f32/") + std::to_string(n) + "/" + std::to_string(nl) + "x" +
         std::to_string(no);
}

template <typename T, int A, int B, int LPW>
static bool fft2_s_launch(cx<T>* W, int nxh, long ls, int no, long os, const cx<T>* tw, T sgn, hipStream_t s) {
  dim3 g((unsigned)(((nxh + LPW - 1) / LPW) * no));
  const size_t sh = fft2_lds<T, A, B>(LPW);
  if (sgn < T(0))
    hipLaunchKernelGGL((k_fft2_s<T, A, B, LPW, true>), g, dim3(LPW * A), sh, s, W, nxh, ls, os, tw);
  else
    hipLaunchKernelGGL((k_fft2_s<T, A, B, LPW, false>), g, dim3(LPW * A), sh, s, W, nxh, ls, os, tw);
  return hipGetLastError() == hipSuccess;
}

template <typename T, int A, int B>
static bool fft2_s_lpw(int v, cx<T>* W, int nxh, long ls, int no, long os, const cx<T>* tw, T sgn, hipStream_t s) {
  switch (v) {
    case 1: return fft2_s_launch<T, A, B, 8>(W, nxh, ls, no, os, tw, sgn, s);
    case 2: return fft2_s_launch<T, A, B, 16>(W, nxh, ls, no, os, tw, sgn, s);
  }
  return false;
}

// Two-pass strided transform of length n with variant v; false when n is not
// a two-pass length.
template <typename T>
static bool fft2_s_variant(int v, cx<T>* W, int nxh, int n, long ls, int no, long os, const cx<T>* tw, T sgn,
                           hipStream_t s) {
#define X(A, B) \
  if (n == A * B) return fft2_s_lpw<T, A, B>(v, W, nxh, ls, no, os, tw, sgn, s);
  CHS_FFT2_LENGTHS(X)
#undef X
  return false;
}

template <typename T, int A, int B, int LPW>
static bool fft2_x_launch(bool fwd, const T* in, cx<T>* W, T* out, long nlines, const cx<T>* tw, const cx<T>* rot,
                          T sc, hipStream_t s) {
  dim3 g((unsigned)((nlines + LPW - 1) / LPW));
  const size_t sh = fft2_lds<T, A, B>(LPW);
  if (fwd)
    hipLaunchKernelGGL((k_fft2_x_fwd<T, A, B, LPW>), g, dim3(LPW * A), sh, s, in, W, nlines, tw, rot, sc);
  else
    hipLaunchKernelGGL((k_fft2_x_inv<T, A, B, LPW>), g, dim3(LPW * A), sh, s, W, out, nlines, tw, rot, sc);
  return hipGetLastError() == hipSuccess;
}

template <typename T, int A, int B>
static bool fft2_x_lpw(int v, bool fwd, const T* in, cx<T>* W, T* out, long nlines, const cx<T>* tw,
                       const cx<T>* rot, T sc, hipStream_t s) {
  switch (v) {
    case 1: return fft2_x_launch<T, A, B, 8>(fwd, in, W, out, nlines, tw, rot, sc, s);
    case 2: return fft2_x_launch<T, A, B, 16>(fwd, in, W, out, nlines, tw, rot, sc, s);
  }
  return false;
}

template <typename T>
static bool fft2_x_variant(int v, bool fwd, const T* in, cx<T>* W, T* out, int nx, long nlines, const cx<T>* tw,
                           const cx<T>* rot, T sc, hipStream_t s) {
#define X(A, B) \
  if (nx / 2 == A * B) return fft2_x_lpw<T, A, B>(v, fwd, in, W, out, nlines, tw, rot, sc, s);
  CHS_FFT2_LENGTHS(X)
#undef X
  return false;
}

// the general Stockham kernels (any 2,3,5-smooth length of one tile)
template <typename T>
static void fft_s_general(cx<T>* W, int nxh, int n, long ls, int no, long os, const Radices& rp, const cx<T>* tw,
                          T sgn, hipStream_t s) {
  const int lpb = kTileC / n;
  dim3 g((unsigned)(((nxh + lpb - 1) / lpb) * no));
  hipLaunchKernelGGL(k_fft_s<T>, g, dim3(kThreads), sizeof(cx<T>) * (size_t)lpb * n, s, W, nxh, n, ls, no, os, rp,
                     tw, sgn);
}

template <typename T>
static void fft_x_general(bool fwd, const T* in, cx<T>* W, T* out, int nx, long nlines, const Radices& rp,
                          const cx<T>* tw, const cx<T>* rot, T sc, hipStream_t s) {
  const int N = nx / 2;
  const int lpb = kTileC / N;
  dim3 g((unsigned)((nlines + lpb - 1) / lpb));
  const size_t sh = sizeof(cx<T>) * (size_t)lpb * N;
  if (fwd)
    hipLaunchKernelGGL(k_fft_x_fwd<T>, g, dim3(kThreads), sh, s, in, W, nx, nlines, rp, tw, rot, sc);
  else
    hipLaunchKernelGGL(k_fft_x_inv<T>, g, dim3(kThreads), sh, s, W, out, nx, nlines, rp, tw, rot, sc);
}

template <typename T>
void launch_fft_s(cx<T>* W, int nxh, int n, long ls, int no, long os, const Radices& rp, const cx<T>* tw,
                         T sgn, hipStream_t s) {
  const int v = fft2_shape(fft_key(sgn < T(0) ? "fft_s+" : "fft_s-", sizeof(T), n, nxh, no), n);
  if (v < kFft2Variants && fft2_s_variant<T>(v, W, nxh, n, ls, no, os, tw, sgn, s)) return;
  fft_s_general<T>(W, nxh, n, ls, no, os, rp, tw, sgn, s);
}

template <typename T>
void launch_fft_x(bool fwd, const T* in, cx<T>* W, T* out, int nx, long nlines, const Radices& rp,
                         const cx<T>* tw, const cx<T>* rot, T sc, hipStream_t s) {
  const int N = nx / 2;
  const int v = fft2_shape(fft_key(fwd ? "fft_x+" : "fft_x-", sizeof(T), N, nlines, 1), N);
  if (v < kFft2Variants && fft2_x_variant<T>(v, fwd, in, W, out, nx, nlines, tw, rot, sc, s)) return;
  fft_x_general<T>(fwd, in, W, out, nx, nlines, rp, tw, rot, sc, s);
}

// Times the two-pass variants of every transform this solver launches (on
// `tmp`, an array as large as the work array, and the work array itself;
// their contents are overwritten by every solve).
template <typename T>
void tune_transforms(int nx, int ny, int nz, int nxh, bool ydir, cx<T>* work, cx<T>* tmp, const cx<T>* twx,
                     const cx<T>* twy, const cx<T>* twz, const cx<T>* rot) {
  hipStream_t s = nullptr;
  const long nlx = (long)ny * nz;
  T* real = reinterpret_cast<T*>(tmp);
  for (int fwd = 1; fwd >= 0; --fwd) {
    tune(fft_key(fwd ? "fft_x+" : "fft_x-", sizeof(T), nx / 2, nlx, 1), kFft2Variants, s, [&](int v) {
      return fft2_x_variant<T>(v, fwd != 0, real, work, real, nx, nlx, twx, rot, T(1), s);
    });
    const T sgn = fwd ? T(-1) : T(1);
    tune(fft_key(fwd ? "fft_s+" : "fft_s-", sizeof(T), nz, nxh, ny), kFft2Variants, s, [&](int v) {
      return fft2_s_variant<T>(v, work, nxh, nz, (long)nxh * ny, ny, (long)nxh, twz, sgn, s);
    });
    if (ydir)
      tune(fft_key(fwd ? "fft_s+" : "fft_s-", sizeof(T), ny, nxh, nz), kFft2Variants, s, [&](int v) {
        return fft2_s_variant<T>(v, work, nxh, ny, (long)nxh, nz, (long)nxh * ny, twy, sgn, s);
      });
  }
}


}  // namespace chs
