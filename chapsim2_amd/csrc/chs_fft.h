// Complex arithmetic and the batched transforms of the pressure solve: real to
// complex along x, complex along y or z, for FP64 and FP32 spectra.
#pragma once

#include <hip/hip_runtime.h>

namespace chs {

template <typename T>
struct cx {
  T re, im;
};
template <typename T>
__device__ inline cx<T> cadd(cx<T> a, cx<T> b) { return {a.re + b.re, a.im + b.im}; }
template <typename T>
__device__ inline cx<T> csub(cx<T> a, cx<T> b) { return {a.re - b.re, a.im - b.im}; }
template <typename T>
__device__ inline cx<T> cmul(cx<T> a, cx<T> b) { return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re}; }
template <typename T>
__device__ inline cx<T> cscale(cx<T> a, T s) { return {a.re * s, a.im * s}; }
// multiply by s*i (s = +-1)
template <typename T>
__device__ inline cx<T> cmuli(cx<T> a, T s) { return {-s * a.im, s * a.re}; }

// A store and a load of two neighbouring values that do not displace what the
// L2 holds.  The real lines are the caller's array, which may start at any
// element: the pair has an element's alignment, which the compiler still
// serves with one 16-byte (FP32: 8-byte) access.
template <typename T>
struct Pair {
  typedef T vec __attribute__((ext_vector_type(2)));
  typedef vec type __attribute__((aligned(sizeof(T))));
  static_assert(alignof(type) == alignof(T), "no more than an element's alignment is assumed");
};
template <typename T>
__device__ __forceinline__ void st_stream(T* p, cx<T> v) {
  const typename Pair<T>::vec x = {v.re, v.im};
  __builtin_nontemporal_store(x, reinterpret_cast<typename Pair<T>::type*>(p));
}

template <typename T>
__device__ __forceinline__ cx<T> ld_stream(const T* p) {
  const typename Pair<T>::vec v = __builtin_nontemporal_load(reinterpret_cast<const typename Pair<T>::type*>(p));
  return {v.x, v.y};
}

constexpr int kTileC = 4096;  // longest line (and complex points per workgroup tile of the general kernels)

struct Radices {
  int n;
  int r[12];
};

// Transform in place of every line of the spectrum W(nxh, ny, nz) along one
// strided dimension (n points at stride ls; kx < nxh and `no` values at stride
// os of the other index), sign sgn < 0 forward.
template <typename T>
void launch_fft_s(cx<T>* W, int nxh, int n, long ls, int no, long os, const Radices& rp, const cx<T>* tw, T sgn,
                  hipStream_t s);
// fwd: real lines `in` (nx values, times sc) -> W (nx/2 + 1 modes); else W -> out, times sc.
template <typename T>
void launch_fft_x(bool fwd, const T* in, cx<T>* W, T* out, int nx, long nlines, const Radices& rp, const cx<T>* tw,
                  const cx<T>* rot, T sc, hipStream_t s);
// Times the variants of every transform of a solver once per shape (on work and
// tmp, whose contents are lost).
template <typename T>
void tune_transforms(int nx, int ny, int nz, int nxh, bool ydir, cx<T>* work, cx<T>* tmp, const cx<T>* twx,
                     const cx<T>* twy, const cx<T>* twz, const cx<T>* rot);

}  // namespace chs
