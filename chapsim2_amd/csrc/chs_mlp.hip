// MLP surrogate of the property table: h -> (T, rho, mu, kappa, cp).
//
// Network 1 -> 64 -> 64 -> 5 with tanh hidden activations.  The weights used
// by the forward and backward passes are BF16 (round-to-nearest-even copies
// of FP32 master weights); every product is accumulated in FP32.  Training
// data are samples of the table interpolation itself
// (ftp_refresh_thermal_properties_from_H, src/input_thermo.f90:345-374, run on
// the GPU over the table handle), so the table stays both the fallback and
// the yardstick of the surrogate.
//
// Kernels: a sampling kernel (uniform h, table interpolation, normalised
// targets); an inference kernel (one thread per sample, weights staged in LDS
// as FP32 values of the BF16 copies, read as wave-wide broadcasts); a training
// kernel for the forward and backward pass (one lane per unit) that writes the
// activations and layer deltas transposed ([unit][sample]); and deterministic
// batch reductions for the weight gradients (tiles of entries, fixed summation
// order) with the Adam update of the FP32 master weights and the BF16 rounding
// in their epilogue.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include "chs_props.h"

namespace chs {
void set_error(const std::string& msg);
}

namespace {

constexpr int H1 = 64, H2 = 64, NO = 5;
constexpr int OW1 = 0, OB1 = OW1 + H1, OW2 = OB1 + H1, OB2 = OW2 + H2 * H1, OW3 = OB2 + H2, OB3 = OW3 + NO * H2;
constexpr int NP = OB3 + NO;  // 4613 parameters
constexpr int kMaxBatch = 65536;
// table columns predicted, in output order
constexpr int kOutCol[NO] = {CHS_PC_T, CHS_PC_D, CHS_PC_M, CHS_PC_K, CHS_PC_CP};

int fail(int code, const std::string& msg) {
  chs::set_error(msg);
  return code;
}

__host__ __device__ inline uint32_t mix32(uint32_t x) {  // integer hash (lowbias32)
  x ^= x >> 16;
  x *= 0x7feb352dU;
  x ^= x >> 15;
  x *= 0x846ca68bU;
  x ^= x >> 16;
  return x;
}

__host__ __device__ inline uint16_t f2bf(float f) {  // round to nearest even
  uint32_t u;
  memcpy(&u, &f, 4);
  u += 0x7FFFU + ((u >> 16) & 1U);
  return (uint16_t)(u >> 16);
}

__host__ __device__ inline float bf2f(uint16_t b) {
  uint32_t u = (uint32_t)b << 16;
  float f;
  memcpy(&f, &u, 4);
  return f;
}

struct Norm {
  float xc, xs;      // x = (h - xc) / xs
  float mu[NO], sd[NO];  // y_o = (v_o - mu_o) / sd_o
};

__device__ inline void bisect(const double* c, int n, double v, int* i1o, int* i2o) {
  int i1 = 0, i2 = n - 1;
  while (i2 - i1 > 1) {
    const int im = i1 + (i2 - i1) / 2;
    const double d1 = c[i1] - v, dm = c[im] - v;
    if (d1 * dm > 1.0e-20) i1 = im;
    else i2 = im;
  }
  *i1o = i1;
  *i2o = i2;
}

// training set: h uniform in [h0, h1], targets by table interpolation in h
__global__ void k_sample(const double* __restrict__ tab, int n, double h0, double h1, int N, uint32_t seed, Norm nm,
                         float* __restrict__ xs, float* __restrict__ ts) {
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= N) return;
  const uint32_t r = mix32(mix32((uint32_t)s * 2654435761U) ^ seed);
  const double u = (double)(r >> 8) * (1.0 / 16777216.0);
  const double h = h0 + (h1 - h0) * u;
  const double* ch = tab + (long)CHS_PC_H * n;
  int i1, i2;
  bisect(ch, n, h, &i1, &i2);
  const double w1 = (ch[i2] - h) / (ch[i2] - ch[i1]), w2 = 1.0 - w1;
  xs[s] = (float)((h - nm.xc) / nm.xs);
  for (int o = 0; o < NO; ++o) {
    const double* c = tab + (long)kOutCol[o] * n;
    const double v = w1 * c[i1] + w2 * c[i2];
    ts[(long)o * N + s] = (float)((v - nm.mu[o]) / nm.sd[o]);
  }
}

__device__ inline void stage_params(const uint16_t* __restrict__ p16, float* sp) {
  for (int i = threadIdx.x; i < NP; i += blockDim.x) sp[i] = bf2f(p16[i]);
  __syncthreads();
}

// double-precision inputs h -> denormalised double outputs (API path)
__global__ void __launch_bounds__(256) k_eval(const uint16_t* __restrict__ p16, Norm nm, const double* __restrict__ h,
                                              long N, double* __restrict__ o0, double* __restrict__ o1,
                                              double* __restrict__ o2, double* __restrict__ o3,
                                              double* __restrict__ o4) {
  __shared__ float sp[NP];
  stage_params(p16, sp);
  const long b = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= N) return;
  const float xv = (float)((h[b] - nm.xc) / nm.xs);
  float a1[H1];
#pragma unroll
  for (int i = 0; i < H1; ++i) a1[i] = tanhf(sp[OW1 + i] * xv + sp[OB1 + i]);
  float out[NO];
#pragma unroll
  for (int o = 0; o < NO; ++o) out[o] = sp[OB3 + o];
  for (int j = 0; j < H2; ++j) {
    float z = sp[OB2 + j];
#pragma unroll
    for (int i = 0; i < H1; ++i) z += sp[OW2 + j * H1 + i] * a1[i];
    const float a2 = tanhf(z);
#pragma unroll
    for (int o = 0; o < NO; ++o) out[o] += sp[OW3 + o * H2 + j] * a2;
  }
  double* dst[NO] = {o0, o1, o2, o3, o4};
#pragma unroll
  for (int o = 0; o < NO; ++o)
    if (dst[o]) dst[o][b] = (double)out[o] * nm.sd[o] + nm.mu[o];
}

// Forward and backward pass of the mean squared error over B samples x 5
// outputs.  Samples are either given (given != 0: sample b of xs / ts) or
// drawn at random from the training set of N samples.  Writes the layer
// quantities transposed ([unit][sample], rows of Bp) for k_grad and one loss
// partial per workgroup.
//
// One lane per unit of a layer, kTS samples per wave: lane j keeps row j of W2
// for the forward pass and column j for the backward pass in registers (128
// of them, FP32 values of the BF16 copies), and the other layer's values
// arrive as wave-wide LDS broadcasts of four, each used for one
// multiply-add.  Every sum runs in one lane over ascending units, as one
// thread per sample would.  Bound by latency: ~20 k multiply-adds per sample
// are 4 us of chip time at 65536 samples, but a batch of 4096 is one wave per
// SIMD.  One thread per sample used 64 waves in all for that batch, each with
// 16 k multiply-adds and their LDS reads in a row: 81 us, now 12.5.
constexpr int kTS = 4, kTW = 4, kTSB = kTS * kTW;  // samples per wave, waves, samples per workgroup
constexpr int kTrainBlocks = 1024;                 // grid limit; workgroups walk over the rest
static_assert(H1 == 64 && H2 == 64 && kTS * NO <= 64, "one lane per unit");

__device__ __forceinline__ float dot64(const float w[64], const float* __restrict__ v, float z) {
#pragma unroll
  for (int i = 0; i < 64; i += 4) {
    const float4 x = *reinterpret_cast<const float4*>(v + i);
    z += w[i] * x.x;
    z += w[i + 1] * x.y;
    z += w[i + 2] * x.z;
    z += w[i + 3] * x.w;
  }
  return z;
}

__global__ void __launch_bounds__(64 * kTW) k_bwd(const uint16_t* __restrict__ p16, const float* __restrict__ xs,
                                                  const float* __restrict__ ts, int N, int B, int Bp, uint32_t seed,
                                                  int given, float* __restrict__ xb, float* __restrict__ a1T,
                                                  float* __restrict__ a2T, float* __restrict__ dz1T,
                                                  float* __restrict__ dz2T, float* __restrict__ dyT,
                                                  float* __restrict__ lossp) {
  constexpr int kP = kTSB + 1;
  __shared__ __align__(16) float ex[kTW][kTS][64];  // a layer's values on their way to the other units
  __shared__ __align__(16) float w3s[NO][68];
  __shared__ float dys[kTW][kTS][NO + 1];
  __shared__ float tr[4][64][kP];
  __shared__ float red[kTW];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  float wr[64], wc[64], w3[NO];
#pragma unroll
  for (int i = 0; i < 64; i += 8) {
    const uint16_t* q = p16 + OW2 + lane * H1 + i;  // rows of 128 bytes
    const uint4 v = *reinterpret_cast<const uint4*>(q);
    const uint32_t u[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      wr[i + 2 * k] = __builtin_bit_cast(float, u[k] << 16);
      wr[i + 2 * k + 1] = __builtin_bit_cast(float, u[k] & 0xFFFF0000U);
    }
  }
#pragma unroll
  for (int j = 0; j < 64; ++j) wc[j] = bf2f(p16[OW2 + j * H1 + lane]);
#pragma unroll
  for (int o = 0; o < NO; ++o) w3[o] = bf2f(p16[OW3 + o * H2 + lane]);
  const float w1 = bf2f(p16[OW1 + lane]), c1 = bf2f(p16[OB1 + lane]), c2 = bf2f(p16[OB2 + lane]);
  const int os = lane / NO, oo = lane % NO;  // sample and output of this lane (lanes below kTS * NO)
  const bool head = lane < kTS * NO;
  const float c3 = bf2f(p16[OB3 + oo]);
  if (w == 0)
#pragma unroll
    for (int o = 0; o < NO; ++o) w3s[o][lane] = w3[o];
  const float sc = 2.0f / (float)(B * NO);
  float lsum = 0.0f;
  for (int b0 = blockIdx.x * kTSB; b0 < B; b0 += gridDim.x * kTSB) {
    const int bw = b0 + w * kTS;  // this wave's first sample
    auto source = [&](int b) {
      return given ? b : (int)(mix32(mix32((uint32_t)b * 2246822519U) ^ seed) % (uint32_t)N);
    };
    float a1[kTS], a2[kTS], d2[kTS];
#pragma unroll
    for (int k = 0; k < kTS; ++k) {
      const float xv = bw + k < B ? xs[source(bw + k)] : 0.0f;
      a1[k] = tanhf(w1 * xv + c1);
      ex[w][k][lane] = a1[k];
      if (!given && lane == 0 && bw + k < B) xb[bw + k] = xv;
    }
    float tv = 0.0f;
    if (head && bw + os < B) tv = ts[(long)oo * (given ? B : N) + source(bw + os)];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTS; ++k) a2[k] = tanhf(dot64(wr, ex[w][k], c2));
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTS; ++k) ex[w][k][lane] = a2[k];
    __syncthreads();
    if (head) {
      float out = c3;
#pragma unroll 4
      for (int j = 0; j < 64; j += 4) {
        const float4 x = *reinterpret_cast<const float4*>(&ex[w][os][j]);
        const float4 y = *reinterpret_cast<const float4*>(&w3s[oo][j]);
        out += y.x * x.x;
        out += y.y * x.y;
        out += y.z * x.z;
        out += y.w * x.w;
      }
      const float e = bw + os < B ? out - tv : 0.0f;
      lsum += e * e;
      dys[w][os][oo] = sc * e;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTS; ++k) {
      float da2 = 0.0f;
#pragma unroll
      for (int o = 0; o < NO; ++o) da2 += w3[o] * dys[w][k][o];
      d2[k] = da2 * (1.0f - a2[k] * a2[k]);
      ex[w][k][lane] = d2[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kTS; ++k) {
      const float da1 = dot64(wc, ex[w][k], 0.0f);
      const int c = w * kTS + k;
      tr[0][lane][c] = a1[k];
      tr[1][lane][c] = a2[k];
      tr[2][lane][c] = da1 * (1.0f - a1[k] * a1[k]);
      tr[3][lane][c] = d2[k];
    }
    __syncthreads();
    // (rows of Bp, a multiple of kTSB: whole 64-byte segments)
    float* const dst[4] = {a1T, a2T, dz1T, dz2T};
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = threadIdx.x; i < 64 * kTSB; i += 64 * kTW)
        dst[q][(long)(i / kTSB) * Bp + b0 + i % kTSB] = tr[q][i / kTSB][i % kTSB];
    if (threadIdx.x < NO * kTSB) {
      const int o = threadIdx.x / kTSB, c = threadIdx.x % kTSB;
      dyT[(long)o * Bp + b0 + c] = dys[c / kTS][c % kTS][o];
    }
    __syncthreads();
  }
  for (int k = 32; k > 0; k >>= 1) lsum += __shfl_xor(lsum, k);
  if (lane == 0) red[w] = lsum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (int i = 0; i < kTW; ++i) t += red[i];
    lossp[blockIdx.x] = t;
  }
}

// Adam's update of FP32 master weight i and its BF16 copy
struct Adam {
  float *p, *m, *v;
  uint16_t* p16;
  float lr, b1, b2, eps, c1, c2;
};

__device__ __forceinline__ void adam_update(const Adam& a, int i, float gi) {
  const float mi = a.b1 * a.m[i] + (1.0f - a.b1) * gi;
  const float vi = a.b2 * a.v[i] + (1.0f - a.b2) * gi * gi;
  a.m[i] = mi;
  a.v[i] = vi;
  const float pi = a.p[i] - a.lr * (mi / a.c1) / (sqrtf(vi / a.c2) + a.eps);
  a.p[i] = pi;
  a.p16[i] = f2bf(pi);
}

// All gradients of a batch, G[r][c] = sum_b U[r][b] * V[c][b], and with
// STEP the Adam update of their weights.  A workgroup of 256 threads owns a
// tile of NR x NC entries (and, with ONES, the NR row sums besides): thread t
// sums b = t, t + 256, ... of every entry of the tile, so a row is read once
// per tile instead of once per entry, and a fixed tree adds the 256 partial
// sums of each.  Tiles of 16: 256 of them fill the chip for the 64 x 64
// layer, and read 8 rows for 16 entries.  With one workgroup per entry and a
// kernel for each of six arrays and for the update a batch of 4096 took 44 us
// in seven launches, now 9.2 in one.
constexpr int kGradThreads = 256;

template <int NR, int NC, bool ONES, bool STEP>
__device__ __forceinline__ void grad_tile(float* red, float* sum, const float* __restrict__ U,
                                          const float* __restrict__ V, int B, int Bp, int iw, int ldw, int ib,
                                          float* __restrict__ G, const Adam& ad) {
  constexpr int E = NR * NC + (ONES ? NR : 0), ND = NC ? NC : 1;
  float acc[E];
#pragma unroll
  for (int e = 0; e < E; ++e) acc[e] = 0.0f;
#pragma unroll 4
  for (int b = threadIdx.x; b < B; b += kGradThreads) {
    float u[NR], v[ND];
#pragma unroll
    for (int r = 0; r < NR; ++r) u[r] = U[(long)r * Bp + b];
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = V[(long)c * Bp + b];
#pragma unroll
    for (int r = 0; r < NR; ++r) {
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[r * NC + c] += u[r] * v[c];
      if (ONES) acc[NR * NC + r] += u[r];
    }
  }
#pragma unroll
  for (int e = 0; e < E; ++e) red[e * kGradThreads + threadIdx.x] = acc[e];
  __syncthreads();
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int e0 = 0; e0 < E; e0 += 4) {
    const int e = e0 + w;
    if (e < E) {
      const float* q = red + e * kGradThreads + lane;
      float t = (q[0] + q[128]) + (q[64] + q[192]);
#pragma unroll
      for (int k = 32; k > 0; k >>= 1) t += __shfl_down(t, k);
      if (lane == 0) sum[e] = t;
    }
  }
  __syncthreads();
  const int e = threadIdx.x;
  if (e < E) {
    const int i = e < NR * NC ? iw + (e / ND) * ldw + e % ND : ib + e - NR * NC;
    if (STEP) adam_update(ad, i, sum[e]);
    else G[i] = sum[e];
  }
}

// blocks: 256 tiles 4 x 4 of W2, 8 of eight rows of W1 with b1, 4 of sixteen
// entries of b2, 16 of W3 (5 x 4) of which the first has b3
constexpr int kGradW2 = (H2 / 4) * (H1 / 4), kGradW1 = H1 / 8, kGradB2 = H2 / 16, kGradW3 = H2 / 4;
constexpr int kGradBlocks = kGradW2 + kGradW1 + kGradB2 + kGradW3;

template <bool STEP>
__global__ void __launch_bounds__(kGradThreads) k_grad(const float* __restrict__ xb, const float* __restrict__ a1T,
                                                       const float* __restrict__ a2T, const float* __restrict__ dz1T,
                                                       const float* __restrict__ dz2T, const float* __restrict__ dyT,
                                                       int B, int Bp, float* __restrict__ G, Adam ad) {
  __shared__ float red[25 * kGradThreads];
  __shared__ float sum[25];
  int k = blockIdx.x;
  if (k < kGradW2) {
    const int r = 4 * (k / (H1 / 4)), c = 4 * (k % (H1 / 4));
    grad_tile<4, 4, false, STEP>(red, sum, dz2T + (long)r * Bp, a1T + (long)c * Bp, B, Bp, OW2 + r * H1 + c, H1, 0, G,
                                 ad);
  } else if ((k -= kGradW2) < kGradW1) {
    grad_tile<8, 1, true, STEP>(red, sum, dz1T + (long)(8 * k) * Bp, xb, B, Bp, OW1 + 8 * k, 1, OB1 + 8 * k, G, ad);
  } else if ((k -= kGradW1) < kGradB2) {
    grad_tile<16, 0, true, STEP>(red, sum, dz2T + (long)(16 * k) * Bp, nullptr, B, Bp, 0, 1, OB2 + 16 * k, G, ad);
  } else if ((k -= kGradB2) == 0) {
    grad_tile<NO, 4, true, STEP>(red, sum, dyT, a2T, B, Bp, OW3, H2, OB3, G, ad);
  } else {
    grad_tile<NO, 4, false, STEP>(red, sum, dyT, a2T + (long)(4 * k) * Bp, B, Bp, OW3 + 4 * k, H2, 0, G, ad);
  }
}

__global__ void k_round(const float* __restrict__ p, uint16_t* __restrict__ q, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) q[i] = f2bf(p[i]);
}

}  // namespace

struct chs_mlp {
  chs_props* tab = nullptr;
  hipStream_t stream = nullptr;
  Norm nm{};
  float *p32 = nullptr, *g32 = nullptr, *m32 = nullptr, *v32 = nullptr;
  uint16_t* p16 = nullptr;
  float *xs = nullptr, *ts = nullptr;
  int nsamp = 0;
  float *xb = nullptr, *a1T = nullptr, *a2T = nullptr, *dz1T = nullptr, *dz2T = nullptr, *dyT = nullptr;
  float *lossp = nullptr, *tin = nullptr;
  int step = 0;
  uint32_t seed = 1;
  bool matrix_cores = true;  // property refresh on the matrix cores (k_mlp_from_dh_mfma)
  void* io = nullptr;
  size_t io_bytes = 0;
  std::vector<void*> owned;
  ~chs_mlp() {
    if (stream) (void)hipStreamSynchronize(stream);
    for (void* q : owned) (void)hipFree(q);
    if (io) (void)hipFree(io);
    if (stream) (void)hipStreamDestroy(stream);
  }
};

namespace {

template <typename T>
bool dalloc(chs_mlp* m, T** p, size_t n) {
  if (hipMalloc(p, sizeof(T) * (n ? n : 1)) != hipSuccess) return false;
  m->owned.push_back(*p);
  return true;
}

// forward and backward pass over a batch, then the gradients into m->g32 or,
// with ad, straight into the weights; loss sum on request
int batch_pass(chs_mlp* m, const float* xs, const float* ts, int N, int B, uint32_t seed, int given, const Adam* ad,
               float* loss) {
  hipStream_t s = m->stream;
  const int Bp = (B + kTSB - 1) / kTSB * kTSB;
  const int nblk = Bp / kTSB < kTrainBlocks ? Bp / kTSB : kTrainBlocks;
  hipLaunchKernelGGL(k_bwd, dim3(nblk), dim3(64 * kTW), 0, s, m->p16, xs, ts, N, B, Bp, seed, given, m->xb, m->a1T,
                     m->a2T, m->dz1T, m->dz2T, m->dyT, m->lossp);
  if (ad)
    hipLaunchKernelGGL(k_grad<true>, dim3(kGradBlocks), dim3(kGradThreads), 0, s, m->xb, m->a1T, m->a2T, m->dz1T,
                       m->dz2T, m->dyT, B, Bp, m->g32, *ad);
  else
    hipLaunchKernelGGL(k_grad<false>, dim3(kGradBlocks), dim3(kGradThreads), 0, s, m->xb, m->a1T, m->a2T, m->dz1T,
                       m->dz2T, m->dyT, B, Bp, m->g32, Adam{});
  if (loss) {
    float h[kTrainBlocks];
    if (hipMemcpyAsync(h, m->lossp, sizeof(float) * nblk, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return fail(CHS_EHIP, "loss copy");
    double t = 0.0;
    for (int i = 0; i < nblk; ++i) t += h[i];
    *loss = (float)(t / ((double)B * NO));
  }
  if (hipGetLastError() != hipSuccess) return fail(CHS_EHIP, "gradient kernels");
  return CHS_OK;
}

}  // namespace

namespace {

// ---- matrix-core form of the network (inference) ----
// v_mfma_f32_16x16x16_bf16: D(16x16) = A(16x16) B(16x16) + C, one wave; lane
// l holds A[l%16][4(l/16)+0..3], B[4(l/16)+0..3][l%16] and
// D[4(l/16)+0..3][l%16].  The 64x64 layer is 4 (output blocks) x 4 (input
// blocks) of these per 16 cells: A = a block of W2 (rows: output units,
// columns: input units), B = the BF16 first-layer activations (rows: input
// units, columns: cells), D = the second-layer pre-activations.
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// tanh x = 1 - 2 / (1 + 2^{2 log2(e) x}) with the hardware base-2
// exponential and reciprocal (v_exp_f32, v_rcp_f32, each ~1 ulp: absolute
// error ~3e-7, below the BF16 rounding of the activations).  Five
// instructions; a written divide (also __fdividef) compiles to the
// correctly rounded IEEE sequence of fifteen.  Saturates to +-1 for large
// |x| (exp2 overflow gives a zero reciprocal).
__device__ __forceinline__ float tanh_fast(float x) {
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(2.8853900817779268f * x));
}

// BF16 of a finite float, rounded to nearest even by the hardware
// conversion (v_cvt_pk_bf16_f32; the same bits as f2bf for finite values)
__device__ __forceinline__ short bf16_rne(float x) { return __builtin_bit_cast(short, (__bf16)x); }

// out[0..4] (normalised) of the 16 cells whose normalised inputs the lanes
// with l%16 = c hold in xv; every lane ends with the outputs of cell l%16.
// wa: this lane's 16 A operands (W2 blocks), sp: the FP32 parameters in LDS.
// Outputs O0 to O1 - 1 only.
template <int O0, int O1>
__device__ __forceinline__ void mlp16_mfma(const bf16x4 wa[16], const float* __restrict__ sp, float xv, float out[NO]) {
  const int q = (threadIdx.x & 63) >> 4;
  bf16x4 bv[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int u = 16 * kk + 4 * q + r;
      bv[kk][r] = bf16_rne(tanh_fast(sp[OW1 + u] * xv + sp[OB1 + u]));
    }
  }
#pragma unroll
  for (int o = O0; o < O1; ++o) out[o] = 0.0f;
#pragma unroll
  for (int mt = 0; mt < 4; ++mt) {
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wa[4 * mt + kk], bv[kk], acc, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int u = 16 * mt + 4 * q + r;
      const float a2 = tanh_fast(acc[r] + sp[OB2 + u]);
#pragma unroll
      for (int o = O0; o < O1; ++o) out[o] += sp[OW3 + o * H2 + u] * a2;
    }
  }
#pragma unroll
  for (int o = O0; o < O1; ++o) {
    out[o] += __shfl_xor(out[o], 16);
    out[o] += __shfl_xor(out[o], 32);
    out[o] += sp[OB3 + o];
  }
}

// k_mlp_from_dh on the matrix cores: 64 cells per wave (one per lane for the
// clamp and the bisection), the network evaluated for them in four passes of
// 16 cells, twice (h from the table, then h = rho*h / rho).
__global__ void __launch_bounds__(256) k_mlp_from_dh_mfma(const uint16_t* __restrict__ p16, Norm nm,
                                                          const double* __restrict__ tab, int nt, double dhmin,
                                                          double dhmax, const double* __restrict__ rhoh, long N,
                                                          double* __restrict__ oh, double* __restrict__ od,
                                                          double* __restrict__ om, double* __restrict__ ok,
                                                          double* __restrict__ ot, int* __restrict__ flag,
                                                          float* __restrict__ fh, float* __restrict__ fm,
                                                          float* __restrict__ fk, float* __restrict__ ft) {
  __shared__ float sp[NP];
  stage_params(p16, sp);
  const int lane = threadIdx.x & 63;
  const int ci = lane & 15, q = lane >> 4;
  bf16x4 wa[16];
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      wa[4 * mt + kk] = *reinterpret_cast<const bf16x4*>(p16 + OW2 + (16 * mt + ci) * H1 + 16 * kk + 4 * q);
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = c < N;
  double v = live ? rhoh[c] : dhmin;
  if (live && v < dhmin) {
    v = dhmin;
    atomicAdd(flag, 1);
  } else if (live && v > dhmax) {
    v = dhmax;
    atomicAdd(flag, 1);
  }
  const double* crh = tab + (long)CHS_PC_RH * nt;
  const double* ch = tab + (long)CHS_PC_H * nt;
  int i1, i2;
  bisect(crh, nt, v, &i1, &i2);
  const double w1 = (crh[i2] - v) / (crh[i2] - crh[i1]), w2 = 1.0 - w1;
  double h = w1 * ch[i1] + w2 * ch[i2];
  float mine[NO];
  // (the first pass needs the density alone: a fifth of the output layer, 180 -> 174 us for 1.3 M cells)
  float x = (float)((h - nm.xc) / nm.xs);
#pragma unroll 1
  for (int p = 0; p < 4; ++p) {
    float out[NO];
    mlp16_mfma<1, 2>(wa, sp, __shfl(x, 16 * p + ci), out);
    if (q == p) mine[1] = out[1];
  }
  h = v / ((double)mine[1] * nm.sd[1] + nm.mu[1]);
  x = (float)((h - nm.xc) / nm.xs);
#pragma unroll 1
  for (int p = 0; p < 4; ++p) {
    float out[NO];
    mlp16_mfma<0, NO>(wa, sp, __shfl(x, 16 * p + ci), out);
    if (q == p)
#pragma unroll
      for (int o = 0; o < NO; ++o) mine[o] = out[o];
  }
  if (!live) return;
  const double vt = (double)mine[0] * nm.sd[0] + nm.mu[0], vm = (double)mine[2] * nm.sd[2] + nm.mu[2],
               vk = (double)mine[3] * nm.sd[3] + nm.mu[3];
  if (oh) oh[c] = h;
  if (ot) ot[c] = vt;
  if (od) od[c] = (double)mine[1] * nm.sd[1] + nm.mu[1];
  if (om) om[c] = vm;
  if (ok) ok[c] = vk;
  if (fh) fh[c] = (float)h;
  if (fm) fm[c] = (float)vm;
  if (fk) fk[c] = (float)vk;
  if (ft) ft[c] = (float)vt;
}

// Properties from rho*h with the surrogate (flow solver's refresh, mode
// CHS_PROPS_MLP): clamp to [dhmin, dhmax] (counted), bisection on the
// table's rho*h column and linear interpolation for the first h (as
// ftp_refresh_thermal_properties_from_DH, src/input_thermo.f90:393-446),
// then the network for the properties from h, h = rho*h / rho, and the
// network again; fh, fm, fk, ft (each possibly null) receive h, mu, kappa
// and T rounded to FP32.  One thread per cell; parameters in LDS as in k_eval.
__global__ void __launch_bounds__(256) k_mlp_from_dh(const uint16_t* __restrict__ p16, Norm nm,
                                                     const double* __restrict__ tab, int nt, double dhmin,
                                                     double dhmax, const double* __restrict__ rhoh, long N,
                                                     double* __restrict__ oh, double* __restrict__ od,
                                                     double* __restrict__ om, double* __restrict__ ok,
                                                     double* __restrict__ ot, int* __restrict__ flag,
                                                     float* __restrict__ fh, float* __restrict__ fm,
                                                     float* __restrict__ fk, float* __restrict__ ft) {
  __shared__ float sp[NP];
  stage_params(p16, sp);
  const long c = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  double v = rhoh[c];
  if (v < dhmin) {
    v = dhmin;
    atomicAdd(flag, 1);
  } else if (v > dhmax) {
    v = dhmax;
    atomicAdd(flag, 1);
  }
  const double* crh = tab + (long)CHS_PC_RH * nt;
  const double* ch = tab + (long)CHS_PC_H * nt;
  int i1, i2;
  bisect(crh, nt, v, &i1, &i2);
  const double w1 = (crh[i2] - v) / (crh[i2] - crh[i1]), w2 = 1.0 - w1;
  double h = w1 * ch[i1] + w2 * ch[i2];
  float out[NO];
  for (int pass = 0; pass < 2; ++pass) {
    const float xv = (float)((h - nm.xc) / nm.xs);
    float a1[H1];
#pragma unroll
    for (int i = 0; i < H1; ++i) a1[i] = tanhf(sp[OW1 + i] * xv + sp[OB1 + i]);
#pragma unroll
    for (int o = 0; o < NO; ++o) out[o] = sp[OB3 + o];
    for (int j = 0; j < H2; ++j) {
      float z = sp[OB2 + j];
#pragma unroll
      for (int i = 0; i < H1; ++i) z += sp[OW2 + j * H1 + i] * a1[i];
      const float a2 = tanhf(z);
#pragma unroll
      for (int o = 0; o < NO; ++o) out[o] += sp[OW3 + o * H2 + j] * a2;
    }
    if (pass == 0) h = v / ((double)out[1] * nm.sd[1] + nm.mu[1]);
  }
  const double vt = (double)out[0] * nm.sd[0] + nm.mu[0], vm = (double)out[2] * nm.sd[2] + nm.mu[2],
               vk = (double)out[3] * nm.sd[3] + nm.mu[3];
  if (oh) oh[c] = h;
  if (ot) ot[c] = vt;
  if (od) od[c] = (double)out[1] * nm.sd[1] + nm.mu[1];
  if (om) om[c] = vm;
  if (ok) ok[c] = vk;
  if (fh) fh[c] = (float)h;
  if (fm) fm[c] = (float)vm;
  if (fk) fk[c] = (float)vk;
  if (ft) ft[c] = (float)vt;
}

}  // namespace

namespace chs {
std::string mlp_refresh_dh(chs_mlp* m, const chs_props* p, const double* rhoh, long n, double* h, double* d,
                           double* mu, double* k, double* t, int* flag, hipStream_t s, float* const* r32) {
  if (n <= 0) return "";
  float* const f[4] = {r32 ? r32[0] : nullptr, r32 ? r32[1] : nullptr, r32 ? r32[2] : nullptr,
                       r32 ? r32[3] : nullptr};
  if (m->matrix_cores)
    hipLaunchKernelGGL(k_mlp_from_dh_mfma, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, m->p16, m->nm, p->dev,
                       p->n, p->dhmin, p->dhmax, rhoh, n, h, d, mu, k, t, flag, f[0], f[1], f[2], f[3]);
  else
    hipLaunchKernelGGL(k_mlp_from_dh, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, m->p16, m->nm, p->dev,
                       p->n, p->dhmin, p->dhmax, rhoh, n, h, d, mu, k, t, flag, f[0], f[1], f[2], f[3]);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return std::string("surrogate kernel: ") + hipGetErrorString(e);
  return "";
}
}  // namespace chs

extern "C" {

int chs_mlp_create(chs_props_t* table, int nsamples, unsigned seed, chs_mlp_t** out) {
  if (!table || !out || nsamples < 1) return fail(CHS_EINVAL, "invalid argument");
  *out = nullptr;
  chs_mlp* m = new chs_mlp();
  m->tab = table;
  m->seed = seed ? seed : 1U;
  m->nsamp = nsamples;
  const std::vector<double>& hc = table->col[CHS_PC_H];
  double h0 = hc[0], h1 = hc[0];
  for (double v : hc) { h0 = std::min(h0, v); h1 = std::max(h1, v); }
  m->nm.xc = (float)(0.5 * (h0 + h1));
  m->nm.xs = (float)(0.5 * (h1 - h0));
  for (int o = 0; o < NO; ++o) {
    const std::vector<double>& c = table->col[kOutCol[o]];
    double mu = 0.0, sd = 0.0;
    for (double v : c) mu += v;
    mu /= (double)c.size();
    for (double v : c) sd += (v - mu) * (v - mu);
    sd = std::sqrt(sd / (double)c.size());
    m->nm.mu[o] = (float)mu;
    m->nm.sd[o] = (float)(sd > 0.0 ? sd : 1.0);
  }
  // Glorot-uniform initial weights from the seed, zero biases
  std::vector<float> p(NP, 0.0f);
  uint32_t st = mix32(m->seed ^ 0x5bd1e995U);
  auto uni = [&](float lim) {
    st = mix32(st + 0x9e3779b9U);
    return lim * (2.0f * (float)(st >> 8) * (1.0f / 16777216.0f) - 1.0f);
  };
  for (int i = 0; i < H1; ++i) p[OW1 + i] = uni(std::sqrt(6.0f / (1 + H1)));
  for (int i = 0; i < H2 * H1; ++i) p[OW2 + i] = uni(std::sqrt(6.0f / (H1 + H2)));
  for (int i = 0; i < NO * H2; ++i) p[OW3 + i] = uni(std::sqrt(6.0f / (H2 + NO)));
  bool ok = hipStreamCreate(&m->stream) == hipSuccess && dalloc(m, &m->p32, NP) && dalloc(m, &m->g32, NP) &&
            dalloc(m, &m->m32, NP) && dalloc(m, &m->v32, NP) && dalloc(m, &m->p16, NP) &&
            dalloc(m, &m->xs, nsamples) && dalloc(m, &m->ts, (size_t)NO * nsamples) && dalloc(m, &m->xb, kMaxBatch) &&
            dalloc(m, &m->a1T, (size_t)H1 * kMaxBatch) && dalloc(m, &m->a2T, (size_t)H2 * kMaxBatch) &&
            dalloc(m, &m->dz1T, (size_t)H1 * kMaxBatch) && dalloc(m, &m->dz2T, (size_t)H2 * kMaxBatch) &&
            dalloc(m, &m->dyT, (size_t)NO * kMaxBatch) && dalloc(m, &m->lossp, kTrainBlocks) &&
            dalloc(m, &m->tin, (size_t)NO * kMaxBatch);
  if (!ok) {
    delete m;
    return fail(CHS_ENOMEM, "device allocation failed");
  }
  hipStream_t s = m->stream;
  ok = hipMemcpyAsync(m->p32, p.data(), sizeof(float) * NP, hipMemcpyHostToDevice, s) == hipSuccess &&
       hipMemsetAsync(m->m32, 0, sizeof(float) * NP, s) == hipSuccess &&
       hipMemsetAsync(m->v32, 0, sizeof(float) * NP, s) == hipSuccess;
  hipLaunchKernelGGL(k_round, dim3((NP + 255) / 256), dim3(256), 0, s, m->p32, m->p16, NP);
  hipLaunchKernelGGL(k_sample, dim3((nsamples + 255) / 256), dim3(256), 0, s, table->dev, table->n, h0, h1, nsamples,
                     m->seed, m->nm, m->xs, m->ts);
  if (!ok || hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) {
    delete m;
    return fail(CHS_EHIP, "initialisation kernels");
  }
  *out = m;
  return CHS_OK;
}

int chs_mlp_destroy(chs_mlp_t* m) {
  delete m;
  return CHS_OK;
}

int chs_mlp_info(const chs_mlp_t* m, int* nparams, float norm[12]) {
  if (!m) return fail(CHS_EINVAL, "null handle");
  if (nparams) *nparams = NP;
  if (norm) {
    norm[0] = m->nm.xc;
    norm[1] = m->nm.xs;
    for (int o = 0; o < NO; ++o) {
      norm[2 + o] = m->nm.mu[o];
      norm[7 + o] = m->nm.sd[o];
    }
  }
  return CHS_OK;
}

int chs_mlp_get_params(chs_mlp_t* m, float* p32, unsigned short* p16) {
  if (!m) return fail(CHS_EINVAL, "null handle");
  if (p32 && hipMemcpyAsync(p32, m->p32, sizeof(float) * NP, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
    return fail(CHS_EHIP, "copy");
  if (p16 && hipMemcpyAsync(p16, m->p16, sizeof(uint16_t) * NP, hipMemcpyDeviceToHost, m->stream) != hipSuccess)
    return fail(CHS_EHIP, "copy");
  if (hipStreamSynchronize(m->stream) != hipSuccess) return fail(CHS_EHIP, "synchronise");
  return CHS_OK;
}

int chs_mlp_set_params(chs_mlp_t* m, const float* p32) {
  if (!m || !p32) return fail(CHS_EINVAL, "invalid argument");
  if (hipMemcpyAsync(m->p32, p32, sizeof(float) * NP, hipMemcpyHostToDevice, m->stream) != hipSuccess)
    return fail(CHS_EHIP, "copy");
  hipLaunchKernelGGL(k_round, dim3((NP + 255) / 256), dim3(256), 0, m->stream, m->p32, m->p16, NP);
  if (hipStreamSynchronize(m->stream) != hipSuccess) return fail(CHS_EHIP, "synchronise");
  return CHS_OK;
}

int chs_mlp_grad(chs_mlp_t* m, const float* x, const float* t, int B, float* grad, float* loss) {
  if (!m || !x || !t || !grad || B < 1 || B > kMaxBatch) return fail(CHS_EINVAL, "invalid argument");
  hipStream_t s = m->stream;
  // stage the given samples: inputs in xb, targets as [o][b]
  std::vector<float> tt((size_t)NO * B);
  for (int b = 0; b < B; ++b)
    for (int o = 0; o < NO; ++o) tt[(size_t)o * B + b] = t[(size_t)b * NO + o];
  if (hipMemcpyAsync(m->tin, tt.data(), sizeof(float) * tt.size(), hipMemcpyHostToDevice, s) != hipSuccess ||
      hipMemcpyAsync(m->xb, x, sizeof(float) * B, hipMemcpyHostToDevice, s) != hipSuccess)
    return fail(CHS_EHIP, "copy in");
  int rc = batch_pass(m, m->xb, m->tin, B, B, 0U, 1, nullptr, loss);
  if (rc != CHS_OK) return rc;
  if (hipMemcpyAsync(grad, m->g32, sizeof(float) * NP, hipMemcpyDeviceToHost, s) != hipSuccess ||
      hipStreamSynchronize(s) != hipSuccess)
    return fail(CHS_EHIP, "copy out");
  return CHS_OK;
}

int chs_mlp_train(chs_mlp_t* m, int steps, int batch, float lr, float* loss) {
  if (!m || steps < 0 || batch < 1 || batch > kMaxBatch || !(lr > 0.0f)) return fail(CHS_EINVAL, "invalid argument");
  hipStream_t s = m->stream;
  const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
  for (int it = 0; it < steps; ++it) {
    ++m->step;
    const uint32_t sd = mix32(m->seed * 747796405U + (uint32_t)m->step);
    const float c1 = 1.0f - std::pow(b1, (float)m->step), c2 = 1.0f - std::pow(b2, (float)m->step);
    const Adam ad{m->p32, m->m32, m->v32, m->p16, lr, b1, b2, eps, c1, c2};
    int rc = batch_pass(m, m->xs, m->ts, m->nsamp, batch, sd, 0, &ad, (loss && it == steps - 1) ? loss : nullptr);
    if (rc != CHS_OK) return rc;
  }
  if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return fail(CHS_EHIP, "training");
  return CHS_OK;
}

int chs_mlp_set_matrix_cores(chs_mlp_t* m, int on) {
  if (!m) return fail(CHS_EINVAL, "null handle");
  m->matrix_cores = on != 0;
  return CHS_OK;
}

int chs_mlp_eval(chs_mlp_t* m, const double* h, long n, double* T, double* rho, double* mu, double* kappa,
                 double* cp, int mem) {
  if (!m || !h || n < 0) return fail(CHS_EINVAL, "invalid argument");
  if (mem != CHS_MEM_HOST && mem != CHS_MEM_DEVICE) return fail(CHS_EINVAL, "invalid mem kind");
  if (n == 0) return CHS_OK;
  hipStream_t s = m->stream;
  double* outs[NO] = {T, rho, mu, kappa, cp};
  const double* din = h;
  double* dout[NO] = {T, rho, mu, kappa, cp};
  if (mem == CHS_MEM_HOST) {
    int nout = 0;
    for (double* o : outs) nout += o != nullptr;
    const size_t need = sizeof(double) * (size_t)n * (1 + nout);
    if (need > m->io_bytes) {
      if (m->io) (void)hipFree(m->io);
      m->io = nullptr;
      m->io_bytes = 0;
      if (hipMalloc(&m->io, need) != hipSuccess) return fail(CHS_ENOMEM, "staging allocation failed");
      m->io_bytes = need;
    }
    double* base = static_cast<double*>(m->io);
    if (hipMemcpyAsync(base, h, sizeof(double) * n, hipMemcpyHostToDevice, s) != hipSuccess)
      return fail(CHS_EHIP, "copy in");
    din = base;
    int slot = 1;
    for (int o = 0; o < NO; ++o) dout[o] = outs[o] ? base + (size_t)n * slot++ : nullptr;
  }
  hipLaunchKernelGGL(k_eval, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, m->p16, m->nm, din, n, dout[0],
                     dout[1], dout[2], dout[3], dout[4]);
  if (hipGetLastError() != hipSuccess) return fail(CHS_EHIP, "inference launch");
  if (mem == CHS_MEM_HOST)
    for (int o = 0; o < NO; ++o)
      if (outs[o] && hipMemcpyAsync(outs[o], dout[o], sizeof(double) * n, hipMemcpyDeviceToHost, s) != hipSuccess)
        return fail(CHS_EHIP, "copy out");
  if (hipStreamSynchronize(s) != hipSuccess) return fail(CHS_EHIP, "synchronise");
  return CHS_OK;
}

}  // extern "C"
