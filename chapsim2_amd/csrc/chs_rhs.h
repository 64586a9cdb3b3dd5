// Fused line operators of the constant-property sub-step.
//
// The momentum right-hand side applies some forty compact operators, and what
// bounds it is the fields they pass to each other through memory.  The kernels
// here keep the staggered operators' partitioned line solve (chs_lineop.hip)
// and put the elementwise work between two operators into the epilogue of the
// first, so that a sub-step reads and writes about 70 fields for its
// right-hand side where one operator per launch moves about 110:
//  - an interpolation and a first derivative of one component in one pass;
//  - that pair along the second direction of a shear stress, which reads the
//    pair of the first direction and stores only
//      f = -(u_i)(u_j) + r (d_j u_i + d_i u_j),
//    the one input of both operators that differentiate it;
//  - the pair of the last normal direction, which forms the divergence and
//    stores the three normal fluxes -u_i u_i + 2 r (d_i u_i - div / 3);
//  - per momentum component one last operator that solves the normal flux and
//    the pressure along the component's own direction and finishes the
//    fractional step (rhs0, the state) in place.
// Several jobs of one kind can share a launch (RhsGroup), y and z lines
// together, which is what small grids need: their launches are latency (ten
// RK3 steps of 64^3 with y and z apart and the corrections on side streams
// 7.06 ms, now 4.6).
// Two RK3 steps at 256x128x256 with the state's copies in and out: FP64 12.8
// -> 9.8 ms, mixed 9.2 -> 7.2 ms; three of six uneven channels as one graph
// 15.5 -> 10.2 ms; ten of 64^3 9.0 -> 4.6 ms.  What bounds the large grids is
// memory: the fields moved per sub-step (about 102 with the projection, 139
// before) at up to the rate of a large copy (4.8 TB/s); in FP64 the register
// spills of the last x operator (132 bytes per lane) and of the normal fluxes
// add 29 and 13 % to those kernels' bytes.  The small grids are bound by each
// launch's serial chain (arguments, one round trip to memory, the solve, the
// stores) and by the code a wave fetches once.
#pragma once

#include <hip/hip_runtime.h>

#include <string>

#include "chs_lineop.h"

namespace chs {

// kinds of job
enum RhsKind : int { RK_SINGLE = 0, RK_PAIR = 1, RK_SHEAR = 2, RK_DIV = 3, RK_FINAL = 4, RK_CORRECT = 5 };

constexpr int kFuseChunks = 32;  // most chunks per line
constexpr int kFuseCo = 6;       // entries of a coefficient row
enum FuseCo : int { FC_LD = 0, FC_AL = 1, FC_SV = 2, FC_SW = 3, FC_LC = 4 };
// Published chunk ends a chunk's two coupling values are formed from: the
// inverse of the reduced system falls off per row with the scheme's decay rate
// (at most 1/3), so the ends of the next d chunks on either side (4 d + 4
// values) hold every term above 2^-59 (FP64) or 2^-36 (FP32) of the largest:
// d = 2 and 1 for the kernels of 16 and 17 rows, 4 and 2 for those of 8 and 9.
// That is checked against the whole inverse when the plan is made.  A short
// last chunk brings the ends beyond it nearer, so a periodic line of many chunks
// whose last has some 2 to 4 rows is refused (x lines of 100, 162, 180, 324, 450
// and 500, in FP32 also 150 and 486; z lines of 324 and 360; in the short form
// more of them) and its flow runs single operators.
template <typename T>
__host__ __device__ constexpr int fuse_band(int rows) {
  return rows >= 16 ? (sizeof(T) == 8 ? 12 : 8) : (sizeof(T) == 8 ? 20 : 12);
}

// Chunks of a fused plan: P chunks of `ell` rows, the last one shorter (at
// least two rows); rows, the kernel's chunk length, is 16 or 17, or 8 or 9 in
// the short form.  x lines take chunks of exactly 16 (8).  y and z lines of a
// multiple of 16 (8) rows do too, up to kFuseChunks of them; others take the
// fewest chunks of at most 17 (9), so the ny + 1 nodes of a channel with a
// multiple of 16 cells need no chunk more than its cells.  False beyond
// kFuseChunks chunks.
// The short form halves each lane's serial work and the code a wave runs
// through, and doubles the waves: what a small grid wants, whose kernels are
// bound by both (kShortCells in chs_flow.hip has the figures).
bool fuse_chunks(int dir, int n, bool short_form, int* P, int* ell, int* rows);

// Kernel view of a fused plan: a staggered operator (interpolation or first
// derivative, cells to nodes or back) whose chunks all carry the same
// coefficient rows, except the first and the last.
template <typename T>
struct FusePlan {
  int n_in, n_out, P, ell;
  int solve, wrap, ends;  // line solve; periodic; the four boundary rows have weights of their own
  int sh;                 // window start: row - 2 + sh (0: to nodes, 1: to cells)
  T c1, c2, sgn;          // bulk weights, 1/h included
  const T* tab;           // 3 x rows x kFuseCo (first, inner, last chunk), P x 2 x fuse_band, P x ell metric
  int ntab, met, neu_lo, neu_hi;
  const T* edge;          // 4 rows x (rows + 3 window weights, 4 wall-value weights), 1/h included
};

// Device copy of a fused plan (ok false: the line does not have the form).
template <typename T>
struct DevFusePlan {
  FusePlan<T> k{};
  int rows = 16;
  T* mem = nullptr;
  bool ok = false;
  ~DevFusePlan();
};
template <typename T>
std::string upload_fuse_plan(const LinePlan& p, int rows, DevFusePlan<T>* out);

// One job.  Fields A (and, RK_FINAL, A2) are read along the line; o1..o4 are
// read, out, out2, out3 written at the output's own points.
//  SINGLE: out = op1(A)
//  PAIR:   out = op1(A), out2 = op2(A)
//  SHEAR:  out = -op1(A) o1 + r (op2(A) + o2)
//  DIV:    div = o1 + o2 + op2(A); out = -op1(A)^2 + 2 r (op2(A) - div / 3);
//          o3 <- -o3^2 + 2 r (o1 - div / 3), o4 <- -o4^2 + 2 r (o2 - div / 3)
//  FINAL:  cur = op1(A) + o1 + o2; rhs = dt (tg cur + tz r0 - ta op2(A2));
//          r0 = cur; q += rhs, or out = rhs when q is null
//  CORRECT (FP64): out += sOut op1(A), out32 its rounding; x lines also subtract
//          bulk[0] and do add += A, add32 its rounding; y lines set the wall
//          rows from fbw (each pointer possibly null)
template <typename T>
struct RhsJob {
  int dir, rows;              // direction; the plans' chunk length
  int nlines, e1;             // lines; lines per plane (y: nx; z: nx)
  long is, ips, os, ops;      // element strides along the line and per plane, input and output
  const T *A, *A2, *fbc, *fbc2;
  FusePlan<T> p1, p2;
  const T *o1, *o2;
  T *o3, *o4;
  T *out, *out2;
  T r, sOut;
  float* out32;
  const double* bulk;
  double* add;
  float* add32;
  // FINAL
  T tg, tz, ta, dt;
  T* r0;
  double* q;
  const double* fbw;          // wall values of q (first and last row of the line)
  double* partial;            // per-block sums of rhs dyw dx dz (x lines)
  const double* dyw;
  double dxdz;
  int n2;                     // y extent (weight index of a line)
};

constexpr int kGroupJobs = 4;
template <typename T>
struct RhsGroup {
  int n = 0;
  int P;                      // most chunks of a job (y and z lines)
  int first[kGroupJobs + 1];  // first block of each job
  RhsJob<T> job[kGroupJobs];
};

// Launch the jobs (all of one kind, chunk length `rows`) as one grid: x lines
// (periodic, contiguous, n_in = n_out), or y and z lines in any mixture.
template <typename T>
std::string launch_rhs_x(int kind, int rows, RhsGroup<T>& g, hipStream_t s);
// y and z lines: the workgroups have lanes for the most chunks of a job (G.P); a
// job's plans have one geometry, and all tables are laid out for `rows`.
template <typename T>
std::string launch_rhs_yz(int kind, int rows, RhsGroup<T>& g, hipStream_t s);
// number of blocks launch_rhs_x takes for one job (entries of its partial sums)
template <typename T>
int rhs_x_blocks(const RhsJob<T>& j);

// Wall values of the y-normal flux, (nx, 4, nz): -v_w^2 + r 2 (dv/dy - (dv/dy) / 3)
// with dv/dy the end rows of the y derivative `P` of the cell values qyiy
// (walls of uniform velocity have no tangential derivatives).
template <typename T>
std::string launch_wall_flux(const DevPlan<T>& P, const Ext3& ein, const T* qyiy, const T* fbc, T r, T* flux,
                             hipStream_t s);

}  // namespace chs
