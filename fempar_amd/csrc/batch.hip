// batch.hip -- many independent Poisson problems advanced together.
//
// Problem = FEMPAR's test_poisson setting on its own structured mesh: Q1 on the
// unit square/cube, strong Dirichlet on the whole boundary, constant k, source
// f = f0 k d pi^2 prod sin(pi x) (Sources/Tests/Serial/test_poisson/modules/
// poisson_discrete_integration.f90:62-141 with a coefficient).  With the whole
// boundary fixed, first-touch numbering (Integration/FESpace/
// sbm_serial_fe_space.i90:2623-2922) numbers the free nodes lexicographically,
// so row r is interior node (a,b,c) = r in base m = n-1 and every row's columns
// are r + dx + m dy + m^2 dz, (dx,dy,dz) in {-1,0,1}^d: the matrix is a
// diagonal matrix with 3^d diagonals.  Each problem stores its diagonals
// [k][row] (rows padded to 64) in a shared pool at a per-problem offset.
//
// Assembly: one launch over (problem, 256-row chunk) tasks; a thread owns a
// row and writes its entries, which are the same in every row that has them, and
// its load, a product of 1-D integrals (k_batch_loads).
//
// Solve, problems up to about 16000 rows: a workgroup each (k_batch_small).
//
// Solve, the others: every problem advances by one CG iteration in each pass.  A
// pass is one launch over the workgroups of all problems (a table gives each its
// problem and its tile there, a problem's workgroups on one XCD), in which a
// problem goes through the slots of the FP32-refined solver: FP32 CG in the
// one-launch form with FP64 reliable updates, its products formed from the
// cells, which with constant k are one stencil: 32 B a row and pass, nothing
// stored but the vectors.  With the whole boundary fixed every diagonal entry
// is the same, so Jacobi is a division by it: the passes run on A / diag.
// Problems that are done return at entry; the host queues chunks of passes (a
// hipGraph) until the device has counted every problem done.  Completion is
// stamped with the device wall clock.
// (One workgroup a problem whatever its size leaves the end of a batch to the
// largest, each at the rate of one CU: 512 problems up to 256^2 and 48^3 took
// 66 ms of solving to 1e-8 and 110 ms to 1e-10, now 8.2 and 13.0 ms; one 40^3 23.5
// and 39 ms, now 0.44 and 0.76 ms.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <numeric>

#include "femhip_internal.h"
#include "cg_state.h"
#include "lattice.h"
#include "lattice_io.h"

namespace femhip {
namespace {

constexpr double kPi = 3.14159265358979323846;
constexpr int kChunk = 256;   // rows per assembly task

struct BProb {
  int dim, n, m, nrows, K, stride, cls, pad;
  int64_t voff;   // entry offset of diagonal 0 in the value pools
  int64_t xoff;   // entry offset in the vector pools
  double k, f0;
};

struct BOut {
  int iters, updates, conv, pad;
  double rnorm, bnorm;
  long long t_end;
};

struct BTables {             // per (dim, n) class: element stiffness, weighted shapes
  double E[64];              // unit-coefficient element matrix, row-major [i][j]
  double xi[8][3];           // quadrature points on the reference cell [0,1]^d
  double S[27];              // entries of a row's diagonals, unit coefficient
  int nd, n;
  int64_t loff;              // its loads
};

__device__ __forceinline__ void diag_shift(int k, int dim, int &dx, int &dy, int &dz) {
  dx = k % 3 - 1;
  dy = dim > 1 ? (k / 3) % 3 - 1 : 0;
  dz = dim > 2 ? k / 9 - 1 : 0;
}

// ---------------------------------------------------------------- assembly ---

// The load integrals of a side of n cells, int sin(pi x) N_i over the two cells
// around node i with two Gauss points each; one workgroup a size.  The source is
// a product of sines and so is a shape function of 1-D ones: a row's load is the
// product of its node's integrals.
__global__ __launch_bounds__(kChunk) void k_batch_loads(const BTables *__restrict__ tabs, double *__restrict__ loads) {
  const BTables &T = tabs[blockIdx.x];
  const double h = 1.0 / T.n;
  for (int i = 1 + threadIdx.x; i < T.n; i += kChunk) {
    double s = 0.0;
    for (int q = 0; q < 2; ++q) {
      const double xi = T.xi[q][0];   // in the first direction the points ascend with q
      s += sin(kPi * (((double)(i - 1) + xi) * h)) * xi + sin(kPi * (((double)i + xi) * h)) * (1.0 - xi);
    }
    loads[T.loff + i] = 0.5 * h * s;
  }
}

// With the whole boundary fixed every row has all the cells around its node, so
// a diagonal's entry is the same in every row that has it: BTables::S, summed on
// the host over the cells in ascending order.  512 problems up to 256^2 and 48^3:
// 2.7 ms with the cells summed and the source's sines formed row by row, 0.45 so.
__global__ __launch_bounds__(kChunk) void k_batch_assemble(const BProb *__restrict__ probs, int count,
                                                           const int64_t *__restrict__ task_ptr,
                                                           const BTables *__restrict__ tabs,
                                                           const double *__restrict__ loads,
                                                           double *__restrict__ v64, double *__restrict__ bvec) {
  // problem of this block: last p with task_ptr[p] <= blockIdx.x
  int lo = 0, hi = count - 1;
  const int64_t t = blockIdx.x;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (task_ptr[mid] <= t) lo = mid;
    else hi = mid - 1;
  }
  const BProb P = probs[lo];
  const BTables &T = tabs[P.cls];
  const int r = (int)(t - task_ptr[lo]) * kChunk + threadIdx.x;
  if (r >= P.stride) return;
  double *V = v64 + P.voff;
  if (r >= P.nrows) {   // padding rows
    for (int k = 0; k < P.K; ++k) {
      V[(int64_t)k * P.stride + r] = 0.0;
    }
    bvec[P.xoff + r] = 0.0;
    return;
  }
  const int dim = P.dim, m = P.m;
  const int a[3] = {r % m, dim > 1 ? (r / m) % m : 0, dim > 2 ? r / (m * m) : 0};
  for (int k = 0; k < P.K; ++k) {
    int dd[3];
    diag_shift(k, dim, dd[0], dd[1], dd[2]);
    bool valid = true;
    for (int d = 0; d < dim; ++d) valid = valid && (a[d] + dd[d] >= 0) && (a[d] + dd[d] < m);
    V[(int64_t)k * P.stride + r] = valid ? T.S[k] * P.k : 0.0;
  }
  const double *load = loads + T.loff + 1;
  double bsum = P.f0 * P.k * dim * kPi * kPi;
  for (int d = 0; d < dim; ++d) bsum *= load[a[d]];
  bvec[P.xoff + r] = bsum;
}

// ------------------------------------------------------------------- solve ---

constexpr int kBatchThreads = 256;

// A problem in the passes.
struct BSolve {
  Lattice g;
  int dim, nrows, blocks, id;
  int64_t xoff, poff;        // offsets in the vector pools and in the partial sums
  double c[3], cu[3];        // cell weights of A, and of A / diag
  double inv_diag;
};

struct BPools {
  const double *b;
  double *x;
  PairOf<float> r, q, p;
  float *d;
  double *part[2];           // the passes' sums, alternating
};

struct BCount {
  int done;
  int pad;
  long long t0;
};

// problem and logical workgroup of this block (problem -1: none)
__device__ __forceinline__ int2 batch_block(const int2 *__restrict__ table) { return table[blockIdx.x]; }

__global__ void k_batch_start(BCount *count) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    count->done = 0;
    count->t0 = (long long)wall_clock64();
  }
}

// x = 0, d = 0, r = b / diag; partials ||r32||^2, ||b||^2
__global__ __launch_bounds__(kBatchThreads) void k_batch_init(const BSolve *__restrict__ probs,
                                                              const int2 *__restrict__ table, BPools pl) {
  const int2 at = batch_block(table);
  if (at.x < 0) return;
  const BSolve &P = probs[at.x];
  double v[2] = {0.0, 0.0};
  for (int64_t i = (int64_t)at.y * kBatchThreads + threadIdx.x; i < P.nrows; i += (int64_t)P.blocks * kBatchThreads) {
    const double bi = pl.b[P.xoff + i];
    const float rf = (float)(P.inv_diag * bi);
    pl.x[P.xoff + i] = 0.0;
    pl.d[P.xoff + i] = 0.0f;
    pl.r.v[0][P.xoff + i] = rf;
    v[0] += (double)rf * (double)rf;
    v[1] += bi * bi;
  }
  group_partials<2>(v, pl.part[0] + P.poff, P.blocks, at.y);
}

// one wave a problem: its first state (RES_RES, x0 = 0: cg.f90:305-307)
__global__ __launch_bounds__(64) void k_batch_begin(const BSolve *__restrict__ probs, int count, BPools pl, CgState *st,
                                                    double rtol, double delta, int maxit, BOut *out, BCount *cnt) {
  const int pi = blockIdx.x;
  if (pi >= count) return;
  const BSolve &P = probs[pi];
  double v[2];
  group_reduce<2>(pl.part[0] + P.poff, P.blocks, v);
  if (threadIdx.x != 0) return;
  CgState s{};
  s.rtol = rtol;
  s.delta = delta;
  s.maxit = maxit;
  s.crit = FEMHIP_RES_RES;
  s.rz = v[0];
  s.bnorm = s.r0norm = s.rnorm = sqrt(v[1]);
  s.rhs_test = rtol * s.bnorm;
  s.rmax = sqrt(v[0]);
  s.rscale = s.bnorm > 0.0 ? s.rmax / s.bnorm : 1.0;
  s.first = 1;
  s.converged = s.bnorm <= s.rhs_test;
  s.done = s.converged || maxit <= 0;
  st[2 * pi] = st[2 * pi + 1] = s;
  BOut o{0, 0, s.converged, 0, s.bnorm, s.bnorm, 0};
  if (s.done) {
    o.t_end = (long long)wall_clock64();
    atomicAdd(&cnt->done, 1);
  }
  out[P.id] = o;
}

template <int DIM>
__device__ __forceinline__ void batch_pass(const BSolve &P, int lb, const BPools &pl, CgState *S, int par, BOut *out,
                                           BCount *cnt, double *lds) {
  double sums_in[kSums];
  group_begin<kSums>(pl.part[par ^ 1] + P.poff, P.blocks, sums_in);
  const CgState &cur = S[par];
  CgState &next = S[par ^ 1];
  const bool lead = lb == 0 && threadIdx.x == 0;
  if (cur.done) {
    if (lead) next.done = 1;
    return;
  }
  double *part_out = pl.part[par] + P.poff;
  const int set = cur.set;
  int64_t row0, rows;
  const Lattice w = lattice_window(P.g, DIM, 1, lb, row0, rows);
  const int64_t off = P.xoff + row0;
  const uint32_t b4 = 4u * (uint32_t)rows, b8 = 8u * (uint32_t)rows;
  CellQ1<DIM, kCoefCell> cell;
  cell.k = CoefDev{};
  if (cur.ru == 1) {
    if (lead) {
      next = cur;
      next.ru = 2;
    }
    IoRes io{pl.x + off, pl.b + off, nullptr, nullptr, nullptr, pl.r.v[set] + off, nullptr, kLatUpdate,
             {0.0, 0.0, 0.0, 0.0}, buf_of(pl.x + off, b8), P.inv_diag};
    for (int d = 0; d < DIM; ++d) cell.k.c[d] = P.c[d];
    lattice_march<DIM, 1>(w, lb, cell, io, lds);
    double v[2] = {io.acc[0], io.acc[1]};
    group_partials<2>(v, part_out, P.blocks, lb);
    return;
  }
  int act = kRfGo;
  auto begin = [&](double &alpha, double &beta) {
    CgResult unused;
    act = rf_begin(cur, next, lead, sums_in, &unused, alpha, beta);
    return act == kRfGo;
  };
  const uint32_t old = cur.first == 1 ? 0 : b4;
  IoRf<decltype(begin)> io{buf_of(pl.r.v[set] + off, b4), buf_of(pl.q.v[set] + off, cur.ru == 2 ? 0 : old),
                           buf_of(nullptr, 0), buf_of(pl.p.v[set] + off, old), buf_of(pl.r.v[set ^ 1] + off, b4),
                           buf_of(pl.q.v[set ^ 1] + off, b4), buf_of(pl.p.v[set ^ 1] + off, b4),
                           buf_of(pl.d + off, b4), false, begin, 0.0f, 0.0f, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}};
  for (int d = 0; d < DIM; ++d) cell.k.c[d] = P.cu[d];
  if (!lattice_march<DIM, 1>(w, lb, cell, io, lds)) io.ready();   // no cells: the decision all the same
  if (act == kRfFold)
    for (int64_t i = (int64_t)lb * kBatchThreads + threadIdx.x; i < P.nrows; i += (int64_t)P.blocks * kBatchThreads) {
      pl.x[P.xoff + i] += (double)pl.d[P.xoff + i];
      pl.d[P.xoff + i] = 0.0f;
    }
  if (act == kRfDone && lead) {
    out->iters = next.iter;
    out->updates = next.updates;
    out->conv = next.converged;
    out->rnorm = next.rnorm;
    out->t_end = (long long)wall_clock64();
    atomicAdd(&cnt->done, 1);
  }
  if (act != kRfGo) return;
  group_partials<kSums>(io.sum, part_out, P.blocks, lb);
}

__global__ __launch_bounds__(kBatchThreads, 4) void k_batch_pass(const BSolve *__restrict__ probs,
                                                                 const int2 *__restrict__ table, BPools pl, CgState *st,
                                                                 int par, BOut *out, BCount *cnt) {
  const int2 at = batch_block(table);
  if (at.x < 0) return;
  const BSolve &P = probs[at.x];
  if (P.dim == 2) batch_pass<2>(P, at.y, pl, st + 2 * at.x, par, out + P.id, cnt, lattice_smem);
  else batch_pass<3>(P, at.y, pl, st + 2 * at.x, par, out + P.id, cnt, lattice_smem);
}

// ------------------------------------------------------- small problems ---
//
// A problem that fits one workgroup's registers (at most RPT rows a thread) is
// solved there from start to end: its direction lies in LDS inside a frame of
// zeros, a thread owns a run of rows along the last direction, and the product
// is the constant stencil by the number of directions two nodes differ in:
// weights w0..w3.  Three LDS (9 in 3-D) reads a row, no memory traffic but the
// reliable updates', three barriers an iteration.  64^2 cells take 5.5 us an
// iteration (10 us with the matrix streamed from memory; 9 us a pass in the
// passes), 500 problems of 58 rows 33 us in all (69 us; 333 us in the passes).

struct BSmall {
  double c[4], inv_diag;     // weights of A; 1 / its diagonal
  float cu[4];               // weights of A / diag
  int id, dim, m, nrows;
  int cols, segs, len, plane;   // columns, runs a column, rows a run, frame entries a plane
  int64_t xoff;
};

struct BParams {
  double rtol, delta;
  int maxit, pad;
};

// sums of v over the workgroup, the same in every thread; sm: NV rows
template <int T, int NV>
__device__ __forceinline__ void small_sum(double (&v)[NV], double *sm) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int k = 0; k < NV; ++k) v[k] += __shfl_xor(v[k], off, 64);
  if constexpr (T > 64) {
    const int w = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0)
#pragma unroll
      for (int k = 0; k < NV; ++k) sm[k * (T / 64) + w] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      double s = 0.0;
#pragma unroll
      for (int i = 0; i < T / 64; ++i) s += sm[k * (T / 64) + i];
      v[k] = s;
    }
  } else {
    __syncthreads();
  }
}

// The stencil along a run: f(j, centre, w0 u + ...) for rows j < len
template <int DIM, int RPT, class Real, class F>
__device__ __forceinline__ void run_stencil(const Real *u, int at, int L, int plane, int len, const Real (&w)[4], F &&f) {
  Real a[3], b[3], c[3];   // in-plane sums: own node, the neighbours' share, centre
#pragma unroll
  for (int j = 0; j < RPT + 2; ++j) {
    if (j < len + 2) {
      if (j > 0) {
        at += plane;
        asm volatile("" : "+v"(at));   // formed here: addresses kept for every row would spill
      }
      const Real *q = u + at;
      const Real p0 = q[0], p1 = q[-1] + q[1] + (DIM == 3 ? q[-L] + q[L] : Real(0));
      Real own = w[0] * p0 + w[1] * p1, side = w[1] * p0 + w[2] * p1;
      if (DIM == 3) {
        const Real p2 = (q[-L - 1] + q[-L + 1]) + (q[L - 1] + q[L + 1]);
        own += w[2] * p2;
        side += w[3] * p2;
      }
      a[j % 3] = own;
      b[j % 3] = side;
      c[j % 3] = p0;
      if (j >= 2) f(j - 2, c[(j - 1) % 3], a[(j - 1) % 3] + (b[j % 3] + b[(j - 2) % 3]));
      if (RPT > 8 || sizeof(Real) > 4) __builtin_amdgcn_sched_barrier(0);   // a row's loads at a time: registers
    }
  }
}

template <int DIM, int T, int RPT>
__device__ __forceinline__ void small_solve(const BSmall &P, const BPools &pl, const BParams &prm, BOut *out, double *lds) {
  __shared__ double sums[6][T / 64];
  const int tid = threadIdx.x, L = P.m + 2, plane = P.plane, len = P.len;
  const int seg = tid / P.cols, col = tid % P.cols, z0 = seg * len;
  const bool active = seg < P.segs;
  const int rows = active ? min(len, P.m - z0) : 0;   // may be < 0: a run past the last row
  // frame entry of the column's own node, in the plane before the run
  const int at = active ? (DIM == 3 ? (col % P.m + 1) + L * (col / P.m + 1) : col + 1) + plane * z0 : L + 1 < plane ? L + 1 : 1;
  const int entries = plane * (P.segs * len + 2);
  const uint32_t row0 = (uint32_t)(col + P.cols * z0), cols = (uint32_t)P.cols;
  double *x = pl.x + P.xoff;
  const double *rhs = pl.b + P.xoff;
  float *u32 = reinterpret_cast<float *>(lds);
  const float w32[4] = {P.cu[0], P.cu[1], P.cu[2], P.cu[3]};
  float r[RPT], p[RPT], d[RPT], q[RPT];
  for (int i = tid; i < entries; i += T) u32[i] = 0.0f;
  double s2[2] = {0.0, 0.0};
#pragma unroll
  for (int j = 0; j < RPT; ++j) {
    r[j] = d[j] = q[j] = 0.0f;
    if (j < rows) {
      const uint32_t i = row0 + cols * (uint32_t)j;
      const double b = rhs[i];
      r[j] = (float)(P.inv_diag * b);
      s2[0] += (double)r[j] * (double)r[j];
      s2[1] += b * b;
      x[i] = 0.0;
    }
    p[j] = r[j];
  }
  small_sum<T>(s2, sums[0]);   // also: the frame is cleared
  auto put = [&]() {
#pragma unroll
    for (int j = 0, to = at; j < RPT; ++j) {
      to += plane;
      asm volatile("" : "+v"(to));
      if (j < rows) u32[to] = p[j];
    }
  };
  double rz = s2[0], rmax = sqrt(s2[0]), rnorm64 = sqrt(s2[1]);
  const double bnorm = rnorm64, rhs_test = prm.rtol * bnorm, scale = fabs(P.inv_diag);
  // readfirstlane: wave-uniform for the compiler as well
  int it = 0, upd = 0, conv = __builtin_amdgcn_readfirstlane(bnorm <= rhs_test ? 1 : 0);
  while (!conv && it < prm.maxit) {
    put();
    __syncthreads();
    double s1[1] = {0.0};
    run_stencil<DIM, RPT>(u32, at, L, plane, len, w32, [&](int j, float, float y) {
      q[j] = j < rows ? y : 0.0f;
      s1[0] += (double)p[j] * (double)q[j];
    });
    small_sum<T>(s1, sums[2]);
    const double alpha = s1[0] != 0.0 ? rz / s1[0] : 0.0;
    const float af = (float)alpha;
    double sr[1] = {0.0};
#pragma unroll
    for (int j = 0; j < RPT; ++j) {
      d[j] = __builtin_fmaf(af, p[j], d[j]);
      r[j] = __builtin_fmaf(-af, q[j], r[j]);
      sr[0] += (double)r[j] * (double)r[j];
    }
    small_sum<T>(sr, sums[3]);
    ++it;
    const double rnorm = sqrt(sr[0]);
    double rz_new = sr[0];
    rmax = fmax(rmax, rnorm);
    const int update = __builtin_amdgcn_readfirstlane((rnorm < prm.delta * rmax || rnorm <= rhs_test * scale || it >= prm.maxit) ? 1 : 0);
    if (update) {   // x += d; r = b - A x in FP64 replaces the FP32 residual
      for (int e = tid; e < entries; e += T) lds[e] = 0.0;
      __syncthreads();
      uint32_t i = row0;
#pragma unroll
      for (int j = 0, to = at; j < RPT; ++j) {
        to += plane;
        asm volatile("" : "+v"(to), "+v"(i));
        if (j < rows) lds[to] = x[i] + (double)d[j];
        i += cols;
      }
      i = row0;
      __syncthreads();
      double t2[2] = {0.0, 0.0};
      run_stencil<DIM, RPT>(lds, at, L, plane, len, P.c, [&](int j, double xj, double y) {
        asm volatile("" : "+v"(i));
        if (j < rows) {
          x[i] = xj;
          const double ri = rhs[i] - y;
          r[j] = (float)(P.inv_diag * ri);
          t2[0] += (double)r[j] * (double)r[j];
          t2[1] += ri * ri;
        }
        d[j] = 0.0f;
        i += cols;
      });
      small_sum<T>(t2, sums[4]);
      for (int i = tid; i < entries; i += T) u32[i] = 0.0f;   // the frame again
      __syncthreads();
      ++upd;
      rz_new = t2[0];
      rmax = sqrt(t2[0]);
      rnorm64 = sqrt(t2[1]);
      conv = __builtin_amdgcn_readfirstlane(rnorm64 <= rhs_test ? 1 : 0);
    }
    const float beta = (float)(rz_new / rz);
    rz = rz_new;
#pragma unroll
    for (int j = 0; j < RPT; ++j) p[j] = dir_value(beta, p[j], r[j]);
  }
  if (tid == 0) {
    BOut o{it, upd, conv, 0, rnorm64, bnorm, (long long)wall_clock64()};
    out[P.id] = o;
  }
}

template <int T, int RPT>
__global__ __launch_bounds__(T) void k_batch_small(const BSmall *__restrict__ probs, int count, BPools pl, BParams prm,
                                                   BOut *out) {
  if ((int)blockIdx.x >= count) return;
  const BSmall P = probs[blockIdx.x];
  if (P.dim == 2) small_solve<2, T, RPT>(P, pl, prm, out, lattice_smem);
  else small_solve<3, T, RPT>(P, pl, prm, out, lattice_smem);
}

// the count of finished problems, for the host
__global__ void k_batch_poll(const BCount *cnt, int *host) {
  if (threadIdx.x == 0) *host = cnt->done;
}

}  // namespace
}  // namespace femhip

using namespace femhip;

// workgroups of the small problems: threads, rows a thread
constexpr int kSmallClasses = 3;
constexpr int kSmallT[kSmallClasses] = {64, 256, 1024}, kSmallRows[kSmallClasses] = {8, 8, 16};
constexpr size_t kSmallLds = 144 * 1024;

struct femhip_batch {
  femhip_ctx *ctx = nullptr;
  femhip_cg_params_t prm{};
  std::vector<BProb> probs;
  std::vector<int64_t> task_ptr;
  int64_t entries = 0, vec = 0;
  DevBuf<BProb> d_probs;
  DevBuf<int64_t> d_task;
  DevBuf<BTables> d_tabs;
  DevBuf<double> v64, b, x, loads;
  int sizes = 0;                     // distinct (dim, n)
  // passes
  DevBuf<BSmall> d_small;            // by class
  int small_at[kSmallClasses + 1] = {};
  size_t small_lds[kSmallClasses] = {};
  DevBuf<BSolve> d_solve;
  int passes = 0;                    // problems in the passes
  DevBuf<int2> table;
  int blocks = 0;                    // entries of the table
  size_t lds = 0;
  DevBuf<float> r[2], p[2], q[2], d;
  DevBuf<double> part[2];
  DevBuf<CgState> st;
  DevBuf<BOut> out;
  DevBuf<BCount> cnt;
  int *h_done[2] = {nullptr, nullptr}, *d_done[2] = {nullptr, nullptr};   // pinned, mapped
  hipEvent_t ev[2] = {nullptr, nullptr};
  hipGraphExec_t graph[2] = {nullptr, nullptr};
  bool assembled = false;
  ~femhip_batch() {
    for (auto g : graph)
      if (g) (void)hipGraphExecDestroy(g);
    for (auto *h : h_done)
      if (h) (void)hipHostFree(h);
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
  }
};

namespace femhip {
namespace {

BPools pools(femhip_batch &B);

template <int K>
constexpr auto small_kernel = k_batch_small<kSmallT[K], kSmallRows[K]>;

template <int K>
void launch_small(femhip_batch &B, const BParams &prm) {
  const int count = B.small_at[K + 1] - B.small_at[K];
  if (!count) return;
  hipLaunchKernelGGL(small_kernel<K>, dim3((unsigned)count), dim3(kSmallT[K]), B.small_lds[K], B.ctx->stream,
                     B.d_small.p + B.small_at[K], count, pools(B), prm, B.out.p);
}

BPools pools(femhip_batch &B) {
  return BPools{B.b.p, B.x.p, {{B.r[0].p, B.r[1].p}}, {{B.q[0].p, B.q[1].p}}, {{B.p[0].p, B.p[1].p}}, B.d.p,
                {B.part[0].p, B.part[1].p}};
}

// The class a problem is solved in by one workgroup, -1: in the passes.
int small_class(const BProb &P, BSmall &S) {
  for (int k = 0; k < kSmallClasses; ++k) {
    const int64_t cols = P.dim == 3 ? (int64_t)P.m * P.m : P.m;
    if (cols > kSmallT[k]) continue;
    S.dim = P.dim;
    S.m = P.m;
    S.nrows = P.nrows;
    S.xoff = P.xoff;
    S.cols = (int)cols;
    S.segs = std::min(P.m, kSmallT[k] / S.cols);
    S.len = (P.m + S.segs - 1) / S.segs;
    S.segs = (P.m + S.len - 1) / S.len;
    S.plane = P.dim == 3 ? (P.m + 2) * (P.m + 2) : P.m + 2;
    if (S.len <= kSmallRows[k] && sizeof(double) * S.plane * (S.segs * S.len + 2) <= kSmallLds) return k;
  }
  return -1;
}

// Each problem's path; tiles of the problems in the passes and the table of
// their workgroups.  A workgroup takes about an eighth of what would fill every
// CU once, within bounds: long marches repeat little, short ones leave no CU
// waiting for the last problem (512 mixed problems to 1e-8: 8.2 ms, a quarter 9.6, a
// half 12.3).  Each workgroup of a problem reads the partial sums of all of them, so
// a problem has at most kMostGroups, or as many as its tiles and windows need (four
// of 1000^2 cells: 33.3 ms with 570, 23.0; the mixed problems 8.2 either way).
constexpr int kMostGroups = 192;
void plan_passes(femhip_batch &B, const std::vector<BTables> &tabs) {
  const int count = (int)B.probs.size();
  std::vector<BSmall> small[kSmallClasses];
  std::vector<BSolve> sv;
  std::vector<int> large;
  int64_t total = 0;
  for (int i = 0; i < count; ++i) {
    const BProb &P = B.probs[(size_t)i];
    BSmall S{};
    const int cls = small_class(P, S);
    if (cls < 0) {
      large.push_back(i);
      total += P.nrows;
      continue;
    }
    const BTables &T = tabs[(size_t)P.cls];
    double w[4] = {0.0, 0.0, 0.0, 0.0};   // the entries of a class are the same but for rounding
    for (int a = 0; a < T.nd; ++a)
      for (int b2 = 0; b2 < T.nd; ++b2) w[__builtin_popcount((unsigned)(a ^ b2))] += T.E[a * T.nd + b2];
    // 2^d C(d, t) pairs differ in t directions; 2^(d-t) cells hold such a pair
    const double pairs[2][4] = {{1, 2, 1, 1}, {1, 3, 3, 1}};
    for (int t = 0; t <= P.dim; ++t) w[t] /= pairs[P.dim - 2][t] * (double)(1 << t);
    for (int t = 0; t < 4; ++t) {
      S.c[t] = P.k * w[t];
      S.cu[t] = (float)(w[t] / w[0]);
    }
    S.inv_diag = 1.0 / (P.k * w[0]);
    S.id = i;
    small[cls].push_back(S);
    B.small_lds[cls] = std::max(B.small_lds[cls], sizeof(double) * (size_t)S.plane * (size_t)(S.segs * S.len + 2));
  }
  size_t nsmall = 0;
  for (int k = 0; k < kSmallClasses; ++k) {
    std::stable_sort(small[k].begin(), small[k].end(), [](const BSmall &a, const BSmall &b2) { return a.nrows > b2.nrows; });
    B.small_at[k] = (int)nsmall;
    nsmall += small[k].size();
  }
  B.small_at[kSmallClasses] = (int)nsmall;
  if (nsmall) {
    B.d_small.alloc(nsmall);
    for (int k = 0; k < kSmallClasses; ++k)
      if (!small[k].empty())
        FH_HIP(hipMemcpy(B.d_small.p + B.small_at[k], small[k].data(), sizeof(BSmall) * small[k].size(), hipMemcpyHostToDevice));
    const void *fn[kSmallClasses] = {(const void *)small_kernel<0>, (const void *)small_kernel<1>, (const void *)small_kernel<2>};
    for (int k = 0; k < kSmallClasses; ++k)
      FH_HIP(hipFuncSetAttribute(fn[k], hipFuncAttributeMaxDynamicSharedMemorySize, (int)kSmallLds));
  }
  B.cnt.alloc(1);
  B.passes = (int)large.size();
  if (large.empty()) return;
  const int per = (int)std::min<int64_t>(16384, std::max<int64_t>(1024, total / (8 * std::max(1, B.ctx->num_cus))));
  std::vector<std::vector<int2>> lists(8);   // one an XCD: a problem's workgroups share an L2
  int64_t poff = 0;
  for (int i : large) {
    const BProb &P = B.probs[(size_t)i];
    femhip_mesh_desc_t mesh{};
    mesh.dim = P.dim;
    mesh.order = 1;
    mesh.num_components = 1;
    mesh.dirichlet = FEMHIP_BC_ALL_BOUNDARY;
    for (int d = 0; d < 3; ++d) {
      mesh.n[d] = d < P.dim ? P.n : 1;
      mesh.limits[2 * d + 1] = 1.0;
    }
    LatticeOp L;
    FH_CHECK(lattice_plan(mesh, 0, L, kBatchThreads, std::max(per, P.nrows / kMostGroups)), FEMHIP_ERR_INVALID, "batch problem too large");
    BSolve S{};
    S.g = L.g;
    S.dim = P.dim;
    S.nrows = P.nrows;
    S.blocks = L.grid;
    S.id = i;
    S.xoff = P.xoff;
    S.poff = poff;
    poff += (int64_t)kSums * L.grid;
    const BTables &T = tabs[(size_t)P.cls];
    double diag = 0.0;   // every row's: the 2^d cells around its node
    for (int a = 0; a < T.nd; ++a) diag += T.E[a * T.nd + a];
    const double h = 1.0 / P.n, w = std::pow(0.5 * h, P.dim) * 4.0 / (h * h) / (double)(1 << (2 * P.dim));
    for (int d = 0; d < 3; ++d) {
      S.c[d] = d < P.dim ? P.k * w : 0.0;
      S.cu[d] = d < P.dim ? w / diag : 0.0;
    }
    S.inv_diag = 1.0 / (P.k * diag);
    B.lds = std::max(B.lds, L.lds);
    sv.push_back(S);
  }
  std::stable_sort(sv.begin(), sv.end(), [](const BSolve &a, const BSolve &b2) { return a.blocks > b2.blocks; });
  for (size_t i = 0; i < sv.size(); ++i) {   // largest first to the shortest list
    auto &l = *std::min_element(lists.begin(), lists.end(), [](const auto &a, const auto &b2) { return a.size() < b2.size(); });
    for (int k = 0; k < sv[i].blocks; ++k) l.push_back(int2{(int)i, k});
  }
  size_t rows = 0;
  for (auto &l : lists) rows = std::max(rows, l.size());
  FH_CHECK(rows * 8 < (size_t)INT32_MAX, FEMHIP_ERR_INVALID, "batch too large");
  std::vector<int2> table(rows * 8, int2{-1, 0});
  for (int x = 0; x < 8; ++x)
    for (size_t j = 0; j < lists[(size_t)x].size(); ++j) table[j * 8 + (size_t)x] = lists[(size_t)x][j];
  B.blocks = (int)table.size();
  B.table.alloc(table.size());
  B.d_solve.alloc(sv.size());
  FH_HIP(hipMemcpy(B.table.p, table.data(), sizeof(int2) * table.size(), hipMemcpyHostToDevice));
  FH_HIP(hipMemcpy(B.d_solve.p, sv.data(), sizeof(BSolve) * sv.size(), hipMemcpyHostToDevice));
  for (auto *v : {&B.r[0], &B.r[1], &B.p[0], &B.p[1], &B.q[0], &B.q[1], &B.d}) v->alloc((size_t)B.vec);
  for (auto &v : B.part) v.alloc((size_t)poff);
  B.st.alloc(2 * sv.size());
  for (int k = 0; k < 2; ++k) {   // written by the GPU, read by the host: mapped, coherent
    FH_HIP(hipHostMalloc((void **)&B.h_done[k], sizeof(int), hipHostMallocMapped | hipHostMallocCoherent));
    FH_HIP(hipHostGetDevicePointer((void **)&B.d_done[k], B.h_done[k], 0));
    FH_HIP(hipEventCreateWithFlags(&B.ev[k], hipEventDisableTiming));
  }
}

constexpr int kBatchChunk = 16;   // passes a graph (even: the parity restarts at 0)

// the chunk's graph for result slot k, node by node (a stream capture would
// make other threads' synchronous calls fail)
void ensure_chunk(femhip_batch &B, int k) {
  if (B.graph[k]) return;
  hipGraph_t g;
  FH_HIP(hipGraphCreate(&g, 0));
  try {
    hipGraphNode_t last = nullptr;
    auto add = [&](void *fn, dim3 grid, dim3 block, size_t lds, void **args) {
      hipKernelNodeParams prm{};
      prm.func = fn;
      prm.gridDim = grid;
      prm.blockDim = block;
      prm.sharedMemBytes = (unsigned)lds;
      prm.kernelParams = args;
      hipGraphNode_t node;
      FH_HIP(hipGraphAddKernelNode(&node, g, last ? &last : nullptr, last ? 1 : 0, &prm));
      last = node;
    };
    const BSolve *probs = B.d_solve.p;
    const int2 *table = B.table.p;
    BPools pl = pools(B);
    CgState *st = B.st.p;
    BOut *out = B.out.p;
    BCount *cnt = B.cnt.p;
    for (int i = 0; i < kBatchChunk; ++i) {
      int par = i & 1;
      void *args[] = {&probs, &table, &pl, &st, &par, &out, &cnt};
      add((void *)k_batch_pass, dim3((unsigned)B.blocks), dim3(kBatchThreads), B.lds, args);
    }
    const BCount *cc = cnt;
    int *host = B.d_done[k];
    void *args[] = {&cc, &host};
    add((void *)k_batch_poll, dim3(1), dim3(64), 0, args);
    FH_HIP(hipGraphInstantiate(&B.graph[k], g, nullptr, nullptr, 0));
  } catch (...) {
    (void)hipGraphDestroy(g);
    throw;
  }
  FH_HIP(hipGraphDestroy(g));
}

// The small problems (the quickest class first, its largest first), then the passes: enqueue chunks, one
// ahead, until every problem is done.  A problem takes at most 4 maxit + 8
// passes (an update takes three, at most one an iteration).
void run_passes(femhip_batch &B) {
  hipStream_t st = B.ctx->stream;
  const BParams prm{B.prm.rtol, B.prm.inner_rtol > 0 ? B.prm.inner_rtol : 0.1, B.prm.max_num_iterations, 0};
  hipLaunchKernelGGL(k_batch_start, dim3(1), dim3(64), 0, st, B.cnt.p);
  launch_small<0>(B, prm);
  launch_small<1>(B, prm);
  launch_small<2>(B, prm);
  FH_HIP(hipGetLastError());
  const int count = B.passes;
  if (!count) {
    FH_HIP(hipStreamSynchronize(st));
    return;
  }
  for (int k = 0; k < 2; ++k) ensure_chunk(B, k);
  BPools pl = pools(B);
  hipLaunchKernelGGL(k_batch_init, dim3((unsigned)B.blocks), dim3(kBatchThreads), 0, st, B.d_solve.p, B.table.p, pl);
  hipLaunchKernelGGL(k_batch_begin, dim3((unsigned)count), dim3(64), 0, st, B.d_solve.p, count, pl, B.st.p, prm.rtol,
                     prm.delta, prm.maxit, B.out.p, B.cnt.p);
  FH_HIP(hipGetLastError());
  const int64_t most = 4 * (int64_t)B.prm.max_num_iterations + 8;
  int64_t queued = 0;
  auto push = [&](int k) {
    *B.h_done[k] = 0;
    FH_HIP(hipGraphLaunch(B.graph[k], st));
    FH_HIP(hipEventRecord(B.ev[k], st));
    queued += kBatchChunk;
  };
  push(0);
  push(1);
  for (int k = 0;; k ^= 1) {
    FH_HIP(hipEventSynchronize(B.ev[k]));
    if (*B.h_done[k] >= count || queued >= most + 2 * kBatchChunk) break;
    push(k);
  }
  FH_HIP(hipStreamSynchronize(st));
}

}  // namespace
}  // namespace femhip

extern "C" {

int femhip_batch_create(femhip_ctx_t *ctx, int32_t count, const femhip_batch_problem_t *problems,
                        const femhip_cg_params_t *params, femhip_batch_t **batch) {
  try {
    FH_CHECK(ctx && problems && params && batch && count > 0, FEMHIP_ERR_INVALID, "bad argument");
    FH_CHECK(params->precision == FEMHIP_PRECISION_FP32_REFINED, FEMHIP_ERR_INVALID,
             "the batched solver runs the FP32-refined CG");
    FH_CHECK(params->max_num_iterations >= 1 && params->rtol >= 0, FEMHIP_ERR_INVALID, "bad solver parameters");
    FH_HIP(hipSetDevice(ctx->device));
    auto *B = new femhip_batch();
    B->ctx = ctx_retain(ctx);
    try {
      B->prm = *params;
      // classes (dim, n) -> element tables
      std::vector<std::pair<int, int>> cls;
      std::vector<BTables> tabs;
      B->probs.resize((size_t)count);
      int64_t voff = 0, xoff = 0, loff = 0;
      for (int i = 0; i < count; ++i) {
        const femhip_batch_problem_t &pp = problems[i];
        FH_CHECK((pp.dim == 2 || pp.dim == 3) && pp.n >= 2 && pp.n <= 4096, FEMHIP_ERR_INVALID,
                 "batch problem needs dim 2/3 and 2 <= n <= 4096");
        BProb &P = B->probs[(size_t)i];
        P.dim = pp.dim;
        P.n = pp.n;
        P.m = pp.n - 1;
        P.nrows = 1;
        for (int d = 0; d < pp.dim; ++d) P.nrows *= P.m;
        P.K = pp.dim == 2 ? 9 : 27;
        P.stride = (P.nrows + 63) / 64 * 64;
        P.k = pp.k;
        P.f0 = pp.f0;
        auto key = std::make_pair(pp.dim, pp.n);
        auto it = std::find(cls.begin(), cls.end(), key);
        if (it == cls.end()) {
          RefFE fe;
          const double hh = 1.0 / pp.n;
          double h[3] = {hh, hh, hh};
          build_reffe(fe, pp.dim, 1, 1, h);
          BTables T{};
          T.nd = fe.nd;
          T.n = pp.n;
          T.loff = loff;
          loff += pp.n;
          for (int q = 0; q < fe.nq; ++q) {
            const double factor = fe.detj[q] * fe.qw[q];
            for (int a = 0; a < fe.nd; ++a) {
              for (int b2 = 0; b2 < fe.nd; ++b2) {
                double dot = 0.0;
                for (int k = 0; k < 3; ++k) dot += fe.grad[b2][k][q] * fe.grad[a][k][q];
                T.E[a * fe.nd + b2] += factor * dot;
              }
            }
            for (int d = 0; d < 3; ++d) T.xi[q][d] = 0.5 * (fe.qp[d][q] + 1.0);
          }
          for (int k = 0; k < (pp.dim == 2 ? 9 : 27); ++k) {
            const int dd[3] = {k % 3 - 1, (k / 3) % 3 - 1, k / 9 - 1};
            for (int e = 0; e < fe.nd; ++e) {   // cell = node - 1 + e: the node is local 1 - e there
              int li = 0, lj = 0;
              bool in = true;
              for (int d = 0; d < pp.dim; ++d) {
                const int lid = 1 - ((e >> d) & 1), ljd = lid + dd[d];
                in = in && ljd >= 0 && ljd <= 1;
                li |= lid << d;
                lj |= (ljd & 1) << d;
              }
              if (in) T.S[k] += T.E[li * fe.nd + lj];
            }
          }
          cls.push_back(key);
          tabs.push_back(T);
          P.cls = (int)cls.size() - 1;
        } else {
          P.cls = (int)(it - cls.begin());
        }
        P.voff = voff;
        P.xoff = xoff;
        voff += (int64_t)P.K * P.stride;
        xoff += P.stride;
      }
      B->entries = voff;
      B->vec = xoff;
      B->task_ptr.resize((size_t)count + 1);
      B->task_ptr[0] = 0;
      for (int i = 0; i < count; ++i)
        B->task_ptr[(size_t)i + 1] = B->task_ptr[(size_t)i] + (B->probs[(size_t)i].stride + kChunk - 1) / kChunk;
      B->d_probs.alloc((size_t)count);
      B->d_task.alloc((size_t)count + 1);
      B->d_tabs.alloc(tabs.size());
      B->out.alloc((size_t)count);
      FH_HIP(hipMemcpy(B->d_probs.p, B->probs.data(), sizeof(BProb) * count, hipMemcpyHostToDevice));
      FH_HIP(hipMemcpy(B->d_task.p, B->task_ptr.data(), sizeof(int64_t) * (count + 1), hipMemcpyHostToDevice));
      FH_HIP(hipMemcpy(B->d_tabs.p, tabs.data(), sizeof(BTables) * tabs.size(), hipMemcpyHostToDevice));
      B->sizes = (int)tabs.size();
      B->loads.alloc((size_t)loff);
      B->v64.alloc((size_t)B->entries);
      B->b.alloc((size_t)B->vec);
      B->x.alloc((size_t)B->vec);
      plan_passes(*B, tabs);
    } catch (...) {
      femhip_batch_destroy(B);
      throw;
    }
    *batch = B;
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  } catch (const std::bad_alloc &) {
    set_error("host allocation failed");
    return FEMHIP_ERR_OOM;
  }
}

int femhip_batch_assemble(femhip_batch_t *B, double *ms) {
  try {
    FH_CHECK(B, FEMHIP_ERR_INVALID, "null batch");
    FH_HIP(hipSetDevice(B->ctx->device));
    hipStream_t st = B->ctx->stream;
    hipEvent_t e0, e1;
    FH_HIP(hipEventCreate(&e0));
    FH_HIP(hipEventCreate(&e1));
    FH_HIP(hipEventRecord(e0, st));
    const int64_t tasks = B->task_ptr.back();
    FH_CHECK(tasks < (int64_t)INT32_MAX, FEMHIP_ERR_INVALID, "batch too large");
    hipLaunchKernelGGL(k_batch_loads, dim3((unsigned)B->sizes), dim3(kChunk), 0, st, B->d_tabs.p, B->loads.p);
    hipLaunchKernelGGL(k_batch_assemble, dim3((unsigned)tasks), dim3(kChunk), 0, st, B->d_probs.p,
                       (int)B->probs.size(), B->d_task.p, B->d_tabs.p, B->loads.p, B->v64.p, B->b.p);
    FH_HIP(hipGetLastError());
    FH_HIP(hipEventRecord(e1, st));
    FH_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    FH_HIP(hipEventElapsedTime(&t, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (ms) *ms = t;
    B->assembled = true;
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_batch_autotune(femhip_batch_t *B, int32_t *threads) {
  try {
    FH_CHECK(B, FEMHIP_ERR_INVALID, "null batch");
    FH_CHECK(B->assembled, FEMHIP_ERR_STATE, "assemble the batch first");
    FH_HIP(hipSetDevice(B->ctx->device));
    if (threads) *threads = kBatchThreads;   // the passes have one workgroup size
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_batch_solve(femhip_batch_t *B, femhip_batch_result_t *results, double *ms) {
  try {
    FH_CHECK(B, FEMHIP_ERR_INVALID, "null batch");
    FH_CHECK(B->assembled, FEMHIP_ERR_STATE, "assemble the batch first");
    FH_HIP(hipSetDevice(B->ctx->device));
    hipStream_t st = B->ctx->stream;
    hipEvent_t e0, e1;
    FH_HIP(hipEventCreate(&e0));
    FH_HIP(hipEventCreate(&e1));
    FH_HIP(hipEventRecord(e0, st));
    run_passes(*B);
    FH_HIP(hipEventRecord(e1, st));
    FH_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    FH_HIP(hipEventElapsedTime(&t, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (ms) *ms = t;
    if (results) {
      const size_t count = B->probs.size();
      std::vector<BOut> out(count);
      BCount cnt{};
      FH_HIP(hipMemcpy(out.data(), B->out.p, sizeof(BOut) * count, hipMemcpyDeviceToHost));
      FH_HIP(hipMemcpy(&cnt, B->cnt.p, sizeof(cnt), hipMemcpyDeviceToHost));
      int rate_khz = 0;
      FH_HIP(hipDeviceGetAttribute(&rate_khz, hipDeviceAttributeWallClockRate, B->ctx->device));
      const double us_per_tick = rate_khz > 0 ? 1e3 / rate_khz : 0.01;
      for (size_t i = 0; i < count; ++i) {
        femhip_batch_result_t &R = results[i];
        R.num_iterations = out[i].iters;
        R.updates = out[i].updates;
        R.did_converge = out[i].conv;
        R.num_dofs = B->probs[i].nrows;
        R.true_residual = out[i].rnorm;
        R.rhs_norm = out[i].bnorm;
        R.latency_us = (double)(out[i].t_end - cnt.t0) * us_per_tick;
      }
    }
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_batch_get_solution(const femhip_batch_t *B, int32_t i, double *x) {
  try {
    FH_CHECK(B && x && i >= 0 && i < (int)B->probs.size(), FEMHIP_ERR_INVALID, "bad argument");
    FH_HIP(hipSetDevice(B->ctx->device));
    const BProb &P = B->probs[(size_t)i];
    FH_HIP(hipMemcpy(x, B->x.p + P.xoff, sizeof(double) * P.nrows, hipMemcpyDeviceToHost));
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_batch_get_problem_matrix(const femhip_batch_t *B, int32_t i, int32_t *irp, int32_t *ja, double *val,
                                    double *rhs, int64_t *nnz) {
  try {
    FH_CHECK(B && i >= 0 && i < (int)B->probs.size(), FEMHIP_ERR_INVALID, "bad argument");
    FH_CHECK(B->assembled, FEMHIP_ERR_STATE, "assemble the batch first");
    FH_HIP(hipSetDevice(B->ctx->device));
    const BProb &P = B->probs[(size_t)i];
    std::vector<double> V((size_t)P.K * P.stride);
    FH_HIP(hipMemcpy(V.data(), B->v64.p + P.voff, sizeof(double) * V.size(), hipMemcpyDeviceToHost));
    if (rhs) FH_HIP(hipMemcpy(rhs, B->b.p + P.xoff, sizeof(double) * P.nrows, hipMemcpyDeviceToHost));
    int64_t k_out = 0;
    const int m = P.m;
    for (int r = 0; r < P.nrows; ++r) {
      if (irp) irp[r] = (int32_t)(k_out + 1);
      const int a[3] = {r % m, P.dim > 1 ? (r / m) % m : 0, P.dim > 2 ? r / (m * m) : 0};
      for (int k = 0; k < P.K; ++k) {   // ascending offsets = ascending columns
        const int dx = k % 3 - 1, dy = P.dim > 1 ? (k / 3) % 3 - 1 : 0, dz = P.dim > 2 ? k / 9 - 1 : 0;
        const int dd[3] = {dx, dy, dz};
        bool valid = true;
        for (int d = 0; d < P.dim; ++d) valid = valid && a[d] + dd[d] >= 0 && a[d] + dd[d] < m;
        if (!valid) continue;
        const int c = r + dx + m * (dy + m * dz);
        if (ja) ja[k_out] = c + 1;
        if (val) val[k_out] = V[(size_t)k * P.stride + r];
        ++k_out;
      }
    }
    if (irp) irp[P.nrows] = (int32_t)(k_out + 1);
    if (nnz) *nnz = k_out;
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_batch_destroy(femhip_batch_t *B) {
  if (B) {
    femhip_ctx *c = B->ctx;
    if (c) {
      (void)hipSetDevice(c->device);
      (void)hipStreamSynchronize(c->stream);
    }
    delete B;
    ctx_release(c);
  }
  return FEMHIP_OK;
}

}  // extern "C"
