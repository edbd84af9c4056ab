// multifield.hip -- several scalar fields on one structured mesh with a block
// layout, assembled into a block sparse matrix and solved by a block CG, on
// the device.
//
// FEMPAR's multi-field serial_fe_space_t numbers each field's DOFs by first
// touch with its own counter, started at the number of free DOFs of the
// earlier fields of the same block (sbm_serial_fe_space.i90:2676-2700), and
// its strong Dirichlet sweep runs field by field with one counter
// (:584-640).  Each field here is a femhip space numbered on the device as if
// alone; the block layout adds the offsets.  block_layout_t
// (Integration/FEOperator/block_layout.f90:36-264) maps fields to blocks and
// says which field pairs couple; the block_sparse_assembler_t
// (Integration/FEOperator/block_sparse_assembler.f90:47-224) inserts each
// coupled (row field, column field) part of the element matrix into block
// (block(f), block(g)) of a block_sparse_matrix_t
// (LinearAlgebra/SparseMatrix/block_sparse_matrix.f90), and the element
// vector into the block array.
//
// Device layout: per coupled block (ib, jb) a full-storage CSR (rowptr, col,
// val; a diagonal block's symmetric-storage view is taken row by row when the
// host asks), rows of a block ordered field by field; one vector of all
// blocks' rows concatenated in block order for the RHS and the solver.
// Kernels: the pattern, one wavefront per block row (the columns of the coupled
// fields in the cells around the row's vef, sorted in LDS); the assembly (every
// entry summed over the cells it lies in, in ascending order, from element
// tables, no atomics); a CSR SpMV that adds the blocks of a block row in block
// order.
//
// The coefficients are constants and the mesh is uniform, so every cell has the
// same element tables: where the fields' free nodes are boxes of the grid
// (every numbering of the structured generator; checked on the device), the CG
// forms its products from those tables in the boxes' order, and the assembly
// finds an entry's cells from the two nodes' grid positions.  Numberings that
// are no box lattice keep the row-wise assembly and the CSR product.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "femhip_internal.h"
#include "cg_state.h"
#include "lattice.h"
#include "lattice_io.h"

using namespace femhip;

namespace {

constexpr int kMaxFields = FEMHIP_MAX_FIELDS;
constexpr int kCand = 1024;   // 2^3 cells x 4 fields x 27 DOFs = 864 candidate columns at most

// The column side of one (row field, column block) launch: the coupled
// column fields, their DOF lists, local DOF counts, offsets in the block and
// the offset of the (row field, column field) element table.
struct ColSet {
  int32_t ng;
  const int32_t *dofs[kMaxFields];
  int32_t nd[kMaxFields];
  int32_t off[kMaxFields];
  int32_t tab[kMaxFields];
  int32_t fld[kMaxFields], rows[kMaxFields];   // which field, its free rows
};

__device__ __forceinline__ int col_candidate(const ColSet &cs, int tot, int i, int &b, int &g, int &j) {
  b = i / tot;
  int rem = i % tot;
  g = 0;
  while (g < cs.ng - 1 && rem >= cs.nd[g]) {
    rem -= cs.nd[g];
    ++g;
  }
  j = rem;
  return 0;
}

// The cells around the vef of a row's representative (cell, local DOF):
// along each axis the vef is not tangent to, the two cells on either side
// (clipped to the mesh).  Bit e of b picks the upper cell along the e-th such
// axis, so b ascending visits the cells in ascending index.
struct Around {
  int ijk[3];
  int ax[3];
  int m;
  int f;     // the vef's n-face in the representative's cell
  int pos;   // the DOF's position in that n-face's own list
};

__device__ __forceinline__ Around around_of(const FaceTab &t, int64_t rep) {
  Around a;
  const int64_t cell = rep / t.nd;
  const int l = (int)(rep % t.nd);
  a.f = t.face_of[l];
  a.pos = t.pos_of[l];
  cell_ijk(t, cell, a.ijk);
  a.m = 0;
  for (int k = 0; k < t.dim; ++k)
    if (!((t.type[a.f] >> k) & 1)) a.ax[a.m++] = k;
  return a;
}

// cell b around the vef (false outside the mesh) and the row DOF's local
// index in it: the same vef is the n-face of the same type whose anchor is
// the vef's position relative to that cell
__device__ __forceinline__ bool around_cell(const FaceTab &t, const Around &a, int b, int64_t &cell, int &lc) {
  int cj[3] = {a.ijk[0], a.ijk[1], a.ijk[2]}, anc = 0;
  for (int e = 0; e < a.m; ++e) {
    const int k = a.ax[e], w = a.ijk[k] + ((t.anchor[a.f] >> k) & 1);
    cj[k] = w - 1 + ((b >> e) & 1);
    if (cj[k] < 0 || cj[k] >= t.n[k]) return false;
    anc |= (w - cj[k]) << k;
  }
  cell = cell_index(t, cj);
  lc = t.lst[t.ptr[t.face_by[t.type[a.f]][anc]] + a.pos];
  return true;
}

// Block pattern, one wavefront per row of the row field (block row = off +
// field row): the distinct free columns of the coupled column fields in the
// cells around the row's vef, sorted (bitonic, in LDS).  Pass 0 counts them
// (and those on or above the diagonal, for a diagonal block's symmetric
// storage), pass 1 writes them.
constexpr int kPatWaves = 2;
template <int PASS>
__global__ __launch_bounds__(kPatWaves * 64) void k_block_pattern(FaceTab t, int32_t nrows, int32_t row_off,
                                                                  const int64_t *__restrict__ rep, ColSet cs,
                                                                  int32_t *__restrict__ len,
                                                                  int32_t *__restrict__ ulen,
                                                                  const int32_t *__restrict__ rowptr,
                                                                  int32_t *__restrict__ col) {
  __shared__ int32_t buf[kPatWaves][kCand];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int32_t fr = blockIdx.x * kPatWaves + w;
  int32_t *s = buf[w];
  int tot = 0;
  for (int g = 0; g < cs.ng; ++g) tot += cs.nd[g];
  if (fr < nrows) {
    const Around a = around_of(t, rep[fr]);
    const int ncand = (1 << a.m) * tot;
    for (int q = 0; q < kCand / 64; ++q) {
      const int i = lane + 64 * q;
      int32_t v = INT_MAX;
      if (i < ncand) {
        int b, g, j;
        col_candidate(cs, tot, i, b, g, j);
        int64_t cell;
        int lc;
        if (around_cell(t, a, b, cell, lc)) {
          const int32_t d = cs.dofs[g][cell * cs.nd[g] + j];
          if (d >= 0) v = d + cs.off[g];
        }
      }
      s[i] = v;
    }
  } else {
    for (int q = 0; q < kCand / 64; ++q) s[lane + 64 * q] = INT_MAX;
  }
  __syncthreads();
  for (int size = 2; size <= kCand; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int q = 0; q < kCand / 128; ++q) {
        const int p = lane + 64 * q;
        const int i = 2 * p - (p & (stride - 1));
        const int j = i + stride;
        const bool up = (i & size) == 0;
        const int32_t x = s[i], y = s[j];
        if ((x > y) == up) {
          s[i] = y;
          s[j] = x;
        }
      }
      __syncthreads();
    }
  if (fr >= nrows) return;
  const int32_t r = row_off + fr;
  int32_t cnt = 0, ucnt = 0;
  const int32_t base = PASS == 1 ? rowptr[r] : 0;
  for (int q = 0; q < kCand / 64; ++q) {
    const int i = lane + 64 * q;
    const int32_t v = s[i];
    const bool first = v != INT_MAX && (i == 0 || s[i - 1] != v);
    const uint64_t mask = __ballot(first);
    if (PASS == 1 && first) col[base + cnt + __popcll(mask & ((1ull << lane) - 1))] = v;
    cnt += __popcll(mask);
    ucnt += __popcll(__ballot(first && v >= r));
  }
  if (PASS == 0 && lane == 0) {
    len[r] = cnt;
    ulen[r] = ucnt;
  }
}

// Block assembly, one wavefront per row of the row field: the row's columns
// and a zeroed value per column in LDS; then, cell by cell in ascending index
// and column field by column field, lane j adds the element entry (the row's
// local DOF in that cell, column DOF j) at the slot of its column (binary
// search); within one
// step the lanes' columns are distinct, so the sum of every entry runs over
// the cells in ascending order, the order of the reference's COO append +
// stable sort.  The row is written once.
__global__ __launch_bounds__(64) void k_block_assemble(FaceTab t, int32_t nrows, int32_t row_off,
                                                       const int64_t *__restrict__ rep, ColSet cs,
                                                       const int32_t *__restrict__ rowptr,
                                                       const int32_t *__restrict__ col,
                                                       const double *__restrict__ tab, double *__restrict__ val) {
  __shared__ int32_t sc[kCand];
  __shared__ double sv[kCand];
  const int lane = threadIdx.x;
  const int32_t fr = blockIdx.x;
  if (fr >= nrows) return;
  const int32_t r = row_off + fr;
  const int32_t b0 = rowptr[r], len = rowptr[r + 1] - b0;
  for (int i = lane; i < len; i += 64) {
    sc[i] = col[b0 + i];
    sv[i] = 0.0;
  }
  __syncthreads();
  const Around a = around_of(t, rep[fr]);
  for (int b = 0; b < (1 << a.m); ++b) {
    int64_t cell;
    int l;
    if (!around_cell(t, a, b, cell, l)) continue;   // the same for the whole block (one row)
    for (int g = 0; g < cs.ng; ++g) {
      if (lane < cs.nd[g]) {
        const int32_t d = cs.dofs[g][cell * cs.nd[g] + lane];
        if (d >= 0) {
          const int32_t c = d + cs.off[g];
          int lo = 0;   // = the number of the row's columns below c (fixed steps, len <= kCand)
#pragma unroll
          for (int h = kCand / 2; h > 0; h >>= 1)
            if (lo + h <= len && sc[lo + h - 1] < c) lo += h;
          sv[lo] += tab[cs.tab[g] + l * cs.nd[g] + lane];
        }
      }
      __syncthreads();
    }
  }
  for (int i = lane; i < len; i += 64) val[b0 + i] = sv[i];
}

// Block RHS, one thread per row of the row field: the element vector entry of
// the row's local DOF summed over the cells around its vef in ascending order
// (element_serial_block_array_assembly adds cell by cell).
__global__ void k_block_rhs(FaceTab t, int32_t nrows, int32_t row_off, const int64_t *__restrict__ rep,
                            const double *__restrict__ elvec, double *__restrict__ rhs) {
  const int32_t fr = blockIdx.x * blockDim.x + threadIdx.x;
  if (fr >= nrows) return;
  const Around a = around_of(t, rep[fr]);
  double acc = 0.0;
  for (int b = 0; b < (1 << a.m); ++b) {
    int64_t cell;
    int l;
    if (around_cell(t, a, b, cell, l)) acc += elvec[l];
  }
  rhs[row_off + fr] = acc;
}

// y = A x (add = 0) or y += A x, full-storage CSR, LANES lanes per row
// (rows of 27 to 125 entries): the lanes stride over the row's entries, so
// the value and column loads of a row are contiguous across the lanes; each
// lane issues the loads of 4 of its entries before it uses the first, so a
// long row is not a chain of dependent round trips; a fixed shuffle tree sums
// the lanes; the blocks of a block row are applied in block order (a
// block_sparse_matrix_t apply).
constexpr int kSpmvThreads = 256;
template <int LANES>
__global__ __launch_bounds__(kSpmvThreads) void k_block_spmv(int32_t n, const int32_t *__restrict__ rowptr,
                                                             const int32_t *__restrict__ col,
                                                             const double *__restrict__ val,
                                                             const double *__restrict__ x, double *__restrict__ y,
                                                             int add, const CgState *stop) {
  if (stop && stop->done) return;   // the solve has ended
  const int sub = threadIdx.x % LANES;
  const int64_t r = ((int64_t)blockIdx.x * kSpmvThreads + threadIdx.x) / LANES;
  double acc = 0.0;
  if (r < n) {
    int32_t k = rowptr[r] + sub;
    const int32_t e = rowptr[r + 1];
    for (; k + 3 * LANES < e; k += 4 * LANES) {
      int32_t c[4];
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        c[u] = col[k + u * LANES];
        v[u] = val[k + u * LANES];
      }
      double g[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) g[u] = x[c[u]];
#pragma unroll
      for (int u = 0; u < 4; ++u) acc += v[u] * g[u];
    }
    for (; k < e; k += LANES) acc += val[k] * x[col[k]];
  }
  for (int o = LANES / 2; o > 0; o >>= 1) acc += __shfl_down(acc, o, LANES);
  if (r < n && sub == 0) y[r] = add ? y[r] + acc : acc;
}

// 16 lanes a row: 8 take the same time, 32 are 20 % slower (48^3 Q2 + Q1 block CG)
constexpr int kSpmvLanes = 16;

// ------------------------------------------------- boxes of the fields ---

// A field's free nodes: the box [o, o + m) of the grid of its order, its rows
// in the block vectors (base) and in its block (off), and the box position of
// each of its rows.
struct MfField {
  int p, nd, rows, off;
  int o[3], m[3];
  int64_t base;
  const int32_t *perm;
};

// The nodes of one field whose positions along y and z have the same parities:
// the cells around them and their local nodes there are the same, so the
// element tables are read by scalar loads.  A thread takes the p nodes from one
// vertex of the cells to the next along x.
struct MfSeg {
  int f, rows, blocks, pad;      // rows: threads; blocks: workgroups on each XCD
  int aligned[3], first[3], cnt[3];
};

struct MfPlan {
  int nf, dim, nseg, items;      // items: workgroups in all
  int n[3], pad;
  MfField fld[kMaxFields];
  MfSeg seg[kMaxFields * 4];
  int tab[kMaxFields][kMaxFields];   // element table of (row, column) fields, -1: not coupled
};

constexpr int kMfThreads = 256;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// A thread's nodes: cell i along x (its first node is the cell's vertex), grid
// positions gy, gz.
struct MfAt {
  int i, g[3];
};

// y[a] += sum over the cells around node a of the element rows times field g's
// values.  The values of 2 PG + 1 nodes along x serve both nodes of a thread
// and both cells of the vertex, in pairs (16 B a lane, so a wave reads whole
// lines); O: field g's box begins at node O, which decides the pairs that never
// begin before it.  Nodes outside the box and cells outside the mesh count 0:
// along y and z by an offset out of the vector's range, along x by selects.
template <int DIM, int PF, int PG, int O>
__device__ __forceinline__ void mf_rows(const MfPlan &P, const MfField &G, const MfSeg &s, const MfAt &at,
                                        const double *__restrict__ tab, BufRsrc x, double (&y)[PF]) {
  constexpr int N1 = PG + 1, NZ = DIM == 3 ? N1 : 1, ND = N1 * N1 * NZ, F1 = PF + 1, NX = 2 * PG + 1;
  const uint32_t sy = 8u * (uint32_t)G.m[0], sz = sy * (uint32_t)G.m[1];
  const bool lower = at.i >= 1, upper = at.i < P.n[0];   // the cells before and after the vertex
  bool in[NX];
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    const int v = PG * at.i - PG + j - G.o[0];
    in[j] = v >= 0 && v < G.m[0];
  }
  auto xoff = [&](int j) { return 8u * (uint32_t)max(PG * at.i - PG + j - G.o[0], 0); };
  auto axis = [&](int d, int e, uint32_t stride, uint32_t (&off)[N1]) {   // local node; byte offsets along d
    const int c = s.aligned[d] ? at.g[d] / PF - 1 + e : at.g[d] / PF;
    const bool cell = c >= 0 && c < P.n[d];
#pragma unroll
    for (int j = 0; j < N1; ++j) {
      const int v = PG * c + j - G.o[d];
      off[j] = cell && v >= 0 && v < G.m[d] ? (uint32_t)v * stride : kNoPlane;
    }
    return s.aligned[d] ? (e ? 0 : PF) : 1;
  };
  const uint32_t x0 = xoff(0), x1 = xoff(1), x2 = xoff(2), x3 = PG == 2 ? xoff(3) : 0, x4 = PG == 2 ? xoff(4) : 0;
  auto pair = [&](uint32_t o, double &a, double &b) {
    const f64x2 v = __builtin_bit_cast(f64x2, __builtin_amdgcn_raw_buffer_load_b128(x, (int)o, 0, 0));
    a = v.x;
    b = v.y;
  };
  for (int ez = 0; ez < (DIM == 3 && s.aligned[2] ? 2 : 1); ++ez) {
    uint32_t oz[N1];
    const int lz = DIM == 3 ? axis(2, ez, sz, oz) : 0;
    for (int ey = 0; ey < (s.aligned[1] ? 2 : 1); ++ey) {
      uint32_t oy[N1];
      const int ly = axis(1, ey, sy, oy);
      const double *row = tab + (lz * F1 + ly) * F1 * ND;
#pragma unroll
      for (int k = 0; k < NZ; ++k) {
        double v[N1][NX];
#pragma unroll
        for (int j = 0; j < N1; ++j) {
          const uint32_t o = (DIM == 3 ? oz[k] : 0u) + oy[j];
          if constexpr (PG == 1) {
            v[j][0] = buf_ld64(x, o + x0);
            v[j][1] = buf_ld64(x, o + x1);
            v[j][2] = buf_ld64(x, o + x2);
          } else if constexpr (O == 0) {
            pair(o + x0, v[j][0], v[j][1]);
            pair(o + x2, v[j][2], v[j][3]);
            v[j][4] = buf_ld64(x, o + x4);
          } else {
            v[j][0] = buf_ld64(x, o + x0);
            pair(o + x1, v[j][1], v[j][2]);
            pair(o + x3, v[j][3], v[j][4]);
          }
        }
#pragma unroll
        for (int j = 0; j < N1; ++j) {
          const double *c = row + (k * N1 + j) * N1;   // entries of row (lz, ly, 0); those of (.., a): c + a ND
          double w[NX];
#pragma unroll
          for (int i = 0; i < NX; ++i) w[i] = in[i] ? v[j][i] : 0.0;
          const double wl = lower ? w[PG] : 0.0, wu = upper ? w[PG] : 0.0;
#pragma unroll
          for (int i = 0; i < PG; ++i) y[0] = __builtin_fma(c[PF * ND + i], w[i], y[0]);
          y[0] = __builtin_fma(c[PF * ND + PG], wl, y[0]);
#pragma unroll
          for (int a = 0; a < PF; ++a) {
            y[a] = __builtin_fma(c[a * ND], wu, y[a]);
#pragma unroll
            for (int i = 1; i < N1; ++i) y[a] = __builtin_fma(c[a * ND + i], w[PG + i], y[a]);
          }
        }
      }
    }
  }
}

// The nodes of a workgroup's thread: false past the segment's part on this XCD.
__device__ __forceinline__ bool mf_thread_nodes(const MfPlan &P, int item, int &si, MfAt &at, int64_t &line) {
  const int xcd = item & 7;
  int j = item >> 3;
  si = 0;
  while (si < P.nseg - 1 && j >= P.seg[si].blocks) j -= P.seg[si++].blocks;
  const MfSeg &s = P.seg[si];
  const MfField &F = P.fld[s.f];
  const int lo = (int)((int64_t)s.rows * xcd / 8), hi = (int)((int64_t)s.rows * (xcd + 1) / 8);
  const int t = lo + j * kMfThreads + (int)threadIdx.x;
  const bool on = t < hi;
  int k = on ? t : lo < s.rows ? lo : 0;
  at.i = s.first[0] + k % s.cnt[0];
  at.g[0] = F.p * at.i;
  k /= s.cnt[0];
  const int b = s.first[1] + F.p * (k % s.cnt[1]), c = s.first[2] + F.p * (k / s.cnt[1]);
  at.g[1] = b + F.o[1];
  at.g[2] = c + F.o[2];
  line = F.base + (int64_t)F.m[0] * (b + (int64_t)F.m[1] * c) - F.o[0] + at.g[0];   // row of the first node, if it has one
  return on;
}

template <int DIM, int PF>
__device__ __forceinline__ double mf_item(const MfPlan &P, const MfSeg &s, const MfAt &at, bool on, int64_t line,
                                          const double *__restrict__ tab, const double *__restrict__ x,
                                          double *__restrict__ q) {
  double y[PF];
#pragma unroll
  for (int a = 0; a < PF; ++a) y[a] = 0.0;
  for (int g = 0; g < P.nf; ++g) {
    const MfField &G = P.fld[g];
    const int t = P.tab[s.f][g];
    if (t < 0 || G.rows == 0) continue;
    const BufRsrc xg = buf_of(x + G.base, 8u * (uint32_t)G.rows);
    if (G.p == 1) mf_rows<DIM, PF, 1, 0>(P, G, s, at, tab + t, xg, y);
    else if (G.o[0] == 0) mf_rows<DIM, PF, 2, 0>(P, G, s, at, tab + t, xg, y);
    else mf_rows<DIM, PF, 2, 1>(P, G, s, at, tab + t, xg, y);
  }
  const MfField &F = P.fld[s.f];
  double acc = 0.0;
#pragma unroll
  for (int a = 0; a < PF; ++a) {
    const int v = at.g[0] + a - F.o[0];
    if (on && v >= 0 && v < F.m[0]) {
      q[line + a] = y[a];
      acc += y[a] * x[line + a];
    }
  }
  return acc;
}

// q = A x from the element tables; partials <q, x> (part).  A workgroup takes 256
// threads' nodes of one segment; each XCD a contiguous eighth of every segment.
// 9 (y, z) lines of a cell, one plane of them in flight, all but the first read
// from the L1 and L2; the element entries are scalar operands.  2 x 27 flops for
// each of a node's 1 to 8 cells, but 8 B a row from memory instead of 12 B an
// entry.  32^3 cells of Q2 and Q1 fields: 48 us for the four blocks' CSR rows, 33
// us with a node a thread (loads of every other value: half of each line), 15 us
// so.
template <int DIM>
__global__ __launch_bounds__(kMfThreads) void k_mf_product(const MfPlan *__restrict__ plan,
                                                           const double *__restrict__ tab,
                                                           const double *__restrict__ x, double *__restrict__ q,
                                                           const CgState *S, double *part) {
  if (S && S->done) return;
  const MfPlan &P = *plan;
  double acc[1] = {0.0};
  for (int item = blockIdx.x; item < P.items; item += gridDim.x) {
    int si;
    MfAt at;
    int64_t line;
    const bool on = mf_thread_nodes(P, item, si, at, line);
    const MfSeg &s = P.seg[si];
    acc[0] += P.fld[s.f].p == 2 ? mf_item<DIM, 2>(P, s, at, on, line, tab, x, q)
                                : mf_item<DIM, 1>(P, s, at, on, line, tab, x, q);
  }
  if (part) group_partials<1>(acc, part);
}

// 1 / diagonal in the boxes' order, a row's cells in ascending order as in the
// assembly; a zero pivot raises the flag
__global__ __launch_bounds__(kMfThreads) void k_mf_invdiag(const MfPlan *__restrict__ plan,
                                                           const double *__restrict__ tab, double *__restrict__ invd,
                                                           int *__restrict__ bad) {
  const MfPlan &P = *plan;
  for (int item = blockIdx.x; item < P.items; item += gridDim.x) {
    int si;
    MfAt at;
    int64_t line;
    if (!mf_thread_nodes(P, item, si, at, line)) continue;
    const MfSeg &s = P.seg[si];
    const MfField &F = P.fld[s.f];
    for (int a = 0; a < F.p; ++a) {
      const int g[3] = {at.g[0] + a, at.g[1], at.g[2]};
      if (g[0] < F.o[0] || g[0] >= F.o[0] + F.m[0]) continue;
      double d = 0.0;
      for (int b = 0; b < (1 << P.dim); ++b) {
        int l = 0, stride = 1;
        bool in = true;
        for (int k = 0; k < P.dim; ++k) {
          const int e = (b >> k) & 1, odd = g[k] % F.p;
          const int c = odd ? g[k] / F.p : g[k] / F.p - 1 + e;
          in = in && !(odd && e) && c >= 0 && c < P.n[k];
          l += stride * (odd ? odd : e ? 0 : F.p);
          stride *= F.p + 1;
        }
        if (in) d += tab[P.tab[s.f][s.f] + l * F.nd + l];
      }
      if (d == 0.0) atomicOr(bad, 1);
      invd[line + a] = 1.0 / d;
    }
  }
}

// A field's part of a block vector between the rows' and the box's order
__global__ void k_mf_to_box(int32_t n, const int32_t *__restrict__ perm, const double *__restrict__ from,
                            double *__restrict__ to) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) to[perm[i]] = from[i];
}
__global__ void k_mf_from_box(int32_t n, const int32_t *__restrict__ perm, const double *__restrict__ from,
                              double *__restrict__ to) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) to[i] = from[perm[i]];
}

// Values of block rows off .. off + rows of field f, kSpmvLanes lanes a row: an
// entry's cells are those that hold both its nodes, at most two a direction,
// found from their grid positions; the element entries are summed in ascending
// order of the cells.  (One wavefront a row that searched each element entry's
// column in the row took 2.5 ms for 32^3 cells of Q2 and Q1 fields, 0.5 ms here.)
__global__ __launch_bounds__(256) void k_mf_assemble(const MfPlan *__restrict__ plan, int f, ColSet cs,
                                                     const int32_t *__restrict__ rowptr,
                                                     const int32_t *__restrict__ col,
                                                     const double *__restrict__ tab, double *__restrict__ val) {
  constexpr int LANES = 16;
  const MfPlan &P = *plan;
  const MfField &F = P.fld[f];
  const int r = (int)(((int64_t)blockIdx.x * 256 + threadIdx.x) / LANES), sub = threadIdx.x % LANES;
  if (r >= F.rows) return;
  const int dim = P.dim;
  auto grid = [&](const MfField &A, int row, int (&gi)[3]) {
    int v = A.perm[row];
    gi[0] = v % A.m[0] + A.o[0];
    v /= A.m[0];
    gi[1] = v % A.m[1] + A.o[1];
    gi[2] = v / A.m[1] + A.o[2];
  };
  int gi[3];
  grid(F, r, gi);
  const int e1 = rowptr[F.off + r + 1];
  for (int e = rowptr[F.off + r] + sub; e < e1; e += LANES) {
    const int c = col[e];
    int k = 0;   // the column's field: the last whose first row is not above it
    for (int j = 1; j < cs.ng; ++j)
      if (c >= cs.off[j] && cs.off[j] >= cs.off[k] && cs.rows[j] > 0) k = j;
    const MfField &G = P.fld[cs.fld[k]];
    int gj[3], c0[3], c1[3];
    grid(G, c - cs.off[k], gj);
    for (int d = 0; d < 3; ++d) {   // cells that hold both nodes along d
      c0[d] = c1[d] = 0;
      if (d < dim) {
        c0[d] = max(max((gi[d] + F.p - 1) / F.p, (gj[d] + G.p - 1) / G.p) - 1, 0);
        c1[d] = min(min(gi[d] / F.p, gj[d] / G.p), P.n[d] - 1);
      }
    }
    double s = 0.0;
    for (int z = c0[2]; z <= c1[2]; ++z)
      for (int y = c0[1]; y <= c1[1]; ++y)
        for (int x = c0[0]; x <= c1[0]; ++x) {
          int l = gi[0] - F.p * x + (F.p + 1) * (gi[1] - F.p * y), m = gj[0] - G.p * x + (G.p + 1) * (gj[1] - G.p * y);
          if (dim == 3) {
            l += (F.p + 1) * (F.p + 1) * (gi[2] - F.p * z);
            m += (G.p + 1) * (G.p + 1) * (gj[2] - G.p * z);
          }
          s += tab[cs.tab[k] + l * G.nd + m];
        }
    val[e] = s;
  }
}

// --------------------------------------------------------------- block CG ---
//
// cg.f90:101-238 in three launches an iteration: the product with <q,p>; x, r
// and <r,z>, ||r||^2; the stopping test, beta and p.  Scalars as in cg.hip: each
// launch reduces the partial sums of the one before, the state alternates by
// parity, launches after the end return at entry.  (One launch for each scalar
// and vector operation took 89 of 137 us an iteration with 32^3 cells.)

constexpr int kMfVecBlocks = 512;

// Sums of a producer's block partials by all waves, in two steps as group_begin
// and group_end: there are hundreds of them.
template <int NV>
__device__ __forceinline__ void partials_begin(const double *part, int g, double (&v)[NV]) {
  for (int k = 0; k < NV; ++k) v[k] = 0.0;
  for (int b = threadIdx.x; b < g; b += kMfThreads)
    for (int k = 0; k < NV; ++k) v[k] += part[k * g + b];
}
template <int NV>
__device__ __forceinline__ void partials_end(double (&v)[NV]) {
  __shared__ double sm[NV][kMfThreads / 64];
  block_sums<kMfThreads / 64, NV>(v, sm);
}

// partials <q, p> of a product that has none
__global__ __launch_bounds__(kMfThreads) void k_mf_dot(int64_t n, const double *__restrict__ a,
                                                       const double *__restrict__ b, const CgState *S, double *part) {
  if (S && S->done) return;
  double acc[1] = {0.0};
  for (int64_t i = (int64_t)blockIdx.x * kMfThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kMfThreads)
    acc[0] += a[i] * b[i];
  group_partials<1>(acc, part);
}

// r = b - q; p = z = M r; partials <r,z>, ||r||^2, ||b||^2
__global__ __launch_bounds__(kMfThreads) void k_mf_start(int64_t n, const double *__restrict__ b,
                                                         const double *__restrict__ q,
                                                         const double *__restrict__ invd, double *__restrict__ r,
                                                         double *__restrict__ p, double *part) {
  double acc[3] = {0.0, 0.0, 0.0};
  for (int64_t i = (int64_t)blockIdx.x * kMfThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kMfThreads) {
    const double bi = b[i], ri = bi - q[i], zi = invd ? invd[i] * ri : ri;
    r[i] = ri;
    p[i] = zi;
    acc[0] += ri * zi;
    acc[1] += ri * ri;
    acc[2] += bi * bi;
  }
  group_partials<3>(acc, part);
}

// first state (RES_RES or RES_RHS, cg.f90:279-321); a zero pivot ends the solve
__global__ __launch_bounds__(kMfThreads) void k_mf_begin(const double *part, int groups, double rtol, double atol,
                                                         int crit, int maxit, const int *bad, CgState *S,
                                                         CgResult *R) {
  double v[3];
  group_reduce<3>(part, groups, v);
  if (threadIdx.x != 0) return;
  CgState s{};
  s.rtol = rtol;
  s.atol = atol;
  s.crit = crit;
  s.maxit = maxit;
  s.rz = v[0];
  s.rnrm_m = sqrt(v[0]);
  s.r0norm = s.rnorm = sqrt(v[1]);
  s.bnorm = sqrt(v[2]);
  s.rhs_test = rtol * (crit == FEMHIP_RES_RHS ? s.bnorm : s.r0norm) + atol;
  s.done = bad && *bad;
  S[0] = S[1] = s;
  CgResult r{};
  r.rhs_test = s.rhs_test;
  r.rnorm = s.rnorm;
  r.bnorm = s.bnorm;
  r.done = s.done;
  *R = r;
}

// alpha; x += alpha p, r -= alpha q; partials <r,z>, ||r||^2
__global__ __launch_bounds__(kMfThreads) void k_mf_update(int64_t n, CgState *S, const double *part_in, int groups,
                                                          const double *__restrict__ invd,
                                                          const double *__restrict__ p,
                                                          const double *__restrict__ q, double *__restrict__ x,
                                                          double *__restrict__ r, double *part) {
  double red[1];
  partials_begin(part_in, groups, red);   // beside the state's load
  if (S->done) return;
  partials_end(red);
  const double alpha = red[0] != 0.0 ? S->rz / red[0] : 0.0;   // cg.f90:195-199
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S->alpha = alpha;
    S->pap = red[0];
  }
  double acc[2] = {0.0, 0.0};
  for (int64_t i = (int64_t)blockIdx.x * kMfThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kMfThreads) {
    x[i] = x[i] + alpha * p[i];
    const double ri = r[i] + (-alpha) * q[i];
    r[i] = ri;
    acc[0] += ri * (invd ? invd[i] * ri : ri);
    acc[1] += ri * ri;
  }
  group_partials<2>(acc, part);
}

// stopping test (cg.f90:323-407), beta; p = z + beta p
__global__ __launch_bounds__(kMfThreads) void k_mf_dir(int64_t n, CgState *S, int par, const double *part_in,
                                                       int groups, const double *__restrict__ invd,
                                                       const double *__restrict__ r, double *__restrict__ p,
                                                       CgResult *R, CgResult *Rh) {
  double red[2], beta;
  partials_begin(part_in, groups, red);
  const CgState &cur = S[par];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (cur.done) {   // keep `done` sticky in both parity slots
    if (lead) {
      S[par ^ 1].done = 1;
      if (Rh) *Rh = *R;
    }
    return;
  }
  partials_end(red);
  if (cg_decide(cur, red, lead, S[par ^ 1], nullptr, R, Rh, beta)) return;
  for (int64_t i = (int64_t)blockIdx.x * kMfThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kMfThreads) {
    const double zi = invd ? invd[i] * r[i] : r[i];
    p[i] = beta * p[i] + zi;
  }
}

// partials ||b - q||^2
__global__ __launch_bounds__(kMfThreads) void k_mf_residual(int64_t n, const double *__restrict__ b,
                                                            const double *__restrict__ q, double *part) {
  double acc[1] = {0.0};
  for (int64_t i = (int64_t)blockIdx.x * kMfThreads + threadIdx.x; i < n; i += (int64_t)gridDim.x * kMfThreads) {
    const double ri = b[i] - q[i];
    acc[0] += ri * ri;
  }
  group_partials<1>(acc, part);
}
__global__ __launch_bounds__(kMfThreads) void k_mf_sum(const double *part, int groups, double *out) {
  double v[1];
  group_reduce<1>(part, groups, v);
  if (threadIdx.x == 0) *out = v[0];
}

// inverse of a diagonal block's diagonal (Jacobi on the block matrix); a
// zero pivot raises the flag
__global__ void k_block_invdiag(int32_t n, const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                                const double *__restrict__ val, double *__restrict__ invd, int *__restrict__ bad) {
  const int32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  double d = 0.0;
  for (int32_t k = rowptr[r]; k < rowptr[r + 1]; ++k)
    if (col[k] == r) d = val[k];
  if (d == 0.0) atomicOr(bad, 1);
  invd[r] = 1.0 / d;
}

unsigned nblocks(int64_t n, int t) { return (unsigned)std::max<int64_t>(1, (n + t - 1) / t); }

}  // namespace

struct femhip_block_operator {
  femhip_ctx *ctx = nullptr;
  int nf = 0, nb = 0;
  femhip_space *field[kMaxFields] = {};
  int block[kMaxFields] = {};               // 0-based block of each field
  int coupling[kMaxFields][kMaxFields] = {};
  int sym_storage = 0;                      // diagonal blocks' symmetric storage (the host view)
  int32_t free_off[kMaxFields] = {};        // first row of each field in its block
  int32_t fixed_off[kMaxFields] = {};       // fixed ids of the earlier fields
  int32_t nblk[kMaxFields] = {};            // rows per block
  int64_t boff[kMaxFields + 1] = {};        // first row of each block in the block vectors
  struct Blk {
    bool on = false;
    DevBuf<int32_t> rowptr, col;
    DevBuf<double> val;
    int64_t nnz = 0, nnz_upper = 0;
  } blk[kMaxFields][kMaxFields];
  RefFE fe[kMaxFields];                      // each field on the common quadrature
  femhip_multifield_physics_t phys{};
  bool have_phys = false, computed = false;
  DevBuf<double> tab, elvec, rhs;
  int32_t tab_off[kMaxFields][kMaxFields] = {}, vec_off[kMaxFields] = {};
  DevBuf<double> x, b, r, p, q, invd, part, part_u, scal;
  DevBuf<CgState> st;
  DevBuf<CgResult> res;
  DevBuf<int> bad;
  CgResult *h_res[2] = {nullptr, nullptr}, *d_res[2] = {nullptr, nullptr};   // pinned, mapped
  hipEvent_t ev[2] = {nullptr, nullptr};
  // products from the element tables
  bool lat = false;
  DevBuf<int32_t> perm[kMaxFields];
  MfPlan h_plan{};
  DevBuf<MfPlan> plan;
  int gp = 1, gv = 1;                        // workgroups of the products and vector kernels
  int64_t ntot = 0;
  ~femhip_block_operator() {
    for (auto *h : h_res)
      if (h) (void)hipHostFree(h);
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
    for (int f = 0; f < nf; ++f)
      if (field[f]) femhip_space_destroy(field[f]);
    if (ctx) ctx_release(ctx);
  }
};

namespace {

// the columns of block jb for rows of field f
ColSet col_set(const femhip_block_operator &B, int f, int jb) {
  ColSet cs{};
  for (int g = 0; g < B.nf; ++g) {
    if (B.block[g] != jb || !B.coupling[f][g]) continue;
    cs.dofs[cs.ng] = B.field[g]->d_dofs.p;
    cs.nd[cs.ng] = B.field[g]->fe.nd;
    cs.off[cs.ng] = B.free_off[g];
    cs.tab[cs.ng] = B.tab_off[f][g];
    cs.fld[cs.ng] = g;
    cs.rows[cs.ng] = B.field[g]->n_free;
    ++cs.ng;
  }
  return cs;
}

void build_block_patterns(femhip_block_operator &B) {
  hipStream_t st = B.ctx->stream;
  for (int ib = 0; ib < B.nb; ++ib)
    for (int jb = 0; jb < B.nb; ++jb) {
      auto &K = B.blk[ib][jb];
      K.on = false;
      for (int f = 0; f < B.nf; ++f)
        for (int g = 0; g < B.nf; ++g) K.on = K.on || (B.block[f] == ib && B.block[g] == jb && B.coupling[f][g]);
      if (!K.on) continue;
      const int32_t n = B.nblk[ib];
      DevBuf<int32_t> len, ulen;
      len.alloc((size_t)n + 1);
      ulen.alloc((size_t)n + 1);
      FH_HIP(hipMemsetAsync(len.p, 0, sizeof(int32_t) * ((size_t)n + 1), st));
      FH_HIP(hipMemsetAsync(ulen.p, 0, sizeof(int32_t) * ((size_t)n + 1), st));
      for (int f = 0; f < B.nf; ++f) {
        if (B.block[f] != ib || B.field[f]->n_free == 0) continue;
        const ColSet cs = col_set(B, f, jb);
        if (cs.ng == 0) continue;
        hipLaunchKernelGGL(k_block_pattern<0>, dim3(nblocks(B.field[f]->n_free, kPatWaves)), dim3(kPatWaves * 64), 0,
                           st, face_tab(*B.field[f]), B.field[f]->n_free, B.free_off[f], B.field[f]->d_rep.p, cs,
                           len.p, ulen.p, nullptr, nullptr);
        FH_HIP(hipGetLastError());
      }
      K.rowptr.alloc((size_t)n + 1);
      K.nnz = exclusive_scan(st, len.p, K.rowptr.p, n, true);
      DevBuf<int32_t> utmp;
      utmp.alloc((size_t)n + 1);
      K.nnz_upper = exclusive_scan(st, ulen.p, utmp.p, n, false);
      K.col.alloc((size_t)std::max<int64_t>(1, K.nnz));
      K.val.alloc((size_t)std::max<int64_t>(1, K.nnz));
      for (int f = 0; f < B.nf; ++f) {
        if (B.block[f] != ib || B.field[f]->n_free == 0) continue;
        const ColSet cs = col_set(B, f, jb);
        if (cs.ng == 0) continue;
        hipLaunchKernelGGL(k_block_pattern<1>, dim3(nblocks(B.field[f]->n_free, kPatWaves)), dim3(kPatWaves * 64), 0,
                           st, face_tab(*B.field[f]), B.field[f]->n_free, B.free_off[f], B.field[f]->d_rep.p, cs,
                           nullptr, nullptr, K.rowptr.p, K.col.p);
        FH_HIP(hipGetLastError());
      }
      FH_HIP(hipStreamSynchronize(st));
    }
}

// Element tables of the coupled diffusion-reaction plugin for every field
// pair (row-major nd_f x nd_g) and element vectors, on the common quadrature,
// in the plugin's loop order (q outermost, then i, then j)
void upload_block_physics(femhip_block_operator &B) {
  const femhip_multifield_physics_t &ph = B.phys;
  std::vector<double> t, v;
  const RefFE &f0 = B.fe[0];
  for (int f = 0; f < B.nf; ++f)
    for (int g = 0; g < B.nf; ++g) {
      B.tab_off[f][g] = (int32_t)t.size();
      t.resize(t.size() + (size_t)B.fe[f].nd * B.fe[g].nd, 0.0);
    }
  for (int f = 0; f < B.nf; ++f) {
    B.vec_off[f] = (int32_t)v.size();
    v.resize(v.size() + (size_t)B.fe[f].nd, 0.0);
  }
  for (int q = 0; q < f0.nq; ++q) {
    const double dv = f0.detj[q] * f0.qw[q];
    for (int f = 0; f < B.nf; ++f) {
      const RefFE &A = B.fe[f];
      for (int i = 0; i < A.nd; ++i) {
        for (int g = 0; g < B.nf; ++g) {
          const RefFE &G = B.fe[g];
          for (int j = 0; j < G.nd; ++j) {
            double e;
            if (f == g) {
              double dot = 0.0;
              for (int k = 0; k < 3; ++k) dot = dot + A.grad[j][k][q] * A.grad[i][k][q];
              e = ph.kappa[f] * dot + (B.nf - 1) * ph.sigma * (A.shp[i][q] * A.shp[j][q]);
            } else {
              e = -ph.sigma * (A.shp[i][q] * G.shp[j][q]);
            }
            t[(size_t)B.tab_off[f][g] + (size_t)i * G.nd + j] += dv * e;
          }
        }
        v[(size_t)B.vec_off[f] + i] += dv * ph.f[f] * A.shp[i][q];
      }
    }
  }
  B.tab.alloc(t.size());
  FH_HIP(hipMemcpy(B.tab.p, t.data(), sizeof(double) * t.size(), hipMemcpyHostToDevice));
  B.elvec.alloc(v.size());
  FH_HIP(hipMemcpy(B.elvec.p, v.data(), sizeof(double) * v.size(), hipMemcpyHostToDevice));
}

void block_compute(femhip_block_operator &B, double *ms) {
  hipStream_t st = B.ctx->stream;
  hipEvent_t e0, e1;
  FH_HIP(hipEventCreate(&e0));
  FH_HIP(hipEventCreate(&e1));
  FH_HIP(hipEventRecord(e0, st));
  for (int ib = 0; ib < B.nb; ++ib)
    for (int jb = 0; jb < B.nb; ++jb) {
      auto &K = B.blk[ib][jb];
      if (!K.on) continue;
      for (int f = 0; f < B.nf; ++f) {
        if (B.block[f] != ib || B.field[f]->n_free == 0) continue;
        const ColSet cs = col_set(B, f, jb);
        if (cs.ng == 0) continue;
        if (B.lat)
          hipLaunchKernelGGL(k_mf_assemble, dim3(nblocks((int64_t)B.field[f]->n_free * 16, 256)), dim3(256), 0, st,
                             B.plan.p, f, cs, K.rowptr.p, K.col.p, B.tab.p, K.val.p);
        else
          hipLaunchKernelGGL(k_block_assemble, dim3((unsigned)B.field[f]->n_free), dim3(64), 0, st,
                             face_tab(*B.field[f]), B.field[f]->n_free, B.free_off[f], B.field[f]->d_rep.p, cs,
                             K.rowptr.p, K.col.p, B.tab.p, K.val.p);
        FH_HIP(hipGetLastError());
      }
    }
  for (int f = 0; f < B.nf; ++f) {
    if (B.field[f]->n_free == 0) continue;
    const int ib = B.block[f];
    hipLaunchKernelGGL(k_block_rhs, dim3(nblocks(B.field[f]->n_free, 256)), dim3(256), 0, st, face_tab(*B.field[f]),
                       B.field[f]->n_free, B.free_off[f], B.field[f]->d_rep.p, B.elvec.p + B.vec_off[f],
                       B.rhs.p + B.boff[ib]);
    FH_HIP(hipGetLastError());
  }
  FH_HIP(hipEventRecord(e1, st));
  FH_HIP(hipEventSynchronize(e1));
  float t = 0.f;
  FH_HIP(hipEventElapsedTime(&t, e0, e1));
  if (ms) *ms = t;
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
}

// y = A x over the block vectors (device pointers)
void block_apply(femhip_block_operator &B, const double *x, double *y, const CgState *stop = nullptr) {
  hipStream_t st = B.ctx->stream;
  for (int ib = 0; ib < B.nb; ++ib) {
    int first = 1;
    const int32_t n = B.nblk[ib];
    if (n == 0) continue;
    for (int jb = 0; jb < B.nb; ++jb) {
      auto &K = B.blk[ib][jb];
      if (!K.on) continue;
      hipLaunchKernelGGL(k_block_spmv<kSpmvLanes>, dim3(nblocks((int64_t)n * kSpmvLanes, kSpmvThreads)),
                         dim3(kSpmvThreads), 0, st, n, K.rowptr.p, K.col.p, K.val.p, x + B.boff[jb], y + B.boff[ib],
                         first ? 0 : 1, stop);
      FH_HIP(hipGetLastError());
      first = 0;
    }
    if (first) FH_HIP(hipMemsetAsync(y + B.boff[ib], 0, sizeof(double) * (size_t)n, st));
  }
}

// Boxes of the fields and the segments of the products; B.lat stays false
// where a field's rows are no box.
void plan_products(femhip_block_operator &B) {
  MfPlan &P = B.h_plan;
  const femhip_mesh_desc_t &m = B.field[0]->mesh;
  P.nf = B.nf;
  P.dim = m.dim;
  for (int d = 0; d < 3; ++d) P.n[d] = d < m.dim ? m.n[d] : 1;
  for (int f = 0; f < B.nf; ++f) {
    const femhip_space &s = *B.field[f];
    MfField &F = P.fld[f];
    F.p = s.fe.order;
    F.nd = s.fe.nd;
    F.rows = s.n_free;
    F.off = B.free_off[f];
    F.base = B.boff[B.block[f]] + B.free_off[f];
    for (int d = 0; d < 3; ++d) F.m[d] = 1;
    if (s.n_free == 0) continue;
    LatticeOp L;
    if (s.fe.order > 2 || s.n_free > kLatticeMaxRows - 64 || !lattice_plan(s.mesh, B.ctx->num_cus, L) ||
        !lattice_rows(s, L, B.perm[f]))
      return;
    for (int d = 0; d < m.dim; ++d) {
      F.o[d] = L.g.o[d];
      F.m[d] = L.g.m[d];
    }
    F.perm = B.perm[f].p;
    for (int c = 0; c < (F.p == 2 ? 1 << (m.dim - 1) : 1); ++c) {   // bit d - 1: odd along d
      MfSeg S{};
      S.f = f;
      for (int d = 0; d < 3; ++d) S.aligned[d] = S.cnt[d] = 1;
      // along x a thread per cell vertex: the first may only have nodes after it
      S.first[0] = F.p == 1 ? F.o[0] : 0;
      S.cnt[0] = F.p == 1 ? F.m[0] : P.n[0] + (F.o[0] + F.m[0] > 2 * P.n[0] ? 1 : 0);
      int64_t rows = S.cnt[0];
      for (int d = 1; d < m.dim; ++d) {
        const int odd = (c >> (d - 1)) & 1;
        S.aligned[d] = !odd;
        S.first[d] = F.p == 1 ? 0 : ((odd - F.o[d]) % 2 + 2) % 2;
        S.cnt[d] = F.m[d] > S.first[d] ? (F.m[d] - S.first[d] + F.p - 1) / F.p : 0;
        rows *= S.cnt[d];
      }
      S.rows = (int)rows;
      if (S.rows == 0) continue;
      S.blocks = (int)(((rows + 7) / 8 + kMfThreads - 1) / kMfThreads);
      P.items += 8 * S.blocks;
      P.seg[P.nseg++] = S;
    }
  }
  if (P.nseg == 0) return;
  auto cells = [](const MfSeg &s) { return s.aligned[0] + s.aligned[1] + s.aligned[2]; };
  std::stable_sort(P.seg, P.seg + P.nseg, [&](const MfSeg &a, const MfSeg &b) { return cells(a) > cells(b); });
  B.plan.alloc(1);
  B.lat = true;
}

// the plan with the element tables' places (after set_physics)
void upload_plan(femhip_block_operator &B) {
  if (!B.lat) return;
  for (int f = 0; f < B.nf; ++f)
    for (int g = 0; g < B.nf; ++g) B.h_plan.tab[f][g] = B.coupling[f][g] ? B.tab_off[f][g] : -1;
  FH_HIP(hipMemcpy(B.plan.p, &B.h_plan, sizeof(MfPlan), hipMemcpyHostToDevice));
}

// q = A x in the solver's order with partials <q, x>
void solver_apply(femhip_block_operator &B, const double *x, double *q, const CgState *stop, double *part) {
  hipStream_t st = B.ctx->stream;
  const dim3 T(kMfThreads);
  if (!B.lat) {
    block_apply(B, x, q, stop);
    if (part) hipLaunchKernelGGL(k_mf_dot, dim3(B.gp), T, 0, st, B.ntot, q, x, stop, part);
  } else if (B.h_plan.dim == 3) {
    hipLaunchKernelGGL(k_mf_product<3>, dim3(B.gp), T, 0, st, B.plan.p, B.tab.p, x, q, stop, part);
  } else {
    hipLaunchKernelGGL(k_mf_product<2>, dim3(B.gp), T, 0, st, B.plan.p, B.tab.p, x, q, stop, part);
  }
  FH_HIP(hipGetLastError());
}

// A block vector into the solver's order, and back.
void to_solver(femhip_block_operator &B, const double *from, double *to) {
  hipStream_t st = B.ctx->stream;
  if (!B.lat) {
    FH_HIP(hipMemcpyAsync(to, from, sizeof(double) * (size_t)B.ntot, hipMemcpyDeviceToDevice, st));
    return;
  }
  for (int f = 0; f < B.nf; ++f) {
    const MfField &F = B.h_plan.fld[f];
    if (F.rows)
      hipLaunchKernelGGL(k_mf_to_box, dim3(nblocks(F.rows, 256)), dim3(256), 0, st, F.rows, F.perm, from + F.base,
                         to + F.base);
  }
  FH_HIP(hipGetLastError());
}
void from_solver(femhip_block_operator &B, const double *from, double *to) {
  hipStream_t st = B.ctx->stream;
  if (!B.lat) {
    FH_HIP(hipMemcpyAsync(to, from, sizeof(double) * (size_t)B.ntot, hipMemcpyDeviceToDevice, st));
    return;
  }
  for (int f = 0; f < B.nf; ++f) {
    const MfField &F = B.h_plan.fld[f];
    if (F.rows)
      hipLaunchKernelGGL(k_mf_from_box, dim3(nblocks(F.rows, 256)), dim3(256), 0, st, F.rows, F.perm, from + F.base,
                         to + F.base);
  }
  FH_HIP(hipGetLastError());
}

constexpr int kBlockChunk = 8;   // iterations queued at a time (even: the parity restarts at 0)

// cg_solve_body (cg.f90:101-238) on the block operator with the RES_RES or
// RES_RHS criterion (cg.f90:279-407), identity or Jacobi (the inverse
// diagonals of the diagonal blocks) preconditioner; q holds x0 and p the
// right-hand side in block order, r the solution on return
void block_cg(femhip_block_operator &B, const femhip_cg_params_t &prm, femhip_cg_result_t &res) {
  hipStream_t st = B.ctx->stream;
  const int64_t n = B.ntot;
  const dim3 G((unsigned)B.gv), T(kMfThreads);
  const bool jac = prm.preconditioner == FEMHIP_PREC_JACOBI;
  hipEvent_t e0, e1;
  FH_HIP(hipEventCreate(&e0));
  FH_HIP(hipEventCreate(&e1));
  FH_HIP(hipEventRecord(e0, st));
  if (jac) {
    FH_HIP(hipMemsetAsync(B.bad.p, 0, sizeof(int), st));
    for (int ib = 0; ib < B.nb; ++ib)
      FH_CHECK(B.nblk[ib] == 0 || B.blk[ib][ib].on, FEMHIP_ERR_ZERO_DIAGONAL, "diagonal block missing: Jacobi needs it");
    if (B.lat) {
      hipLaunchKernelGGL(k_mf_invdiag, dim3((unsigned)B.gp), T, 0, st, B.plan.p, B.tab.p, B.invd.p, B.bad.p);
    } else {
      for (int ib = 0; ib < B.nb; ++ib)
        if (B.nblk[ib] > 0)
          hipLaunchKernelGGL(k_block_invdiag, dim3(nblocks(B.nblk[ib], 256)), T, 0, st, B.nblk[ib],
                             B.blk[ib][ib].rowptr.p, B.blk[ib][ib].col.p, B.blk[ib][ib].val.p,
                             B.invd.p + B.boff[ib], B.bad.p);
    }
    FH_HIP(hipGetLastError());
  }
  const double *invd = jac ? B.invd.p : nullptr;
  to_solver(B, B.q.p, B.x.p);
  to_solver(B, B.p.p, B.b.p);
  solver_apply(B, B.x.p, B.q.p, nullptr, nullptr);
  hipLaunchKernelGGL(k_mf_start, G, T, 0, st, n, B.b.p, B.q.p, invd, B.r.p, B.p.p, B.part_u.p);
  hipLaunchKernelGGL(k_mf_begin, dim3(1), T, 0, st, B.part_u.p, B.gv, prm.rtol, prm.atol, prm.stopping_criterion,
                     prm.max_num_iterations, jac ? B.bad.p : nullptr, B.st.p, B.res.p);
  FH_HIP(hipGetLastError());
  // chunks, one ahead; the launches of iterations past the end return at entry
  int64_t queued = 0;
  auto push = [&](int slot) {
    for (int c = 0; c < kBlockChunk; ++c) {
      const int par = c & 1;
      solver_apply(B, B.p.p, B.q.p, B.st.p + par, B.part.p);
      hipLaunchKernelGGL(k_mf_update, G, T, 0, st, n, B.st.p + par, B.part.p, B.gp, invd, B.p.p, B.q.p, B.x.p, B.r.p,
                         B.part_u.p);
      hipLaunchKernelGGL(k_mf_dir, G, T, 0, st, n, B.st.p, par, B.part_u.p, B.gv, invd, B.r.p, B.p.p, B.res.p,
                         c == kBlockChunk - 1 ? B.d_res[slot] : nullptr);
      FH_HIP(hipGetLastError());
    }
    FH_HIP(hipEventRecord(B.ev[slot], st));
    queued += kBlockChunk;
  };
  push(0);
  bool more = queued < prm.max_num_iterations;
  if (more) push(1);
  for (int slot = 0;; slot ^= 1) {
    FH_HIP(hipEventSynchronize(B.ev[slot]));
    if (B.h_res[slot]->done || !more) break;
    more = queued < prm.max_num_iterations;
    if (more) push(slot);
  }
  FH_HIP(hipEventRecord(e1, st));
  // true residual in FP64
  solver_apply(B, B.x.p, B.q.p, nullptr, nullptr);
  hipLaunchKernelGGL(k_mf_residual, G, T, 0, st, n, B.b.p, B.q.p, B.part_u.p);
  hipLaunchKernelGGL(k_mf_sum, dim3(1), T, 0, st, B.part_u.p, B.gv, B.scal.p);
  from_solver(B, B.x.p, B.r.p);
  FH_HIP(hipGetLastError());
  CgResult r;
  double rr = 0.0;
  int bad = 0;
  FH_HIP(hipMemcpyAsync(&r, B.res.p, sizeof(r), hipMemcpyDeviceToHost, st));
  FH_HIP(hipMemcpyAsync(&rr, B.scal.p, sizeof(rr), hipMemcpyDeviceToHost, st));
  if (jac) FH_HIP(hipMemcpyAsync(&bad, B.bad.p, sizeof(bad), hipMemcpyDeviceToHost, st));
  FH_HIP(hipStreamSynchronize(st));
  float t = 0.f;
  FH_HIP(hipEventElapsedTime(&t, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  FH_CHECK(!bad, FEMHIP_ERR_ZERO_DIAGONAL, "op1 cannot be entrywise inverted; there exists a null diagonal entry");
  res.true_residual = std::sqrt(rr);
  res.rhs_norm = r.bnorm;
  res.num_iterations = r.iter;
  res.did_converge = r.converged ? 1 : 0;
  res.outer_iterations = 0;
  res.status = r.converged ? FEMHIP_OK : FEMHIP_ERR_NOT_CONVERGED;
  res.error_estimate = r.est;
  res.rhs_convergence_test = r.rhs_test;
  res.solve_ms = t;
}

void check_block(const femhip_block_operator *B, int32_t ib, int32_t jb) {
  FH_CHECK(B, FEMHIP_ERR_INVALID, "null block operator");
  FH_CHECK(ib >= 1 && ib <= B->nb && jb >= 1 && jb <= B->nb, FEMHIP_ERR_INVALID, "block index out of range");
}

}  // namespace

extern "C" {

int femhip_block_operator_create(femhip_ctx_t *ctx, const femhip_block_layout_t *layout,
                                 int32_t diagonal_blocks_symmetric_storage, femhip_block_operator_t **bop) {
  try {
    FH_CHECK(ctx && layout && bop, FEMHIP_ERR_INVALID, "null argument");
    const int nf = layout->num_fields;
    FH_CHECK(nf >= 1 && nf <= kMaxFields, FEMHIP_ERR_INVALID, "num_fields must be in [1, 4]");
    int maxo = 0;
    for (int f = 0; f < nf; ++f) {
      const femhip_space *s = layout->fields[f];
      FH_CHECK(s, FEMHIP_ERR_INVALID, "null field space");
      FH_CHECK(s->ctx == ctx, FEMHIP_ERR_INVALID, "field spaces must belong to the context");
      FH_CHECK(s->fe.ncomp == 1, FEMHIP_ERR_INVALID, "block operator fields must be scalar");
      const femhip_mesh_desc_t &a = s->mesh, &b = layout->fields[0]->mesh;
      bool same = a.dim == b.dim;
      for (int k = 0; k < 3; ++k) same = same && a.n[k] == b.n[k];
      for (int k = 0; k < 6; ++k) same = same && a.limits[k] == b.limits[k];
      FH_CHECK(same, FEMHIP_ERR_INVALID, "all fields must live on the same mesh");
      FH_CHECK(layout->field_blocks[f] >= 1 && layout->field_blocks[f] <= nf, FEMHIP_ERR_INVALID,
               "field_blocks entries must be in [1, num_fields]");
      FH_CHECK(layout->field_coupling[f * nf + f] != 0, FEMHIP_ERR_INVALID, "every field must couple to itself");
      maxo = std::max(maxo, s->fe.order);
    }
    FH_HIP(hipSetDevice(ctx->device));
    auto *B = new femhip_block_operator();
    try {
      B->ctx = ctx_retain(ctx);
      B->nf = nf;
      B->sym_storage = diagonal_blocks_symmetric_storage ? 1 : 0;
      for (int f = 0; f < nf; ++f) {
        B->field[f] = layout->fields[f];
        B->field[f]->refs.fetch_add(1);
        B->block[f] = layout->field_blocks[f] - 1;
        B->nb = std::max(B->nb, B->block[f] + 1);
        for (int g = 0; g < nf; ++g) B->coupling[f][g] = layout->field_coupling[f * nf + g] != 0;
      }
      // block_layout_t%create: block coupling of coupled fields; offsets in field order
      int32_t fixed = 0;
      for (int f = 0; f < nf; ++f) {
        B->free_off[f] = B->nblk[B->block[f]];
        int64_t nb = (int64_t)B->nblk[B->block[f]] + B->field[f]->n_free;
        FH_CHECK(nb < INT32_MAX, FEMHIP_ERR_INVALID, "block too large for 32-bit ids");
        B->nblk[B->block[f]] = (int32_t)nb;
        B->fixed_off[f] = fixed;
        fixed += B->field[f]->n_fixed;
      }
      for (int b = 0; b < B->nb; ++b) {
        FH_CHECK(B->nblk[b] >= 0, FEMHIP_ERR_INVALID, "bad block");
        B->boff[b + 1] = B->boff[b] + B->nblk[b];
      }
      B->ntot = B->boff[B->nb];
      // every field on the quadrature of the highest order (sbm_serial_fe_space.i90:1891-2006)
      const femhip_mesh_desc_t &m = B->field[0]->mesh;
      double h[3] = {1.0, 1.0, 1.0};
      for (int k = 0; k < m.dim; ++k) {
        const double a = m.limits[2 * k], b = m.limits[2 * k + 1];
        h[k] = ((b - a) * (1.0 / (double)m.n[k]) + a) - a;
      }
      for (int f = 0; f < nf; ++f) build_reffe(B->fe[f], m.dim, B->field[f]->fe.order, 1, h, maxo + 1);
      build_block_patterns(*B);
      const size_t nt = (size_t)std::max<int64_t>(1, B->ntot);
      for (auto *v : {&B->rhs, &B->x, &B->b, &B->r, &B->p, &B->q, &B->invd}) v->alloc(nt);
      plan_products(*B);
      const int64_t rows = B->lat ? (int64_t)B->h_plan.items * kMfThreads : B->ntot;
      B->gp = (int)std::min<int64_t>(B->lat ? 2048 : kMfVecBlocks, nblocks(rows, kMfThreads));
      B->gv = (int)std::min<int64_t>(kMfVecBlocks, nblocks(B->ntot, kMfThreads));
      B->part.alloc((size_t)B->gp);
      B->part_u.alloc((size_t)3 * B->gv);
      B->scal.alloc(1);
      B->st.alloc(2);
      B->res.alloc(1);
      B->bad.alloc(1);
      for (int k = 0; k < 2; ++k) {   // written by the GPU, read by the host: mapped, coherent
        FH_HIP(hipHostMalloc((void **)&B->h_res[k], sizeof(CgResult), hipHostMallocMapped | hipHostMallocCoherent));
        FH_HIP(hipHostGetDevicePointer((void **)&B->d_res[k], B->h_res[k], 0));
        FH_HIP(hipEventCreateWithFlags(&B->ev[k], hipEventDisableTiming));
      }
    } catch (...) {
      delete B;
      throw;
    }
    *bop = B;
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  } catch (const std::bad_alloc &) {
    set_error("host allocation failed");
    return FEMHIP_ERR_OOM;
  }
}

int femhip_block_operator_info(const femhip_block_operator_t *B, int32_t *num_blocks, int32_t *block_sizes,
                               int64_t *nnz) {
  try {
    FH_CHECK(B && num_blocks, FEMHIP_ERR_INVALID, "null argument");
    *num_blocks = B->nb;
    for (int ib = 0; ib < B->nb; ++ib) {
      if (block_sizes) block_sizes[ib] = B->nblk[ib];
      for (int jb = 0; jb < B->nb; ++jb) {
        const auto &K = B->blk[ib][jb];
        if (nnz) nnz[ib * B->nb + jb] = !K.on ? 0 : (B->sym_storage && ib == jb ? K.nnz_upper : K.nnz);
      }
    }
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_get_dofs(const femhip_block_operator_t *B, int32_t field, int32_t *lst_dofs_gids) {
  try {
    FH_CHECK(B && lst_dofs_gids, FEMHIP_ERR_INVALID, "null argument");
    FH_CHECK(field >= 1 && field <= B->nf, FEMHIP_ERR_INVALID, "field index out of range");
    const femhip_space &s = *B->field[field - 1];
    ensure_host_dofs(s);
    const int32_t fo = B->free_off[field - 1], xo = B->fixed_off[field - 1];
    for (size_t i = 0; i < s.dofs.size(); ++i) {
      const int32_t g = s.dofs[i];
      lst_dofs_gids[i] = g > 0 ? g + fo : g - xo;
    }
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_get_block_pattern(const femhip_block_operator_t *B, int32_t ib, int32_t jb, int32_t *irp,
                                            int32_t *ja) {
  try {
    check_block(B, ib, jb);
    FH_CHECK(irp && ja, FEMHIP_ERR_INVALID, "null argument");
    const auto &K = B->blk[ib - 1][jb - 1];
    const int32_t n = B->nblk[ib - 1];
    if (!K.on) {
      for (int32_t r = 0; r <= n; ++r) irp[r] = 1;
      return FEMHIP_OK;
    }
    FH_HIP(hipSetDevice(B->ctx->device));
    std::vector<int32_t> rp((size_t)n + 1), cl((size_t)std::max<int64_t>(1, K.nnz));
    FH_HIP(hipMemcpy(rp.data(), K.rowptr.p, sizeof(int32_t) * rp.size(), hipMemcpyDeviceToHost));
    FH_HIP(hipMemcpy(cl.data(), K.col.p, sizeof(int32_t) * (size_t)K.nnz, hipMemcpyDeviceToHost));
    const bool up = B->sym_storage && ib == jb;
    int64_t k = 0;
    irp[0] = 1;
    for (int32_t r = 0; r < n; ++r) {
      for (int32_t e = rp[r]; e < rp[r + 1]; ++e)
        if (!up || cl[e] >= r) ja[k++] = cl[e] + 1;
      irp[r + 1] = (int32_t)(k + 1);
    }
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_set_physics(femhip_block_operator_t *B, const femhip_multifield_physics_t *ph) {
  try {
    FH_CHECK(B && ph, FEMHIP_ERR_INVALID, "null argument");
    FH_CHECK(ph->sigma >= 0.0, FEMHIP_ERR_INVALID, "sigma must be >= 0");
    FH_HIP(hipSetDevice(B->ctx->device));
    B->phys = *ph;
    upload_block_physics(*B);
    upload_plan(*B);
    B->have_phys = true;
    B->computed = false;
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_compute(femhip_block_operator_t *B, double *ms) {
  try {
    FH_CHECK(B, FEMHIP_ERR_INVALID, "null block operator");
    FH_CHECK(B->have_phys, FEMHIP_ERR_STATE, "set the physics before compute");
    FH_HIP(hipSetDevice(B->ctx->device));
    block_compute(*B, ms);
    B->computed = true;
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_get_block_values(const femhip_block_operator_t *B, int32_t ib, int32_t jb, double *val) {
  try {
    check_block(B, ib, jb);
    FH_CHECK(val, FEMHIP_ERR_INVALID, "null argument");
    FH_CHECK(B->computed, FEMHIP_ERR_STATE, "block operator not computed");
    const auto &K = B->blk[ib - 1][jb - 1];
    if (!K.on) return FEMHIP_OK;
    FH_HIP(hipSetDevice(B->ctx->device));
    const int32_t n = B->nblk[ib - 1];
    std::vector<int32_t> rp((size_t)n + 1), cl((size_t)std::max<int64_t>(1, K.nnz));
    std::vector<double> v((size_t)std::max<int64_t>(1, K.nnz));
    FH_HIP(hipMemcpy(rp.data(), K.rowptr.p, sizeof(int32_t) * rp.size(), hipMemcpyDeviceToHost));
    FH_HIP(hipMemcpy(cl.data(), K.col.p, sizeof(int32_t) * (size_t)K.nnz, hipMemcpyDeviceToHost));
    FH_HIP(hipMemcpy(v.data(), K.val.p, sizeof(double) * (size_t)K.nnz, hipMemcpyDeviceToHost));
    const bool up = B->sym_storage && ib == jb;
    int64_t k = 0;
    for (int32_t r = 0; r < n; ++r)
      for (int32_t e = rp[r]; e < rp[r + 1]; ++e)
        if (!up || cl[e] >= r) val[k++] = v[e];
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_get_rhs(const femhip_block_operator_t *B, int32_t ib, double *rhs) {
  try {
    check_block(B, ib, ib);
    FH_CHECK(rhs, FEMHIP_ERR_INVALID, "null argument");
    FH_CHECK(B->computed, FEMHIP_ERR_STATE, "block operator not computed");
    FH_HIP(hipSetDevice(B->ctx->device));
    if (B->nblk[ib - 1] > 0)
      FH_HIP(hipMemcpy(rhs, B->rhs.p + B->boff[ib - 1], sizeof(double) * (size_t)B->nblk[ib - 1],
                       hipMemcpyDeviceToHost));
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_apply(femhip_block_operator_t *B, const double *x, double *y) {
  try {
    FH_CHECK(B && x && y, FEMHIP_ERR_INVALID, "null argument");
    FH_CHECK(B->computed, FEMHIP_ERR_STATE, "block operator not computed");
    FH_HIP(hipSetDevice(B->ctx->device));
    if (B->ntot == 0) return FEMHIP_OK;
    const size_t bytes = sizeof(double) * (size_t)B->ntot;
    hipStream_t st = B->ctx->stream;
    FH_HIP(hipMemcpyAsync(B->p.p, x, bytes, hipMemcpyHostToDevice, st));
    block_apply(*B, B->p.p, B->q.p);
    FH_HIP(hipMemcpyAsync(y, B->q.p, bytes, hipMemcpyDeviceToHost, st));
    FH_HIP(hipStreamSynchronize(st));
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_solve(femhip_block_operator_t *B, const femhip_cg_params_t *prm, const double *b,
                                double *x, femhip_cg_result_t *res) {
  try {
    FH_CHECK(B && prm && x && res, FEMHIP_ERR_INVALID, "null argument");
    FH_CHECK(B->computed, FEMHIP_ERR_STATE, "block operator not computed");
    FH_CHECK(prm->precision == FEMHIP_PRECISION_FP64, FEMHIP_ERR_INVALID, "the block solver runs in FP64");
    FH_CHECK(prm->stopping_criterion == FEMHIP_RES_RES || prm->stopping_criterion == FEMHIP_RES_RHS,
             FEMHIP_ERR_INVALID, "the block solver supports the RES_RES and RES_RHS criteria");
    FH_CHECK(prm->preconditioner == FEMHIP_PREC_IDENTITY || prm->preconditioner == FEMHIP_PREC_JACOBI,
             FEMHIP_ERR_INVALID, "unknown preconditioner");
    FH_CHECK(prm->max_num_iterations >= 1 && prm->rtol >= 0 && prm->atol >= 0, FEMHIP_ERR_INVALID,
             "bad solver parameters");
    FH_HIP(hipSetDevice(B->ctx->device));
    *res = femhip_cg_result_t{};
    if (B->ntot == 0) {
      res->did_converge = 1;
      return FEMHIP_OK;
    }
    const size_t bytes = sizeof(double) * (size_t)B->ntot;
    hipStream_t st = B->ctx->stream;
    if (b) FH_HIP(hipMemcpyAsync(B->p.p, b, bytes, hipMemcpyHostToDevice, st));
    else FH_HIP(hipMemcpyAsync(B->p.p, B->rhs.p, bytes, hipMemcpyDeviceToDevice, st));
    FH_HIP(hipMemcpyAsync(B->q.p, x, bytes, hipMemcpyHostToDevice, st));
    block_cg(*B, *prm, *res);
    FH_HIP(hipMemcpyAsync(x, B->r.p, bytes, hipMemcpyDeviceToHost, st));
    FH_HIP(hipStreamSynchronize(st));
    return FEMHIP_OK;
  } catch (const Error &e) {
    set_error(e.msg);
    return e.code;
  }
}

int femhip_block_operator_destroy(femhip_block_operator_t *B) {
  if (!B) return FEMHIP_OK;
  (void)hipSetDevice(B->ctx->device);
  (void)hipStreamSynchronize(B->ctx->stream);
  delete B;
  return FEMHIP_OK;
}

}  // extern "C"
