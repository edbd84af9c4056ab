// lattice.hip -- set-up of the matrix-free products (lattice.h): which
// operators they apply to, the map between the operator's rows and the box
// lattice, the split into workgroups, the coefficient tables.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "femhip_internal.h"
#include "lattice.h"

namespace femhip {
namespace {

// grid node (lexicographic position in the box, or -1) of local node l of cell ijk
__device__ __forceinline__ int box_node(const Lattice &g, int dim, int p, const int (&ijk)[3], int l) {
  int idx = 0, stride = 1;
  for (int d = 0; d < dim; ++d) {
    const int a = p * ijk[d] + l % (p + 1) - g.o[d];
    l /= p + 1;
    if (a < 0 || a >= g.m[d]) return -1;
    idx += stride * a;
    stride *= g.m[d];
  }
  return idx;
}

// perm[row] = lattice row, from the row's representative (cell, local DOF)
__global__ void k_lattice_perm(Lattice g, FaceTab t, int32_t n, const int64_t *__restrict__ rep,
                               int32_t *__restrict__ perm, int *__restrict__ bad) {
  const int32_t r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= n) return;
  const int64_t c0 = rep[r];
  int ijk[3];
  cell_ijk(t, c0 / t.nd, ijk);
  const int l = (int)(c0 % t.nd), comp = l / t.nnode;
  const int v = box_node(g, t.dim, t.order, ijk, l % t.nnode);
  const int row = v < 0 ? -1 : comp * g.stride + v;
  perm[r] = row < 0 ? 0 : row;
  int f = row < 0 ? 1 : 0;
  if (row != r) f |= 2;   // not the identity
  if (f) atomicOr(bad, f);
}

// every (cell, local DOF) must be the row its lattice node has, and fixed exactly outside the box
__global__ void k_lattice_check(Lattice g, FaceTab t, int64_t ncells, int32_t n, const int32_t *__restrict__ dofs,
                                const int32_t *__restrict__ perm, int *__restrict__ bad) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ncells * t.nd) return;
  int ijk[3];
  cell_ijk(t, i / t.nd, ijk);
  const int l = (int)(i % t.nd), comp = l / t.nnode;
  const int v = box_node(g, t.dim, t.order, ijk, l % t.nnode);
  const int32_t id = dofs[i];
  const bool ok = v < 0 ? id < 0 : id >= 0 && id < n && perm[id] == comp * g.stride + v;
  if (!ok) atomicOr(bad, 1);
}

// point values [cell][q] -> [q][cell], so the lanes of a wave read one run
__global__ void k_points_by_q(int64_t cells, int nq, const double *__restrict__ in, double *__restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < cells * nq) out[(i % nq) * cells + i / nq] = in[i];
}

// False where no tile fits max_threads: no default split would cover the box.
template <int DIM, int P, int NC = 1>
bool split(LatticeOp &L, int cus, int max_threads, int cells) {
  Lattice &g = L.g;
  const int e0 = g.E[0], e1 = DIM == 3 ? g.E[1] : 1, ez = g.E[DIM - 1];
  // Tile: the least lanes over all tiles.  Neighbouring tiles both compute the
  // row of cells between them, so larger tiles repeat less; TX needs no
  // alignment, the lanes run through the tile row by row.
  double best = 1e300;
  for (int xt = 1; xt <= e0; ++xt) {
    const int TX = (e0 - 1 + xt - 1) / xt + 1;
    if (TX > max_threads) continue;
    // A thread loads one halo node: narrow tiles (Q2, one or two cells along x) are
    // cut short along y by their halo before the threads run out.
    int TY = std::min(max_threads / TX, e1);
    if (DIM == 3) TY = std::min(TY, (max_threads - 1) / P - TX);
    if (TY < std::min(e1, 2)) continue;
    const int yt = e1 > 1 ? (e1 - 1 + TY - 2) / (TY - 1) : 1;
    if (e1 > 1) TY = (e1 - 1 + yt - 1) / yt + 1;
    const int lanes = std::max(TX * TY, lattice_halo<DIM, P>(TX, TY));
    if (lanes > max_threads) continue;
    const int waves = (lanes + 63) / 64;
    const double cost = (double)xt * yt * waves * (1.0 + 0.02 * xt);
    if (cost < best) {
      best = cost;
      g.TX = TX;
      g.TY = TY;
      g.xt = xt;
      g.tiles = xt * yt;
      L.threads = waves * 64;
    }
    if (TX <= 2) break;
  }
  if (best == 1e300) return false;
  L.lds = lattice_lds<DIM, P, NC>(g.TX, g.TY) * sizeof(double);
  // Chunks of the march: each repeats one layer, so few long ones repeat
  // little and many short ones fill the chip; the fewest layers in turn on one
  // CU wins.
  if (cus <= 0) {
    // the planes a chunk reads stay within 30-bit byte offsets (lattice_window)
    const int64_t plane = (int64_t)g.m[0] * (DIM == 3 ? g.m[1] : 1);
    const int64_t most = (kLatticeMaxRows / plane - 1) / P - 1;
    if (most < 1) return false;
    const int layers = (int)std::min<int64_t>(most, std::max(2, std::min(ez, cells / std::max(1, g.TX * g.TY))));
    g.nch = (ez + layers - 1) / layers;
    L.grid = g.tiles * g.nch;
    return true;
  }
  // One launch an iteration: at most one workgroup a CU, also where more would
  // fit (elasticity of 40 x 33 x 47 cells: 16.6 us with 288 of one layer, 15.2 with
  // 144 of two).
  const int fit = std::max(1, std::min(256 * lattice_waves(DIM, P, NC, L.one) / L.threads, (int)(160 * 1024 / std::max<size_t>(1, L.lds))));
  const int per_cu = L.one ? 1 : fit;
  const int64_t slots = (int64_t)per_cu * std::max(1, cus);
  double bestc = 1e300;
  for (int c = 1; c <= ez; ++c) {
    const int64_t blocks = (int64_t)g.tiles * c;
    if (blocks > 4096 && c > 1) break;
    const double layers = std::ceil((double)ez / c) + (c > 1 ? 1.0 : 0.0) + 0.5;
    const double cost = (double)((blocks + slots - 1) / slots) * layers;
    if (cost < bestc * 0.999) {
      bestc = cost;
      g.nch = c;
    }
  }
  const int blocks = g.tiles * g.nch;
  L.grid = (blocks + 7) / 8 * 8;
  L.rounds = (int)((blocks + slots - 1) / slots);
  L.layers = (ez + g.nch - 1) / g.nch + (g.nch > 1 ? 1 : 0);
  return true;
}

}  // namespace

// Box of the free nodes of a structured mesh and its split.  False where the
// free nodes are no box, an index would not fit or no tile covers the box.
bool lattice_plan(const femhip_mesh_desc_t &mesh, int cus, LatticeOp &L, int max_threads, int cells) {
  const int dim = mesh.dim, p = mesh.order;
  L = LatticeOp{};
  L.dim = dim;
  L.order = p;
  L.ncomp = mesh.num_components;
  Lattice &g = L.g;
  int64_t rows = 1;
  for (int d = 0; d < dim; ++d) {
    g.nc[d] = mesh.n[d];
    const bool lo = mesh.dirichlet == FEMHIP_BC_ALL_BOUNDARY || (mesh.dirichlet == FEMHIP_BC_X0_FACE && d == 0);
    const bool hi = mesh.dirichlet == FEMHIP_BC_ALL_BOUNDARY;
    g.o[d] = lo ? 1 : 0;
    const int64_t m = (int64_t)p * mesh.n[d] + 1 - (lo ? 1 : 0) - (hi ? 1 : 0);
    if (m < 1 || m > INT32_MAX) return false;
    g.m[d] = (int)m;
    g.E[d] = mesh.n[d] + (hi ? 0 : 1);
    rows *= m;
    if (rows * L.ncomp > INT32_MAX) return false;
  }
  g.stride = (int)rows;
  L.one = lattice_one(rows * L.ncomp, dim, p, L.ncomp);
  if (max_threads <= 0) max_threads = lattice_tile(rows * L.ncomp, dim, p, L.ncomp);
  if (dim == 2 && p == 1) return split<2, 1>(L, cus, max_threads, cells);
  if (dim == 2) return split<2, 2>(L, cus, max_threads, cells);
  if (p == 1 && L.ncomp == 3) return split<3, 1, 3>(L, cus, max_threads, cells);
  if (p == 1) return split<3, 1>(L, cus, max_threads, cells);
  return split<3, 2>(L, cus, max_threads, cells);
}

// The lattice row of every row of a space, perm, if each (cell, local DOF) of
// its lists is the row its node has in the box (whoever numbered them).
bool lattice_rows(const femhip_space &s, LatticeOp &L, DevBuf<int32_t> &perm) {
  const int32_t n = s.n_free;
  int64_t rows = L.ncomp;
  for (int d = 0; d < s.mesh.dim; ++d) rows *= L.g.m[d];
  if (rows != n) return false;
  hipStream_t st = s.ctx->stream;
  const FaceTab t = face_tab(s);
  DevBuf<int> bad;
  bad.alloc(1);
  perm.alloc((size_t)n);
  FH_HIP(hipMemsetAsync(bad.p, 0, sizeof(int), st));
  hipLaunchKernelGGL(k_lattice_perm, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, L.g, t, n, s.d_rep.p, perm.p,
                     bad.p);
  FH_HIP(hipGetLastError());
  int f = 1;
  FH_HIP(hipMemcpyAsync(&f, bad.p, sizeof(int), hipMemcpyDeviceToHost, st));
  FH_HIP(hipStreamSynchronize(st));
  if (f & 1) return false;
  L.identity = !(f & 2);
  FH_HIP(hipMemsetAsync(bad.p, 0, sizeof(int), st));
  const int64_t cnt = s.ncells * s.fe.nd;
  hipLaunchKernelGGL(k_lattice_check, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, st, L.g, t, s.ncells, n,
                     s.d_dofs.p, perm.p, bad.p);
  FH_HIP(hipGetLastError());
  FH_HIP(hipMemcpyAsync(&f, bad.p, sizeof(int), hipMemcpyDeviceToHost, st));
  FH_HIP(hipStreamSynchronize(st));
  return !f;
}

// The lattice form of a scalar Poisson or a vector Q1 elasticity operator on the
// uniform mesh (checked once against the space's DOF lists, whoever numbered
// them): op.lat, op.lat_perm.  Cells with their own map keep the stored matrix.
bool lattice_operator(femhip_operator &op) {
  if (op.structured) return op.lat_state > 0;
  if (!op.space || op.space->mapped || op.n <= 0) return false;
  if (op.lat_state != 0) return op.lat_state > 0;
  op.lat_state = -1;
  femhip_space &s = *op.space;
  if (op.tab_kind == 0 ? s.fe.ncomp != 1 : s.fe.ncomp != 3 || s.fe.dim != 3 || s.fe.order != 1) return false;
  auto L = std::make_shared<LatticeOp>();
  if (op.n > kLatticeMaxRows || !lattice_plan(s.mesh, op.ctx->num_cus, *L)) return false;   // byte offsets of the vectors
  const bool rows = lattice_rows(s, *L, op.lat_perm);
  if (!rows || L->identity) op.lat_perm.release();
  if (!rows) return false;
  op.lat = L;
  op.lat_state = 1;
  return true;
}

// Elasticity coefficients of cells of sides h.
static CoefDev elastic_coefficient(const double h[3], const femhip_physics_t &ph) {
  CoefDev c;
  const double w = h[0] * h[1] * h[2];   // eight points of weight det J
  c.k0 = w * (ph.nu * ph.E) / ((1 + ph.nu) * (1 - 2 * ph.nu));
  c.mu = w * ph.E / (2 * (1 + ph.nu));
  for (int d = 0; d < 3; ++d) c.c[d] = 1.0 / (4.0 * h[d]);
  return c;
}

// The operator's coefficient as the cells read it (after set_physics).
CoefDev lattice_coefficient(femhip_operator &op) {
  if (op.structured) {
    const double h[3] = {1.0 / op.lat->g.nc[0], 1.0 / op.lat->g.nc[1], 1.0 / op.lat->g.nc[2]};
    return elastic_coefficient(h, op.phys);
  }
  femhip_space &s = *op.space;
  const RefFE &fe = s.fe;
  CoefDev c;
  c.cells = s.ncells;
  c.k0 = op.phys.k0;
  double hs[3] = {1.0, 1.0, 1.0};   // the first cell's sides
  for (int d = 0; d < fe.dim; ++d) {
    const double lo = s.mesh.limits[2 * d], hi = s.mesh.limits[2 * d + 1];
    hs[d] = ((hi - lo) * (1.0 / (double)s.mesh.n[d]) + lo) - lo;
  }
  if (op.tab_kind == 1) return elastic_coefficient(hs, op.phys);
  // Q1: Gauss weights one; Q2: the weights are in the 1-D tables
  for (int d = 0; d < fe.dim; ++d) {
    const double h = hs[d];
    c.c[d] = fe.order == 1 ? fe.detj[0] * (4.0 / (h * h)) / (double)(1 << (2 * fe.dim)) : fe.detj[0] * (4.0 / (h * h));
  }
  if (op.phys.k_kind == FEMHIP_K_CELL) c.kc = op.k_cell.p;
  if (op.phys.k_kind == FEMHIP_K_SIN3) {
    ensure_trig(op);
    c.trig = reinterpret_cast<const double4 *>(op.trig.p);
    for (int d = 0; d < 3; ++d) c.toff[d] = op.trig_off[d];
  }
  if (op.phys.k_kind == FEMHIP_K_QPOINT) {
    if (op.lat_kq_version != op.phys_version) {
      const int64_t cnt = s.ncells * fe.nq;
      if (op.lat_kq.n != (size_t)cnt) op.lat_kq.alloc((size_t)cnt);
      hipLaunchKernelGGL(k_points_by_q, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0, op.ctx->stream, s.ncells,
                         fe.nq, op.k_qp.p, op.lat_kq.p);
      FH_HIP(hipGetLastError());
      op.lat_kq_version = op.phys_version;
    }
    c.kq = op.lat_kq.p;
  }
  return c;
}

Q2Tab lattice_q2_tab() {
  double x[3], w[3], B[3][3], D[3][3];
  gauss_legendre(3, x, w);
  const double t[3] = {-1.0, 0.0, 1.0};
  for (int q = 0; q < 3; ++q)
    for (int i = 0; i < 3; ++i) {
      const int j = (i + 1) % 3, l = (i + 2) % 3;
      // shapes through the nodes at the points, and derivatives at the points
      // of the polynomials through the points
      B[q][i] = std::sqrt(w[q]) * (x[q] - t[j]) * (x[q] - t[l]) / ((t[i] - t[j]) * (t[i] - t[l]));
      D[q][i] = std::sqrt(w[q] / w[i]) * ((x[q] - x[j]) + (x[q] - x[l])) / ((x[i] - x[j]) * (x[i] - x[l]));
    }
  Q2Tab k;
  k.b0 = 0.5 * (B[0][0] + B[0][2]);
  k.b1 = B[0][1];
  k.c = 0.5 * (B[0][0] - B[0][2]);
  k.beta = B[1][1];
  k.r = 0.5 * (D[0][2] - D[0][0]);
  k.ec = -0.5 * (D[0][0] + D[0][2]);
  k.b = D[0][1];
  k.delta = D[1][2];
  return k;
}

}  // namespace femhip
