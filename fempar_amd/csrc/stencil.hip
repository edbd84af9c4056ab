// stencil.hip -- structured elasticity operator for the request server.
//
// The request server's problems are vector-Q1 linear elasticity on the unit
// cube with n cells per direction, all components clamped on x = 0 and
// constant (E, nu, body force).  Every cell has the same element matrix (the
// irreducible plugin, sbm_irreducible_discrete_integration.i90:64-130), and the
// solver forms its products from the cells (lattice.h), so nothing is stored
// but the diagonal and the right-hand side: rows are component-major, row
// (c, node) = c * blk + node, with the free vertices (x index 1..n) numbered
// x-fastest and each component block padded to a multiple of 64 rows (padding
// rows: diagonal 1, RHS 0).  One thread per row sums the element entries of the
// cells around its vertex in ascending cell order.  (With the 81-point stencil
// assembled in the sliced format, 972 B a row, a request of n = 56 held 525 MB
// more and an iteration streamed 324 B a row.)
#include <hip/hip_runtime.h>

#include <vector>

#include "femhip_internal.h"
#include "lattice.h"

namespace femhip {
namespace {

struct StencilDev {
  int n;      // cells per direction
  int blk;    // rows per component block (multiple of 64)
  int nodes;  // free vertices, n (n+1)^2
};

__global__ __launch_bounds__(256) void k_stencil_rows(StencilDev g, const double *__restrict__ Ke,
                                                      const double *__restrict__ Fe, double *__restrict__ diag,
                                                      double *__restrict__ rhs) {
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= 3 * (int64_t)g.blk) return;
  const int c = (int)(r / g.blk);
  const int node = (int)(r % g.blk);
  if (node >= g.nodes) {   // padding row
    diag[r] = 1.0;
    rhs[r] = 0.0;
    return;
  }
  const int n = g.n, mx = n, my = n + 1;
  const int a = node % mx + 1, b = (node / mx) % my, z = node / (mx * my);   // vertex, a in 1..n
  double dacc = 0.0, bacc = 0.0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {   // cells around the vertex, ascending cell index
    const int ex = e & 1, ey = (e >> 1) & 1, ez = e >> 2;
    const int ci = a - 1 + ex, cj = b - 1 + ey, ck = z - 1 + ez;
    if (ci < 0 || ci >= n || cj < 0 || cj >= n || ck < 0 || ck >= n) continue;
    const int il = c * 8 + (1 - ex) + 2 * (1 - ey) + 4 * (1 - ez);   // the DOF in this cell
    bacc += Fe[il];
    dacc += Ke[il * 24 + il];
  }
  diag[r] = dacc;
  rhs[r] = bacc;
}

}  // namespace

// The bound of the earlier stored form (243 x padded vertices indexed with 32
// bits), kept so that a request is accepted or refused as before.
bool structured_elasticity_fits(int32_t n) {
  if (n < 1 || n > 1024) return false;
  const int64_t nodes = (int64_t)n * (n + 1) * (n + 1);
  const int64_t blk = (nodes + 63) / 64 * 64;
  return 3 * blk * 81 < (int64_t)INT32_MAX;
}

femhip_operator *create_structured_elasticity(femhip_ctx *ctx, int32_t n, const femhip_physics_t &ph) {
  FH_CHECK(structured_elasticity_fits(n), FEMHIP_ERR_INVALID,
           "structured elasticity needs 1 <= n with 243 x padded vertices < 2^31 (n <= 206)");
  FH_CHECK(ph.kind == FEMHIP_PHYS_ELASTICITY && ph.E > 0 && ph.nu > -1.0 && ph.nu < 0.5, FEMHIP_ERR_INVALID,
           "invalid elasticity parameters");
  const int64_t nodes = (int64_t)n * (n + 1) * (n + 1);
  const int64_t blk = (nodes + 63) / 64 * 64;
  const int64_t rows = 3 * blk;
  auto *op = new femhip_operator();
  op->ctx = ctx_retain(ctx);
  try {
    hipStream_t st = ctx->stream;
    op->structured = true;
    op->blk = (int32_t)blk;
    op->nodes = (int32_t)nodes;
    op->n = (int32_t)rows;
    op->phys = ph;
    op->has_physics = true;
    // element matrix of the first cell (uniform spacing 1/n)
    RefFE fe;
    const double h[3] = {1.0 / n, 1.0 / n, 1.0 / n};
    build_reffe(fe, 3, 1, 3, h);
    std::vector<double> t(24 * 24 + 24);
    elasticity_element(fe, ph, t.data(), t.data() + 24 * 24);
    op->tab.alloc(t.size());
    FH_HIP(hipMemcpyAsync(op->tab.p, t.data(), sizeof(double) * t.size(), hipMemcpyHostToDevice, st));
    op->rhs.alloc((size_t)rows);
    op->diag.alloc((size_t)rows);
    const StencilDev g{n, (int)blk, (int)nodes};
    hipLaunchKernelGGL(k_stencil_rows, dim3((unsigned)((rows + 255) / 256)), dim3(256), 0, st, g, op->tab.p,
                       op->tab.p + 24 * 24, op->diag.p, op->rhs.p);
    FH_HIP(hipGetLastError());
    femhip_mesh_desc_t mesh{};
    mesh.dim = 3;
    mesh.order = 1;
    mesh.num_components = 3;
    mesh.dirichlet = FEMHIP_BC_X0_FACE;
    for (int k = 0; k < 3; ++k) {
      mesh.n[k] = n;
      mesh.limits[2 * k + 1] = 1.0;
    }
    op->lat = std::make_shared<LatticeOp>();
    FH_CHECK(lattice_plan(mesh, ctx->num_cus, *op->lat), FEMHIP_ERR_INVALID, "mesh too large for the lattice");
    op->lat->g.stride = (int)blk;
    op->lat->identity = true;
    op->lat_state = 1;
    // the host vector above must outlive the copy
    FH_HIP(hipStreamSynchronize(st));
    op->computed = true;
    op->version = 1;
  } catch (...) {
    femhip_operator_destroy(op);
    throw;
  }
  return op;
}

}  // namespace femhip
