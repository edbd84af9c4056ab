// lattice.h -- products with the operator of a uniform structured mesh formed
// from its cells, without a stored matrix (device templates).
//
// On the structured generator's mesh every cell is a translate of the first,
// so the assembled operator is A = sum_c P_c^T K_c P_c with K_c fixed by the
// cell's coefficient alone: one value (or one per quadrature point, or a closed
// form of the position) instead of the 14 to 125 stored values a row of the
// assembled matrix.  The free nodes form a box of the fine grid (p n_k + 1
// nodes per direction, less the fixed faces), the vectors are kept in that
// lexicographic box order, and nodes outside the box are zeros that are never
// loaded.
//
// A workgroup owns a tile of cell columns, one cell per lane, and marches along
// the last direction: the new planes of nodes go through LDS to the lanes of
// the cells around them, each lane applies its cell in registers (sums
// factorised over the directions), the plane below passes its partial sums
// on in registers and the sums of nodes shared within the tile go through LDS.
// The first row and column of a tile (other than at the mesh's start) and the
// layer before a chunk are computed by both neighbours, so no sum crosses
// workgroups: no atomics, a fixed order of summation, every result written
// once.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "femhip_internal.h"

namespace femhip {

// Box lattice of the free nodes and its split into workgroups.  Lane (tx, ty)
// of tile (i, j) is cell (i (TX - 1) + tx, j (TY - 1) + ty); E_k counts the
// cells along k plus one where the last node plane is free (its owner is a
// cell past the mesh that only receives sums).
struct Lattice {
  int nc[3] = {1, 1, 1};   // cells
  int m[3] = {1, 1, 1};    // free nodes
  int o[3] = {0, 0, 0};    // grid index of free node 0
  int E[3] = {1, 1, 1};
  int TX = 1, TY = 1, xt = 1, tiles = 1, nch = 1;   // tile, tiles along x, all tiles, chunks of the march
  int stride = 0;          // rows between the components of a vector field
};

// Logical workgroup: each XCD (workgroups are dispatched round-robin over 8)
// takes a contiguous range, so tiles that share halos share an L2.
__device__ __forceinline__ int lattice_block(const Lattice &g) {
  const int per = (gridDim.x + 7) / 8;
  const int b = (int)(blockIdx.x % 8) * per + (int)(blockIdx.x / 8);
  return gridDim.x % 8 == 0 ? b : (int)blockIdx.x;
}

// Vectors are read and written through buffer resources whose range check
// gives 0 outside the vector and drops the store: nodes outside the box and
// lanes that own nothing need no branch.  Offsets are bytes of an 8-byte
// element; a vector has at most 2^30 bytes, kOutside plus any of them stays out
// of range, and so does kNoPlane plus an offset inside a plane.
constexpr uint32_t kOutside = 0x80000000u, kNoPlane = 0x40000000u;
constexpr int64_t kLatticeMaxRows = (int64_t)1 << 27;
using BufRsrc = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ BufRsrc buf_of(const void *p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, (int)bytes, 0x00027000);
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ double buf_ld64(BufRsrc r, uint32_t o8) {
  return __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, (int)o8, 0, 0));
}
__device__ __forceinline__ float buf_ld32(BufRsrc r, uint32_t o8) {
  return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)(o8 >> 1), 0, 0));
}
__device__ __forceinline__ void buf_st64(BufRsrc r, uint32_t o8, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, (int)o8, 0, 0);
}
__device__ __forceinline__ void buf_st32(BufRsrc r, uint32_t o8, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), r, (int)(o8 >> 1), 0, 0);
}

// The part of a lattice that logical workgroup lb reads, as a lattice of its
// own planes: row0 is its first row.  Vectors of any length then keep 30-bit
// byte offsets, as a chunk's planes do: lattice_plan with `cells` bounds its layers.
__device__ __forceinline__ Lattice lattice_window(const Lattice &g, int dim, int p, int lb, int64_t &row0, int64_t &rows) {
  Lattice w = g;
  const int a = dim - 1, chunk = lb / g.tiles;
  const int z0 = (int)((int64_t)g.E[a] * chunk / g.nch), z1 = (int)((int64_t)g.E[a] * (chunk + 1) / g.nch);
  const int first = max(p * max(z0 - 1, 0) - g.o[a], 0), last = min(p * z1 - g.o[a], g.m[a] - 1);   // planes of the box
  const int64_t plane = dim == 3 ? (int64_t)g.m[0] * g.m[1] : g.m[0];
  w.o[a] = g.o[a] + first;
  w.m[a] = max(last - first + 1, 0);
  row0 = first * plane;
  rows = w.m[a] * plane;
  return w;
}

template <int DIM, int P, int NC = 1>
struct LatticeShape {
  static constexpr int N1 = P + 1;
  static constexpr int NPL = DIM == 3 ? N1 * N1 : N1;   // a cell's nodes in one plane of the march
  static constexpr int OWN = DIM == 3 ? P * P : P;      // those the cell owns
  static constexpr int NX = NPL - OWN;                  // those it shares with the next cells
  // Q1: two sets of the LDS buffers and one barrier a layer, the loads of the
  // next plane in flight while a layer is computed.  Q2 holds too much in
  // registers for that, and vector Q1 in registers and LDS: one set, three
  // barriers.
  static constexpr bool PIPE = P == 1 && NC == 1;
};

// Iterations in one launch or two (cg_lattice.h): us an iteration in one / two,
// FP64 and FP32-refined.  3-D Q1, sin3 field: 24.9 / 31.7 and 28.6 / 29.4 at
// 100^3, 39.2 / 48.3 and 40.6 / 41.7 at 128^3, 66 / 81 and 68 / 62 at 160^3 (cell
// field there 84 / 75 and 53 / 51), 156 / 155 and 114 / 94 at 192^3.  2-D Q1: 19.7 /
// 27.8 at 700,000 rows.  3-D Q2: 20.6 / 32 at 32^3, 34.0 / 38.0 and 33.5 / 37.0 at
// 48^3 cells (857,000 rows), 56 / 54 and 53 / 49 at 64^3.  2-D Q2: 20.4 / 27.4 at
// 400^2 cells, 48 / 50 at 800^2.  Elasticity: 26.6 / 27.8 and 23.7 / 26.0 at 64^3
// (786,000 rows), 39 / 37 and 36 / 33 at 80^3.
__host__ __device__ constexpr bool lattice_one(int64_t rows, int dim, int p, int nc) {
  return rows < (dim == 3 && (p == 2 || nc > 1) ? 1000000 : 3000000);
}
// Largest workgroup and waves a SIMD (registers 512 / waves) of the marches.
// One launch: one workgroup a CU, since each reads all workgroups' partial sums
// at its start (128^3: 45 us an iteration with 768 workgroups of 256 threads, 39
// with 256 of 768; 1001 x 700 Q1: 25 and 20), and registers for twice the
// vectors; the cells of 3-D Q2 take all a wave can have.
__host__ __device__ constexpr int lattice_threads(int dim, int p, int nc, bool one) {
  return one ? (p == 1 && nc == 1 ? 768 : p == 2 && dim == 3 ? 256 : 512) : dim == 3 && p == 1 && nc == 1 ? 512 : 256;
}
__host__ __device__ constexpr int lattice_waves(int dim, int p, int nc, bool one) {
  return one ? (p == 1 && nc == 1 ? 3 : p == 2 && dim == 3 ? 1 : 2) : p == 1 && nc == 1 ? 4 : 2;
}
// Largest tile for a size: smaller ones where a large one would leave CUs
// without work (3-D Q1, 512 / 768 threads: 17.3 / 18.4 us at 80^3, 24.9 / 25.4 at
// 100^3, 48 / 39 at 128^3; elasticity, 256 / 512: 13.4 / 15.0 at 36^3, 19.8 / 18.7 at 50^3).
inline int lattice_tile(int64_t rows, int dim, int p, int nc) {
  const bool one = lattice_one(rows, dim, p, nc);
  const int most = lattice_threads(dim, p, nc, one);
  if (one && nc > 1) return rows < 300000 ? 256 : most;
  if (one && dim == 3 && p == 1) return rows < 1200000 ? 512 : most;
  return most;
}

// What an Io keeps of a node from value() to out(), in doubles (kKeep, at most).
constexpr int kLatticeKeep = 3;
// doubles of LDS a workgroup needs (new node planes, shared sums; PIPE: what
// the lanes keep of their own nodes in the last three planes)
template <int DIM, int P, int NC>
inline size_t lattice_lds(int TX, int TY) {
  using S = LatticeShape<DIM, P, NC>;
  const size_t cells = (size_t)TX * TY, plane = (size_t)(P * TX + 1) * (DIM == 3 ? P * TY + 1 : 1);
  return (S::PIPE ? 2 : 1) * (size_t)(NC * P) * (plane + S::NX * cells) + (S::PIPE ? 3 * kLatticeKeep * cells : 0);
}
// nodes of the row and column after a tile, one a thread
template <int DIM, int P>
inline int lattice_halo(int TX, int TY) {
  return DIM == 3 ? P * (TX + TY) + 1 : 1;
}

// March of logical workgroup lb; false: it has no cells, and ready() was not called.
// Cell: begin(cx, cy, in the mesh), Next prefetch(cz) and
// advance(next) for its coefficient, bottom(u) with the nodes of the first plane,
// step(active, u, s): the P next planes in, the finished sums of the P planes
// before the last of them out (this cell's share).
// Io: Raw fetch(o) loads what the node at offset o needs; ready() then forms
// what the pass needs first (false: nothing to do); value(raw, o, keep) gives
// the node's value and stores what the pass updates there (o = kOutside: not
// this workgroup's); out<FULL>(o, keep, y) takes the finished sum y of the
// node, with all of what value() kept (FULL) or only its value, keep[0].
// halo(o) and halo_value(raw): the value alone, of a node past the tile.
// kAhead3: planes loaded before they are used, in 3-D (> 1: a vector field's
// next plane, too: elasticity 17.2 -> 16.5 us an iteration at 65,000 nodes; in FP64
// it spills, 13.4 -> 15.9).
template <int DIM, int P, class Cell, class Io>
__device__ __forceinline__ bool lattice_march(const Lattice &g, int lb, Cell &cell, Io &io, double *lds) {
  constexpr int NC = Cell::kComps;
  using S = LatticeShape<DIM, P, NC>;
  constexpr int N1 = S::N1, NPL = S::NPL, OWN = S::OWN, NX = S::NX;
  constexpr bool PIPE = S::PIPE;
  constexpr int AX = DIM - 1;
  if (lb >= g.tiles * g.nch) return false;   // the same for the whole workgroup
  const int tile = lb % g.tiles, chunk = lb / g.tiles;
  const int ti = tile % g.xt, tj = tile / g.xt;
  const int TX = g.TX, TY = DIM == 3 ? g.TY : 1;
  const int X0 = ti * (TX - 1), Y0 = DIM == 3 ? tj * (TY - 1) : 0;
  const int tid = threadIdx.x, cells = TX * TY;
  const int tx = DIM == 3 ? tid % TX : tid, ty = DIM == 3 ? tid / TX : 0;
  const bool lane = tid < cells;
  const int cx = X0 + tx, cy = Y0 + ty;
  const bool own_xy = lane && (tx > 0 || ti == 0) && (DIM == 2 || ty > 0 || tj == 0);
  const bool in_xy = lane && cx < g.nc[0] && (DIM == 2 || cy < g.nc[1]);
  const int z0 = (int)((int64_t)g.E[AX] * chunk / g.nch), z1 = (int)((int64_t)g.E[AX] * (chunk + 1) / g.nch);
  if (z0 >= z1) return false;
  const int zs = z0 > 0 ? z0 - 1 : 0;
  const int LX = P * TX + 1, LY = DIM == 3 ? P * TY + 1 : 1, LP = LX * LY;
  const uint32_t plane_bytes = 8u * (uint32_t)(DIM == 3 ? g.m[0] * g.m[1] : g.m[0]);
  // doubles of one set of buffers: U [NC][P][LY][LX], C [NC][P][NX][cells]
  const int half = NC * P * (LP + NX * cells);
  const uint32_t comp_bytes = 8u * (uint32_t)g.stride;

  auto row_offset = [&](int px, int py, bool ok) {
    const int gx = px - g.o[0], gy = DIM == 3 ? py - g.o[1] : 0;
    ok = ok && gx >= 0 && gx < g.m[0] && (DIM == 2 || (gy >= 0 && gy < g.m[1]));
    return ok ? 8u * (uint32_t)(gx + g.m[0] * gy) : kOutside;
  };
  uint32_t off[OWN];   // this lane's own nodes in a plane
#pragma unroll
  for (int j = 0; j < OWN; ++j) off[j] = row_offset(P * cx + j % P, P * cy + j / P, lane);
  // one node of the row and column after the tile
  const int nhalo = DIM == 3 ? LX + P * TY : 1;
  const int hrow = DIM == 2 ? 0 : tid < LX ? P * TY : tid - LX;
  const int hcol = DIM == 2 || tid >= LX ? P * TX : tid;
  const bool halo = tid < nhalo;
  const uint32_t hoff = row_offset(P * X0 + hcol, P * Y0 + hrow, halo);
  const int hat = hrow * LX + hcol;
  const int uat = P * ty * LX + P * tx;

  auto plane_base = [&](int z) {
    const int gz = z - g.o[AX];
    return gz >= 0 && gz < g.m[AX] ? (uint32_t)gz * plane_bytes : kNoPlane;
  };
  constexpr int AHEAD = PIPE && DIM == 3 ? Io::kAhead3 : 1;
  typename Io::Raw raws[AHEAD][NC][P][OWN];   // planes on their way
  typename Io::Halo hraws[AHEAD][NC][P];
  typename Cell::Next next_k[AHEAD];
  constexpr int KEEP = Io::kKeep;
  double *ring = lds + (PIPE ? 2 : 1) * half + (lane ? tid : 0);   // PIPE: [3][KEEP][cells], plane z in part z mod 3
  auto fetch = [&](int slot, int z, int count) {   // planes z .. z + count - 1
    auto &raw = raws[slot];
    auto &hraw = hraws[slot];
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int c = 0; c < P; ++c)
        if (c < count) {
          const uint32_t base = plane_base(z + c) + k * comp_bytes;
#pragma unroll
          for (int j = 0; j < OWN; ++j) raw[k][c][j] = io.fetch(base + off[j]);
          hraw[k][c] = io.halo(base + hoff);
        }
  };
  auto store = [&](int slot, double *U, int z, int count, int part) {
    auto &raw = raws[slot];
    auto &hraw = hraws[slot];
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int c = 0; c < P; ++c)
        if (c < count) {
          const uint32_t base = plane_base(z + c) + k * comp_bytes;
          const bool own = own_xy && (z + c) / P >= z0 && (z + c) / P < z1;   // the layer that owns the plane
          double *Up = U + (k * P + c) * LP;
#pragma unroll
          for (int j = 0; j < OWN; ++j) {
            double keep[KEEP];
            const double v = io.value(raw[k][c][j], own ? base + off[j] : kOutside, keep);
            if (lane) {
              Up[uat + (j / P) * LX + j % P] = v;
              if (PIPE)
#pragma unroll
                for (int i = 0; i < KEEP; ++i) ring[(part * KEEP + i) * cells] = keep[i];
            }
          }
          const double h = io.halo_value(hraw[k][c]);
          if (halo) Up[hat] = h;
        }
  };
  auto read_plane = [&](const double *U, int kc, double (&u)[NPL]) {   // kc = component * P + plane
    const double *Up = U + kc * LP + (lane ? uat : 0);
#pragma unroll
    for (int b = 0; b < (DIM == 3 ? N1 : 1); ++b)
#pragma unroll
      for (int a = 0; a < N1; ++a) u[b * N1 + a] = Up[b * LX + a];
  };
  // sums of shared nodes to their owners: slots (a = P, b < P), (b = P, a < P), (P, P)
  auto share = [&](double *C, const double (&s)[NC][P][NPL]) {
    if (lane) {
#pragma unroll
      for (int kc = 0; kc < NC * P; ++kc) {
        const double(&sp)[NPL] = s[kc / P][kc % P];
        double *Cp = C + kc * NX * cells + tid;
        if (DIM == 2) {
          Cp[0] = sp[P];
        } else {
#pragma unroll
          for (int j = 0; j < P; ++j) {
            Cp[j * cells] = sp[j * N1 + P];
            Cp[(P + j) * cells] = sp[P * N1 + j];
          }
          Cp[2 * P * cells] = sp[P * N1 + P];
        }
      }
    }
  };
  const bool left = tx > 0, below = DIM == 3 && ty > 0, corner = left && below;
  // kept(k, c, j, keep): what is kept of own node j of plane c; so(k, c, j): this cell's sum there
  auto finish = [&](const double *C, int cz, auto &&so, auto &&kept) {
    if (cz < z0) return;
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
      for (int c = 0; c < P; ++c) {
        const uint32_t base = plane_base(P * cz + c) + k * comp_bytes;
        const double *Cp = C + (k * P + c) * NX * cells + (lane ? tid : 0);
#pragma unroll
        for (int j = 0; j < OWN; ++j) {
          const int a = j % P, b = j / P;
          double y = so(k, c, j);
          if (DIM == 2) {
            if (a == 0) y += left ? Cp[-1] : 0.0;
          } else {
            if (a == 0) y += left ? Cp[b * cells - 1] : 0.0;
            if (b == 0) y += below ? Cp[(P + a) * cells - TX] : 0.0;
            if (a == 0 && b == 0) y += corner ? Cp[2 * P * cells - TX - 1] : 0.0;
          }
          double keep[KEEP];
          kept(k, c, j, keep);
          io.template out<PIPE>(own_xy ? base + off[j] : kOutside, keep, y);
        }
      }
  };

  fetch(0, P * zs, 1);
  cell.begin(g, cx, cy, in_xy);
  if (!io.ready()) return true;   // the same for every workgroup
  store(0, lds, P * zs, 1, 0);
  double ub[NC][OWN];   // !PIPE: own nodes of the plane below the layer
  if (PIPE)
#pragma unroll
    for (int a = 0; a < AHEAD; ++a)
      if (zs + a < z1) {
        fetch(a, P * (zs + a) + 1, P);
        next_k[a] = cell.prefetch(g, zs + a, in_xy);
      }
  __syncthreads();
  {
    double u[NC][NPL];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      read_plane(lds, k * P, u[k]);
#pragma unroll
      for (int j = 0; j < OWN; ++j) ub[k][j] = u[k][(j / P) * N1 + j % P];
    }
    cell.bottom(u);
  }

  if (PIPE) {
    double so[OWN];
    int part = 0;   // of the plane below the layer finished next
    auto so_at = [&](int, int, int j) { return so[j]; };
    auto kept = [&](int, int, int, double (&keep)[KEEP]) {
#pragma unroll
      for (int i = 0; i < KEEP; ++i) keep[i] = ring[(part * KEEP + i) * cells];
    };
    int set = 1, next = 1;   // buffers; ring part of the plane stored next
    for (int cb = zs; cb < z1; cb += AHEAD) {
#pragma unroll
      for (int a = 0; a < AHEAD; ++a) {
        const int cz = cb + a;
        if (cz >= z1) break;
        double *U = lds + set * half, *C = U + P * LP;
        store(a, U, P * cz + 1, P, next);
        next = next == 2 ? 0 : next + 1;
        cell.advance(next_k[a]);
        __syncthreads();
        if (cz > zs) {
          finish(lds + (set ^ 1) * half + P * LP, cz - 1, so_at, kept);
          part = part == 2 ? 0 : part + 1;
        }
        if (cz + AHEAD < z1) {
          fetch(a, P * (cz + AHEAD) + 1, P);
          next_k[a] = cell.prefetch(g, cz + AHEAD, in_xy);
        }
        double u[NC][P][NPL], s[NC][P][NPL];
#pragma unroll
        for (int c = 0; c < P; ++c) read_plane(U, c, u[0][c]);
        cell.step(in_xy && cz < g.nc[AX], u, s);
        share(C, s);
#pragma unroll
        for (int j = 0; j < OWN; ++j) so[j] = s[0][0][(j / P) * N1 + j % P];
        set ^= 1;
      }
    }
    __syncthreads();
    finish(lds + (set ^ 1) * half + P * LP, z1 - 1, so_at, kept);
  } else {
    double *U = lds, *C = U + NC * P * LP;
    const double *Uo = U + (lane ? uat : 0);
    auto u_at = [&](int k, int c, int j) { return Uo[(k * P + c) * LP + (j / P) * LX + j % P]; };
    // the next plane's loads while a layer is computed, where there are registers for them
    constexpr bool EARLY = NC > 1 && Io::kAhead3 > 1;
    if (EARLY) fetch(0, P * zs + 1, P);
    for (int cz = zs; cz < z1; ++cz) {
      if (!EARLY) fetch(0, P * cz + 1, P);
      cell.advance(cell.prefetch(g, cz, in_xy));
      __syncthreads();   // the layer before has read U and C
      store(0, U, P * cz + 1, P, 0);
      if (EARLY && cz + 1 < z1) fetch(0, P * (cz + 1) + 1, P);
      __syncthreads();
      double u[NC][P][NPL], s[NC][P][NPL];
#pragma unroll
      for (int kc = 0; kc < NC * P; ++kc) read_plane(U, kc, u[kc / P][kc % P]);
      cell.step(in_xy && cz < g.nc[AX], u, s);
      share(C, s);
      __syncthreads();
      finish(C, cz, [&](int k, int c, int j) { return s[k][c][(j / P) * N1 + j % P]; },
             [&](int k, int c, int j, double (&keep)[KEEP]) { keep[0] = c == 0 ? ub[k][j] : u_at(k, c - 1, j); });
#pragma unroll
      for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int j = 0; j < OWN; ++j) ub[k][j] = u_at(k, P - 1, j);
    }
  }
  return true;
}

// ----------------------------------------------------------------- cells ---

// Where the coefficient of a Poisson cell comes from.
enum { kCoefCell = 0,    // one value: k0, or kc[cell]
       kCoefSin3 = 1,    // 1 + 1/2 prod sin(2 pi x_d), from the sines at the 1-D Gauss points of each layer
       kCoefPoint = 2,   // kq[q cells + cell]
       kElastic = 3 };   // vector Q1, constant Lame coefficients

struct CoefDev {
  double k0 = 1.0, mu = 0.0;       // kElastic: lambda and mu, times the weights of the points
  const double *kc = nullptr, *kq = nullptr;
  const double4 *trig = nullptr;   // {., ., sin 2 pi x, .} per (layer, point), offsets per direction
  int toff[3] = {0, 0, 0};
  int64_t cells = 0;
  double c[3] = {0, 0, 0};         // weight of the squared derivative along each direction
  bool operator==(const CoefDev &o) const {
    bool same = k0 == o.k0 && mu == o.mu && kc == o.kc && kq == o.kq && trig == o.trig && cells == o.cells;
    for (int d = 0; d < 3; ++d) same = same && toff[d] == o.toff[d] && c[d] == o.c[d];
    return same;
  }
};

// Q1: in each direction the two end values become their sum and difference,
// in which the 1-D interpolation to the Gauss points +-1/sqrt(3) is
// (s +- d / sqrt(3)) / 2 and the derivative d / h.  A derivative along x is
// constant along x, so it has 4 (2) values in a cell, each weighted by the
// coefficient summed over the two points along x; the factors 1/2 and 1/h are
// in CoefDev::c.  One value a cell: the weights pull out and the form is
// diagonal in these modes.  About 55 (one value) to 140 FP64 operations a cell
// in 3-D against 2 x 27 a row of the assembled matrix, but no stored value.
constexpr double kGauss2 = 0.57735026918962576451;   // 1 / sqrt(3)

template <int DIM, int KIND>
struct CellQ1 {
  static constexpr int kComps = 1, NPL = DIM == 3 ? 4 : 2, NV = 1 << DIM, NK = KIND == kCoefPoint ? NV : 1;
  CoefDev k;
  struct Next {                   // a layer's coefficient, loaded ahead
    double v[KIND == kCoefSin3 ? 2 : NK];
  };
  double kv[NK];                  // this layer's values
  double sz[2];                   // sines at the march's points
  double ka[2], kb[2], kc4[4];    // in-plane factors of the coefficient summed along x, y and the march
  double below[NPL], carry[NPL];  // modes of the plane below, unfinished sums of its modes
  int64_t col, plane;

  __device__ __forceinline__ void begin(const Lattice &g, int cx, int cy, bool in) {
    col = in ? cx + (int64_t)g.nc[0] * (DIM == 3 ? cy : 0) : 0;
    plane = (int64_t)g.nc[0] * (DIM == 3 ? g.nc[1] : 1);
    if (KIND == kCoefSin3) {
      const int x = in ? cx : 0, y = in ? cy : 0;
      const double x0 = k.trig[k.toff[0] + 2 * x].z, x1 = k.trig[k.toff[0] + 2 * x + 1].z;
      if (DIM == 3) {
        const double y0 = k.trig[k.toff[1] + 2 * y].z, y1 = k.trig[k.toff[1] + 2 * y + 1].z;
        ka[0] = 0.5 * (x0 + x1) * y0;
        ka[1] = 0.5 * (x0 + x1) * y1;
        kb[0] = 0.5 * (y0 + y1) * x0;
        kb[1] = 0.5 * (y0 + y1) * x1;
        kc4[0] = x0 * y0;
        kc4[1] = x1 * y0;
        kc4[2] = x0 * y1;
        kc4[3] = x1 * y1;
      } else {
        ka[0] = 0.5 * (x0 + x1);
        kb[0] = x0;
        kb[1] = x1;
      }
    }
#pragma unroll
    for (int i = 0; i < NPL; ++i) carry[i] = 0.0;
  }
  __device__ __forceinline__ Next prefetch(const Lattice &g, int cz, bool in) const {
    const int z = min(cz, g.nc[DIM - 1] - 1);
    const int64_t at = col + plane * z;
    Next n;
    if (KIND == kCoefCell) {
      n.v[0] = k.kc ? k.kc[at] : k.k0;
    } else if (KIND == kCoefPoint) {
#pragma unroll
      for (int q = 0; q < NV; ++q) n.v[q % NK] = k.kq[q * k.cells + at];
    } else {
      n.v[0] = k.trig[k.toff[DIM - 1] + 2 * z].z;
      n.v[1 % (KIND == kCoefSin3 ? 2 : NK)] = k.trig[k.toff[DIM - 1] + 2 * z + 1].z;
    }
    return n;
  }
  __device__ __forceinline__ void advance(const Next &n) {
    if (KIND == kCoefSin3) {
      sz[0] = n.v[0];
      sz[1] = n.v[1 % (KIND == kCoefSin3 ? 2 : NK)];
    } else {
#pragma unroll
      for (int q = 0; q < NK; ++q) kv[q] = n.v[q];
    }
  }
  // coefficient summed over the two points along direction d, at point (qe, qf)
  // of the other directions (ascending)
  __device__ __forceinline__ double ksum(int d, int qe, int qf) const {
    if (KIND == kCoefPoint) {
      const int e = d == 0 ? 1 : 0, f = 3 - d - e;
      const int q = (qe << e) | (DIM == 3 ? qf << f : 0);
      return kv[q] + kv[q | (1 << d)];
    }
    if (DIM == 2) return d == 0 ? __builtin_fma(ka[0], sz[qe], 2.0) : __builtin_fma(kb[qe], 0.5 * (sz[0] + sz[1]), 2.0);
    if (d == 0) return __builtin_fma(ka[qe], sz[qf], 2.0);
    if (d == 1) return __builtin_fma(kb[qe], sz[qf], 2.0);
    return __builtin_fma(kc4[qe + 2 * qf], 0.5 * (sz[0] + sz[1]), 2.0);
  }
  // nodes of a plane -> sums and differences in the plane (bit set = difference)
  static __device__ __forceinline__ void modes(const double (&u)[NPL], double (&m)[NPL]) {
    if (DIM == 2) {
      m[0] = u[0] + u[1];
      m[1] = u[1] - u[0];
    } else {
      const double a = u[0] + u[1], b = u[1] - u[0], c = u[2] + u[3], d = u[3] - u[2];
      m[0] = a + c;
      m[1] = b + d;
      m[2 % NPL] = c - a;
      m[3 % NPL] = d - b;
    }
  }
  // and the transpose
  static __device__ __forceinline__ void nodes(const double (&m)[NPL], double (&u)[NPL]) {
    if (DIM == 2) {
      u[0] = m[0] - m[1];
      u[1] = m[0] + m[1];
    } else {
      const double a = m[0] - m[2 % NPL], b = m[1] - m[3 % NPL], c = m[0] + m[2 % NPL], d = m[1] + m[3 % NPL];
      u[0] = a - b;
      u[1] = a + b;
      u[2 % NPL] = c - d;
      u[3 % NPL] = c + d;
    }
  }
  __device__ __forceinline__ void bottom(const double (&u)[1][NPL]) { modes(u[0], below); }
  __device__ __forceinline__ void step(bool active, const double (&u)[1][1][NPL], double (&s)[1][1][NPL]) {
    double h[NV], r[NV], top[NPL], sum[NPL];
    modes(u[0][0], top);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      h[i] = below[i] + top[i];
      h[NPL + i] = top[i] - below[i];
      below[i] = top[i];
    }
    constexpr double al = kGauss2, t = 1.0 / 3.0;   // interpolation's difference factor and its square
    if (KIND == kCoefCell) {
      const double kc = active ? kv[0] : 0.0;
      r[0] = 0.0;
#pragma unroll
      for (int i = 1; i < NV; ++i) {
        const int others = __builtin_popcount(i) - 1;
        const double f = (others == 0 ? 1.0 : others == 1 ? t : t * t) * (double)NV;
        double w = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d)
          if ((i >> d) & 1) w += k.c[d];
        r[i] = (w * f) * h[i];
      }
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        sum[i] = __builtin_fma(kc, r[i] - r[NPL + i], carry[i]);
        carry[i] = kc * (r[i] + r[NPL + i]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NV; ++i) r[i] = 0.0;
      if (active) {   // lanes past the mesh only pass sums on
#pragma unroll
        for (int d = 0; d < DIM; ++d) {
          const int D = 1 << d, e = d == 0 ? 1 : 0, E = 1 << e;
          if (DIM == 2) {
            const double g0 = __builtin_fma(-al, h[D | E], h[D]), g1 = __builtin_fma(al, h[D | E], h[D]);
            const double w0 = g0 * ksum(d, 0, 0), w1 = g1 * ksum(d, 1, 0);
            r[D] = __builtin_fma(k.c[d], w0 + w1, r[D]);
            r[D | E] = __builtin_fma(k.c[d] * al, w1 - w0, r[D | E]);
          } else {
            const int f = 3 - d - e, F = 1 << f;
            const double a0 = __builtin_fma(-al, h[D | E], h[D]), a1 = __builtin_fma(al, h[D | E], h[D]);
            const double b0 = __builtin_fma(-al, h[D | E | F], h[D | F]), b1 = __builtin_fma(al, h[D | E | F], h[D | F]);
            const double w00 = __builtin_fma(-al, b0, a0) * ksum(d, 0, 0);
            const double w10 = __builtin_fma(-al, b1, a1) * ksum(d, 1, 0);
            const double w01 = __builtin_fma(al, b0, a0) * ksum(d, 0, 1);
            const double w11 = __builtin_fma(al, b1, a1) * ksum(d, 1, 1);
            const double s0 = w00 + w10, d0 = w10 - w00, s1 = w01 + w11, d1 = w11 - w01;
            r[D] = __builtin_fma(k.c[d], s0 + s1, r[D]);
            r[D | E] = __builtin_fma(k.c[d] * al, d0 + d1, r[D | E]);
            r[D | F] = __builtin_fma(k.c[d] * al, s1 - s0, r[D | F]);
            r[D | E | F] = __builtin_fma(k.c[d] * al * al, d1 - d0, r[D | E | F]);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        sum[i] = carry[i] + (r[i] - r[NPL + i]);
        carry[i] = r[i] + r[NPL + i];
      }
    }
    nodes(sum, s[0][0]);
  }
};

// Vector Q1, lambda div div + 2 mu eps : eps with constant lambda, mu.  In the
// sums and differences of CellQ1 the derivative along i at the Gauss points is
// a polynomial in the point's signs: one coefficient for each subset of the
// other directions, and products of different subsets sum to zero over the
// points.  So the form is a few 3 x 3 couplings, one for each subset.
struct CellElastic {
  static constexpr int kComps = 3, NPL = 4, NV = 8;
  CoefDev k;   // c[i] = 1 / (4 h_i); k0, mu = lambda, mu times the eight points' weights
  double below[3][NPL], carry[3][NPL];

  __device__ __forceinline__ void begin(const Lattice &, int, int, bool) {
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int i = 0; i < NPL; ++i) carry[c][i] = 0.0;
  }
  struct Next {};
  __device__ __forceinline__ Next prefetch(const Lattice &, int, bool) const { return {}; }
  __device__ __forceinline__ void advance(const Next &) {}
  __device__ __forceinline__ void bottom(const double (&u)[3][NPL]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) CellQ1<3, kCoefCell>::modes(u[c], below[c]);
  }
  __device__ __forceinline__ void step(bool active, const double (&u)[3][1][NPL], double (&s)[3][1][NPL]) {
    double h[3][NV], r[3][NV];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double top[NPL];
      CellQ1<3, kCoefCell>::modes(u[c][0], top);
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        h[c][i] = below[c][i] + top[i];
        h[c][NPL + i] = top[i] - below[c][i];
        below[c][i] = top[i];
      }
#pragma unroll
      for (int i = 0; i < NV; ++i) r[c][i] = 0.0;
    }
    if (active) {   // lanes past the mesh only pass sums on
      constexpr double al = kGauss2;
      auto power = [](int S) { return S == 0 ? 1.0 : (S & (S - 1)) == 0 ? al : al * al; };
#pragma unroll
      for (int S = 0; S < 7; ++S) {   // subsets of the directions
        const double f = power(S);
        double div = 0.0;
#pragma unroll
        for (int c = 0; c < 3; ++c)
          if (!((S >> c) & 1)) div = __builtin_fma(k.c[c] * f, h[c][(1 << c) | S], div);
        div *= k.k0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          if ((S >> c) & 1) continue;
          const double g = (k.c[c] * f) * h[c][(1 << c) | S];
          r[c][(1 << c) | S] = __builtin_fma(k.c[c] * f, __builtin_fma(2.0 * k.mu, g, div), r[c][(1 << c) | S]);
        }
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int i = c + 1; i < 3; ++i) {   // shear: derivatives of component c along i and of i along c
            const bool ci = !((S >> i) & 1), ic = !((S >> c) & 1);
            if (!ci && !ic) continue;
            double e = 0.0;
            if (ci) e = (k.c[i] * f) * h[c][((1 << i) | S) & 7];
            if (ic) e = __builtin_fma(k.c[c] * f, h[i][((1 << c) | S) & 7], e);
            e *= k.mu;
            if (ci) r[c][((1 << i) | S) & 7] = __builtin_fma(k.c[i] * f, e, r[c][((1 << i) | S) & 7]);
            if (ic) r[i][((1 << c) | S) & 7] = __builtin_fma(k.c[c] * f, e, r[i][((1 << c) | S) & 7]);
          }
      }
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      double sum[NPL];
#pragma unroll
      for (int i = 0; i < NPL; ++i) {
        sum[i] = carry[c][i] + (r[c][i] - r[c][NPL + i]);
        carry[c][i] = r[c][i] + r[c][NPL + i];
      }
      CellQ1<3, kCoefCell>::nodes(sum, s[c][0]);
    }
  }
};

// Q2: interpolation to the 3 Gauss points in every direction (values scaled by
// the square roots of the weights, so no weight is left), then along each
// direction the derivative at the points, the coefficient, and the transposes.
// Both 3 x 3 factors split into the even and odd parts of the three values.
struct Q2Tab {
  double b0, b1, c, beta;      // interpolation: E = b0 (u0 + u2) + b1 u1, +- c (u2 - u0); centre beta u1
  double r, delta, ec, b;      // derivative: R = r (v2 - v0), Q = ec (v0 + v2) - b v1; R -+ Q; centre delta (v2 - v0)
};

template <int DIM, int KIND>
struct CellQ2 {
  static constexpr int kComps = 1, NPL = DIM == 3 ? 9 : 3, N = DIM == 3 ? 27 : 9;
  CoefDev k;
  Q2Tab t;
  struct Next {                    // a layer's coefficient
    double kv, sz[3];
    int64_t at;
  };
  double kv;
  double sz[3], kxy[NPL];
  double below[NPL], carry[NPL];   // the plane below interpolated in the plane, its unfinished sums
  int64_t col, plane, at0;

  __device__ __forceinline__ void begin(const Lattice &g, int cx, int cy, bool in) {
    col = in ? cx + (int64_t)g.nc[0] * (DIM == 3 ? cy : 0) : 0;
    plane = (int64_t)g.nc[0] * (DIM == 3 ? g.nc[1] : 1);
    if (KIND == kCoefSin3) {
      const int x = in ? cx : 0, y = in ? cy : 0;
#pragma unroll
      for (int i = 0; i < NPL; ++i)
        kxy[i] = k.trig[k.toff[0] + 3 * x + i % 3].z * (DIM == 3 ? k.trig[k.toff[1] + 3 * y + i / 3].z : 1.0);
    }
#pragma unroll
    for (int i = 0; i < NPL; ++i) carry[i] = 0.0;
  }
  __device__ __forceinline__ Next prefetch(const Lattice &g, int cz, bool in) const {
    const int z = min(cz, g.nc[DIM - 1] - 1);
    Next n{};
    n.at = col + plane * z;
    if (KIND == kCoefCell) {
      n.kv = k.kc ? k.kc[n.at] : k.k0;
    } else if (KIND == kCoefSin3) {
#pragma unroll
      for (int a = 0; a < 3; ++a) n.sz[a] = 0.5 * k.trig[k.toff[DIM - 1] + 3 * z + a].z;
    }
    return n;
  }
  __device__ __forceinline__ void advance(const Next &n) {
    at0 = n.at;
    kv = n.kv;
#pragma unroll
    for (int a = 0; a < 3; ++a) sz[a] = n.sz[a];
  }
  __device__ __forceinline__ double at(int q) const {
    if (KIND == kCoefPoint) return k.kq[q * k.cells + at0];
    if (KIND == kCoefSin3) return __builtin_fma(kxy[q % NPL], sz[q / NPL], 1.0);
    return 1.0;
  }
  // The coefficients of a cell's points are formed (or loaded) again for each
  // direction: 27 of them kept would spill.
  __device__ __forceinline__ void forget() {
    if (KIND == kCoefSin3) {
#pragma unroll
      for (int a = 0; a < 3; ++a) asm volatile("" : "+v"(sz[a]));
    } else if (KIND == kCoefPoint) {
      asm volatile("" : "+v"(at0));
    }
  }
  // interpolation along the direction of stride st of M values, and its transpose
  template <int st, int M>
  __device__ __forceinline__ void interp(double (&v)[M]) const {
#pragma unroll
    for (int i = 0; i < M; ++i)
      if ((i / st) % 3 == 0) {
        const double u0 = v[i], u1 = v[i + st], u2 = v[i + 2 * st];
        const double o = u2 - u0, e = __builtin_fma(t.b1, u1, t.b0 * (u0 + u2));
        v[i] = __builtin_fma(-t.c, o, e);
        v[i + st] = t.beta * u1;
        v[i + 2 * st] = __builtin_fma(t.c, o, e);
      }
  }
  template <int st, int M>
  __device__ __forceinline__ void interp_t(double (&v)[M]) const {
#pragma unroll
    for (int i = 0; i < M; ++i)
      if ((i / st) % 3 == 0) {
        const double y0 = v[i], y1 = v[i + st], y2 = v[i + 2 * st];
        const double e = y0 + y2, o = y2 - y0, E = t.b0 * e;
        v[i] = __builtin_fma(-t.c, o, E);
        v[i + st] = __builtin_fma(t.b1, e, t.beta * y1);
        v[i + 2 * st] = __builtin_fma(t.c, o, E);
      }
  }
  template <int st>
  __device__ __forceinline__ void derive(double cd, const double (&v)[N], double (&w)[N]) const {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if ((i / st) % 3 == 0) {
        const double v0 = v[i], v1 = v[i + st], v2 = v[i + 2 * st];
        const double o = v2 - v0, Q = __builtin_fma(t.ec, v0 + v2, -t.b * v1);
        double g0 = __builtin_fma(t.r, o, -Q), g1 = t.delta * o, g2 = __builtin_fma(t.r, o, Q);
        if (KIND != kCoefCell) {
          g0 *= at(i);
          g1 *= at(i + st);
          g2 *= at(i + 2 * st);
        }
        const double R = g0 + g2, D = g2 - g0;
        const double oc = __builtin_fma(t.r, R, t.delta * g1), e = t.ec * D;
        w[i] = __builtin_fma(cd, e - oc, w[i]);
        w[i + st] = __builtin_fma(-cd * t.b, D, w[i + st]);
        w[i + 2 * st] = __builtin_fma(cd, e + oc, w[i + 2 * st]);
      }
  }
  __device__ __forceinline__ void in_plane(double (&v)[NPL]) const {
    interp<1, NPL>(v);
    if (DIM == 3) interp<DIM == 3 ? 3 : 1, NPL>(v);
  }
  __device__ __forceinline__ void bottom(const double (&u)[1][NPL]) {
#pragma unroll
    for (int i = 0; i < NPL; ++i) below[i] = u[0][i];
    in_plane(below);
  }
  __device__ __forceinline__ void step(bool active, double (&uc)[1][2][NPL], double (&sc)[1][2][NPL]) {
    double v[N], w[N];
    auto &u = uc[0];
    auto &s = sc[0];
    in_plane(u[0]);
    in_plane(u[1]);
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      v[i] = below[i];
      v[NPL + i] = u[0][i];
      v[2 * NPL + i] = u[1][i];
      below[i] = u[1][i];
    }
#pragma unroll
    for (int i = 0; i < N; ++i) w[i] = 0.0;
    if (active) {   // lanes past the mesh only pass sums on
      interp<NPL, N>(v);
      const double f = KIND == kCoefCell ? kv : 1.0;
      derive<1>(f * k.c[0], v, w);
      forget();
      derive<3>(f * k.c[1], v, w);
      forget();
      if (DIM == 3) derive<DIM == 3 ? 9 : 1>(f * k.c[2], v, w);
      interp_t<NPL, N>(w);
    }
#pragma unroll
    for (int i = 0; i < NPL; ++i) {
      s[0][i] = carry[i] + w[i];
      s[1][i] = w[NPL + i];
      carry[i] = w[2 * NPL + i];
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (DIM == 3) interp_t<DIM == 3 ? 3 : 1, NPL>(s[c]);
      interp_t<1, NPL>(s[c]);
    }
  }
};

// A lattice operator on the host (lattice.hip).
struct LatticeOp {
  Lattice g;
  int dim = 0, order = 0, ncomp = 1;
  bool one = false;                 // an iteration in one launch
  int threads = 64, grid = 8;       // workgroup size and count
  size_t lds = 0;                   // bytes of LDS a workgroup
  bool identity = false;            // lattice rows are the operator's rows
  int rounds = 1, layers = 1;       // workgroups a CU's slot takes in turn, layers each marches
};
// cus > 0: chunks that fill that many CUs; otherwise of about `cells` cells a workgroup
bool lattice_plan(const femhip_mesh_desc_t &mesh, int cus, LatticeOp &L, int max_threads = 0, int cells = 0);
bool lattice_rows(const femhip_space &s, LatticeOp &L, DevBuf<int32_t> &perm);
bool lattice_operator(femhip_operator &op);
CoefDev lattice_coefficient(femhip_operator &op);
Q2Tab lattice_q2_tab();

}  // namespace femhip
