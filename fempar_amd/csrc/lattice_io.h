// lattice_io.h -- what a lattice march (lattice.h) reads and writes at the nodes
// in the FP32-refined CG passes and in FP64 residuals, and the sums of a pass
// (device code shared by cg.hip and batch.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "cg_state.h"
#include "lattice.h"

namespace femhip {
namespace {

extern __shared__ double lattice_smem[];

// v plus the value of the lanes a DPP control names (no LDS round trip).
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_add(double v) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, CTRL, ROWS, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), CTRL, ROWS, 0xf, true);
  return v + __builtin_bit_cast(double, (uint64_t)(uint32_t)lo | ((uint64_t)(uint32_t)hi << 32));
}
// Sum over each row of 16 lanes, in its last lane.
__device__ __forceinline__ double row_sum15(double v) {
  v = dpp_add<0x111, 0xf>(v);   // row_shr:1
  v = dpp_add<0x112, 0xf>(v);   // row_shr:2
  v = dpp_add<0x114, 0xf>(v);   // row_shr:4
  return dpp_add<0x118, 0xf>(v);   // row_shr:8
}
// Sum over the wave, in lane 63.
__device__ __forceinline__ double wave_sum63(double v) {
  v = row_sum15(v);
  v = dpp_add<0x142, 0xa>(v);      // row_bcast:15 to rows 1 and 3
  return dpp_add<0x143, 0xc>(v);   // row_bcast:31 to rows 2 and 3
}
__device__ __forceinline__ double read_lane(double v, int lane) {
  const uint64_t b = __builtin_bit_cast(uint64_t, v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
  return __builtin_bit_cast(double, (uint64_t)lo | ((uint64_t)hi << 32));
}

// Sums over the workgroup, the same in every thread; sm: NV rows, free until
// the second barrier after this one.
template <int W, int NV>
__device__ __forceinline__ void block_sums(double (&v)[NV], double (*sm)[W]) {
  const int w = threadIdx.x >> 6;
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum63(v[k]);
  if ((threadIdx.x & 63) == 63)
#pragma unroll
    for (int k = 0; k < NV; ++k) sm[k][w] = v[k];
  __syncthreads();
  static_assert(W <= 16 && NV <= 4, "a row of 16 lanes takes a sum");
  const int lane = threadIdx.x & 63;
  const double a = row_sum15(lane < 16 * NV && (lane & 15) < W ? sm[lane >> 4][lane & (W - 1)] : 0.0);
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = read_lane(a, 16 * k + 15);
}

// Partial sums of workgroup lb of g: part[k * g + lb].
template <int NV>
__device__ __forceinline__ void group_partials(double (&v)[NV], double *part, int g, int lb) {
  __shared__ double sm[NV][16];
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = wave_sum63(v[k]);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
  if (lane == 63)
#pragma unroll
    for (int k = 0; k < NV; ++k) sm[k][w] = v[k];
  __syncthreads();
  if (threadIdx.x < NV) {
    double s = 0.0;
    for (int i = 0; i < nw; ++i) s += sm[threadIdx.x][i];
    part[threadIdx.x * g + lb] = s;
  }
}
// Sums of a launch's partials, in the same order in every workgroup: a wave
// takes a whole sum.  In two steps: the loads of the first need nothing but the
// kernel's arguments, so they run beside those of the state.
template <int NV>
__device__ __forceinline__ void group_begin(const double *part, int g, double (&a)[NV]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = w + i * nw;
    a[i] = 0.0;
    if (k < NV)
      for (int b = lane; b < g; b += 64) a[i] += part[k * g + b];
  }
}
template <int NV>
__device__ __forceinline__ void group_end(double (&a)[NV], double (&v)[NV]) {
  __shared__ double sm[NV];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int k = w + i * nw;
    if (k < NV) {
      const double s = wave_sum63(a[i]);
      if (lane == 63) sm[k] = s;
    }
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NV; ++k) v[k] = sm[k];
}
template <int NV>
__device__ __forceinline__ void group_reduce(const double *part, int g, double (&v)[NV]) {
  double a[NV];
  group_begin<NV>(part, g, a);
  group_end<NV>(a, v);
}
template <int NV>
__device__ __forceinline__ void group_partials(double (&v)[NV], double *part) {
  group_partials<NV>(v, part, (int)gridDim.x, (int)blockIdx.x);
}

// Sums of a pass.
enum { kSumMu = 0, kSumDelta = 1, kSumGamma = 2, kSumNu = 3, kSumRr = 4, kSumPp = 5, kSums = 6 };

// alpha and beta from the sums of the pass before; `lead` notes them in the next state
__device__ __forceinline__ void pr_scalars(const double (&red)[kSums], bool lead, CgState &next, double &alpha,
                                           double &beta) {
  const double nu = red[kSumNu];
  alpha = red[kSumMu] != 0.0 ? nu / red[kSumMu] : 0.0;   // cg.f90:195-199
  const double pred = __builtin_fma(alpha, __builtin_fma(alpha, red[kSumGamma], -2.0 * red[kSumDelta]), nu);
  beta = nu != 0.0 ? pred / nu : 0.0;
  if (lead) {
    next.alpha = alpha;
    next.pap = red[kSumMu];
    next.pp = red[kSumPp];
  }
}

// The vectors that alternate between two sets: pass `par` reads set par.
template <typename T>
struct PairOf {
  T *v[2];
};

// Residuals of x in FP64, r = b - A x, for what mode asks.
enum { kLatInit64 = 0,   // r64; partials <r,z>, ||r||^2, ||b||^2, <b,Mb>
       kLatInit32 = 1,   // r32 = S r, d = 0; partials <r32,r32>, ||r||^2, ||b||^2, <r32,r32>
       kLatTrue = 2,     // partial ||r||^2 (reporting only)
       kLatUpdate = 3 }; // r32 = S r; partials <r32,r32>, ||r||^2

struct IoRes {
  static constexpr int kKeep = 1, kAhead3 = 1;
  struct Raw {
    double x;
  };
  using Halo = Raw;
  const double *__restrict__ x, *__restrict__ b, *__restrict__ invd;
  const double *__restrict__ sc;
  double *__restrict__ r64;
  float *__restrict__ r32, *__restrict__ d32;
  int mode;
  double acc[4];
  BufRsrc xb;
  double scale = 1.0;        // S r = sc r, or scale r without sc
  __device__ __forceinline__ bool ready() const { return true; }
  __device__ __forceinline__ Raw fetch(uint32_t o) const { return Raw{buf_ld64(xb, o)}; }
  __device__ __forceinline__ Halo halo(uint32_t o) const { return fetch(o); }
  __device__ __forceinline__ double halo_value(const Halo &w) const { return w.x; }
  __device__ __forceinline__ double value(const Raw &w, uint32_t, double (&)[kKeep]) const {
    return w.x;
  }
  template <bool FULL>
  __device__ __forceinline__ void out(uint32_t o, const double (&)[kKeep], double y) {
    if (o < kNoPlane) row((int)(o >> 3), y);
  }
  __device__ __forceinline__ void row(int i, double y) {
    const double bi = b[i], ri = bi - y;
    if (mode == kLatTrue) {
      acc[0] += ri * ri;
    } else if (mode == kLatInit64) {
      const double di = invd ? invd[i] : 1.0;
      r64[i] = ri;
      acc[0] += ri * (di * ri);
      acc[1] += ri * ri;
      acc[2] += bi * bi;
      acc[3] += bi * (di * bi);
    } else {
      const float rf = (float)(sc ? sc[i] * ri : scale * ri);
      r32[i] = rf;
      const double rr = (double)rf * (double)rf;
      acc[0] += rr;
      acc[1] += ri * ri;
      if (mode == kLatInit32) {
        d32[i] = 0.0f;
        acc[2] += bi * bi;
        acc[3] += rr;
      }
    }
  }
};

// What a pass of the FP32 one-launch form does, from its state and the sums of
// the pass before (group_begin): an iteration with alpha and beta, the fold of a
// reliable update, or nothing more.  `lead` writes the next state.
enum { kRfGo, kRfFold, kRfDone };
__device__ __forceinline__ int rf_begin(const CgState &cur, CgState &next, bool lead, double (&sums)[kSums],
                                        CgResult *R, double &alpha, double &beta) {
  const int other = cur.set ^ 1;
  alpha = beta = 0.0;
  if (cur.first == 1) {   // p = r
    if (lead) {
      next = cur;
      next.first = 2;
      next.set = other;
    }
    return kRfGo;
  }
  double red[kSums];
  group_end<kSums>(sums, red);
  if (cur.ru == 2) {
    const double rd[2] = {red[0], red[1]};
    const RfStep step = rf_decide(cur, rd, lead, next, R);   // FP64 stopping test, beta
    if (lead) {
      next.first = 2;
      next.set = other;
    }
    beta = step.beta;
    return step.done ? kRfDone : kRfGo;
  }
  const double rd[2] = {red[kSumNu], 0.0};
  if (cur.first == 2) {   // no iteration made since the direction was set
    if (lead) {
      next = cur;
      next.first = 0;
      next.rz = red[kSumNu];
    }
  } else if (rf_decide(cur, rd, lead, next, R).fold) {   // back to the set of the direction before last
    if (lead) {
      next.ru = 1;
      next.set = other;
    }
    return kRfFold;
  }
  pr_scalars(red, lead, next, alpha, beta);
  if (lead) next.set = other;
  return kRfGo;
}

// FP32 passes of the one-launch form: p, r, s are those of the scaled system S A S (sc = S in FP64,
// null: S = I), d the increment in its variables.  begin(alpha, beta) takes the
// pass's decision once the first loads are under way; false: no iteration.
template <class Begin>
struct IoRf {
  static constexpr int kKeep = 3;
  static constexpr int kAhead3 = 2;   // 40.6 against 42.0 us an iteration at 128^3, 32.4 against 35.9 with a cell field
  struct Halo {
    double s;
    float r, q, p;
  };
  struct Raw : Halo {
    float d;
  };
  BufRsrc r, q, sc, p, rn, qn, pn, d;   // q = S A S p; q and p have no bytes in the first pass: read as 0
  bool jac;
  Begin begin;
  float alpha, beta;
  double sum[kSums];
  __device__ __forceinline__ bool ready() {
    double a = 0.0, b = 0.0;
    const bool go = begin(a, b);
    alpha = (float)a;
    beta = (float)b;
    return go;
  }
  __device__ __forceinline__ Raw fetch(uint32_t o) const {
    return Raw{halo(o), buf_ld32(d, o)};
  }
  __device__ __forceinline__ Halo halo(uint32_t o) const {
    return Halo{jac ? buf_ld64(sc, o) : 1.0, buf_ld32(r, o), buf_ld32(q, o), buf_ld32(p, o)};
  }
  __device__ __forceinline__ double halo_value(const Halo &w) const {
    return w.s * (double)dir_value(beta, w.p, __builtin_fmaf(-alpha, w.q, w.r));
  }
  __device__ __forceinline__ double value(const Raw &w, uint32_t o, double (&keep)[kKeep]) {
    const float ri = __builtin_fmaf(-alpha, w.q, w.r), pi = dir_value(beta, w.p, ri);
    buf_st32(rn, o, ri);
    buf_st32(pn, o, pi);
    buf_st32(d, o, __builtin_fmaf(alpha, w.p, w.d));
    const double rm = o < kNoPlane ? (double)ri : 0.0;   // 0 where a neighbour owns the node
    sum[kSumNu] += rm * rm;
    const double u = w.s * (double)pi;
    keep[0] = u;
    keep[1] = (double)ri;
    keep[2] = w.s;
    return u;
  }
  template <bool FULL>
  __device__ __forceinline__ void out(uint32_t o, const double (&keep)[kKeep], double y) {
    const double si = FULL ? keep[2] : jac ? buf_ld64(sc, o) : 1.0;
    const double ri = FULL ? keep[1] : (double)buf_ld32(rn, o);
    const float qi = (float)(si * y);
    buf_st32(qn, o, qi);
    const double ym = o < kNoPlane ? y : 0.0, qm = o < kNoPlane ? (double)qi : 0.0;
    sum[kSumMu] += keep[0] * ym;
    sum[kSumDelta] += ri * qm;
    sum[kSumGamma] += qm * qm;
  }
};

}  // namespace
}  // namespace femhip
