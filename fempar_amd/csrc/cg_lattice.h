// cg_lattice.h -- CG kernels on the lattice products (lattice.h); included by
// cg.hip inside its namespaces, after the scalar state and the decisions.
//
// Two forms of an iteration, chosen by size (lattice_one):
//
// Two launches, the form of cg.f90:101-238:
//   A: stopping test, x += alpha p, p = z + beta p and s = A p in one march over
//      the cells (a node next to a workgroup's tile is formed by both
//      neighbours, so p alternates between two vectors); partials <p,s>, ||p||^2
//   B: r -= alpha s; partials <r,z>, ||r||^2
// FP64, a row and iteration: 56 B in A (r, M, p, x in; p, x, s out), 32 B in B,
// against 128 B (Q1) to 1000 B (Q2) for the product with a stored matrix and 80 B
// of vector passes in two more launches.
//
// One launch, the predict-and-recompute form (Chen and Carson, SIAM J. Sci.
// Comput. 42, 2020): every sum an iteration needs is taken in one pass.  With
// M = diag(A)^-1, s = A p and the sums of the pass before
//   mu = <p,s>, delta = <Mr,s>, gamma = <s,Ms>, nu = <r,Mr>
// a pass forms alpha = nu / mu, predicts the next nu as
// nu - 2 alpha delta + alpha^2 gamma, beta = that / nu, and then
//   r -= alpha s ; x += alpha p ; p = M r + beta p ; s = A p
// in one march, with the sums of the new vectors (nu itself is summed again, only
// beta uses its prediction).  The vectors, and so the attainable accuracy, are
// those of the two-launch form: against long double at 20^3, alpha ||p|| after 39
// iterations is off by 1.4e-8 (two reductions: 1.0e-8, the sequential sums of the
// oracle: 9.7e-8).  72 B a row, and r and s alternate too; it saves a launch and
// its wait, but its march holds twice the vectors in flight, and where memory
// bounds it the two launches' 88 B in smaller workgroups are as fast.
//
// The FP32 iterations keep FP32 vectors of the scaled system S A S, but their
// products are formed in FP64 from the same coefficients as the FP64 ones: only
// the vectors round.

template <int DIM, int P, int KIND>
using LatticeCell = std::conditional_t<KIND == kElastic, CellElastic, std::conditional_t<P == 1, CellQ1<DIM, KIND>, CellQ2<DIM, KIND>>>;

template <int DIM, int P, int KIND>
__device__ __forceinline__ LatticeCell<DIM, P, KIND> lattice_cell(const CoefDev &c, const Q2Tab &t) {
  LatticeCell<DIM, P, KIND> cell;
  cell.k = c;
  if constexpr (P == 2) cell.t = t;
  return cell;
}

struct IoCg {
  static constexpr int kKeep = 3, kAhead3 = 1;
  struct Halo {
    double r, s, d, p;
  };
  struct Raw : Halo {
    double x;
  };
  const CgState &cur;
  CgState &next;
  double (&part_in)[kSums];   // of group_begin
  double *hist;
  CgResult *R, *Rh;
  BufRsrc r, s, invd, p, rn, sn, pn, x;   // s and p have no bytes in the first pass: read as 0
  bool jac;
  double alpha, beta;
  double sum[kSums];

  __device__ __forceinline__ Raw fetch(uint32_t o) const {
    return Raw{halo(o), buf_ld64(x, o)};
  }
  __device__ __forceinline__ Halo halo(uint32_t o) const {
    return Halo{buf_ld64(r, o), buf_ld64(s, o), jac ? buf_ld64(invd, o) : 1.0, buf_ld64(p, o)};
  }
  __device__ __forceinline__ double halo_value(const Halo &w) const {
    return __builtin_fma(beta, w.p, w.d * __builtin_fma(-alpha, w.s, w.r));
  }
  // the stopping test on the last pass's residual, and this pass's scalars
  __device__ __forceinline__ bool ready() {
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    alpha = beta = 0.0;
    if (cur.first == 1) {   // p = M r, s = A p
      if (lead) {
        next = cur;
        next.first = 2;
        if (Rh) *Rh = *R;
      }
      return true;
    }
    double red[kSums];
    group_end<kSums>(part_in, red);
    if (cur.first == 2) {   // no iteration made yet
      if (lead) {
        next = cur;
        next.first = 0;
        if (Rh) *Rh = *R;
      }
    } else {
      const double rd[2] = {red[kSumNu], red[kSumRr]};
      double unused;
      if (cg_decide(cur, rd, lead, next, hist, R, Rh, unused)) return false;
    }
    pr_scalars(red, lead, next, alpha, beta);
    return true;
  }
  __device__ __forceinline__ double value(const Raw &w, uint32_t o, double (&keep)[kKeep]) {
    const double ri = __builtin_fma(-alpha, w.s, w.r), zi = w.d * ri, u = __builtin_fma(beta, w.p, zi);
    buf_st64(rn, o, ri);
    buf_st64(pn, o, u);
    buf_st64(x, o, __builtin_fma(alpha, w.p, w.x));
    const double rm = o < kNoPlane ? ri : 0.0, um = o < kNoPlane ? u : 0.0;   // 0 where a neighbour owns the node
    sum[kSumNu] += rm * zi;
    sum[kSumRr] += rm * ri;
    sum[kSumPp] += um * u;
    keep[0] = u;
    keep[1] = zi;
    keep[2] = w.d;
    return u;
  }
  template <bool FULL>
  __device__ __forceinline__ void out(uint32_t o, const double (&keep)[kKeep], double y) {
    buf_st64(sn, o, y);
    const double di = FULL ? keep[2] : jac ? buf_ld64(invd, o) : 1.0;
    const double zi = FULL ? keep[1] : di * buf_ld64(rn, o);
    const double ym = o < kNoPlane ? y : 0.0;
    sum[kSumMu] += keep[0] * ym;
    sum[kSumDelta] += zi * ym;
    sum[kSumGamma] += di * ym * y;
  }
};

#define FEMHIP_LATTICE_BOUNDS(ONE)                                         \
  __launch_bounds__(lattice_threads(DIM, P, KIND == kElastic ? 3 : 1, ONE), \
                    lattice_waves(DIM, P, KIND == kElastic ? 3 : 1, ONE))

template <int DIM, int P, int KIND>
__global__ FEMHIP_LATTICE_BOUNDS(true) void k_lat_cg(Lattice g, CoefDev c, Q2Tab t, int32_t n, PairOf<double> r,
                                               PairOf<double> s, PairOf<double> p, double *x, const double *invd,
                                               CgState *S, int par, const double *part_in, double *part_out,
                                               double *hist, CgResult *R, CgResult *Rh) {
  double sums_in[kSums];
  group_begin<kSums>(part_in, (int)gridDim.x, sums_in);
  const CgState &cur = S[par];
  if (cur.done) {   // keep `done` sticky in both parity slots
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      S[par ^ 1].done = 1;
      if (Rh) *Rh = *R;
    }
    return;
  }
  const uint32_t bytes = 8u * (uint32_t)n, old = cur.first == 1 ? 0 : bytes;
  IoCg io{cur, S[par ^ 1], sums_in, hist, R, Rh, buf_of(r.v[par], bytes), buf_of(s.v[par], old),
          buf_of(invd, invd ? bytes : 0), buf_of(p.v[par], old), buf_of(r.v[par ^ 1], bytes),
          buf_of(s.v[par ^ 1], bytes), buf_of(p.v[par ^ 1], bytes), buf_of(x, bytes), invd != nullptr,
          0.0, 0.0, {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}};
  auto cell = lattice_cell<DIM, P, KIND>(c, t);
  lattice_march<DIM, P>(g, lattice_block(g), cell, io, lattice_smem);
  group_partials<kSums>(io.sum, part_out);
}

template <int DIM, int P, int KIND>
__global__ FEMHIP_LATTICE_BOUNDS(true) void k_lat_res(Lattice g, CoefDev c, Q2Tab t, int32_t n, int mode, int x_zero,
                                                const double *__restrict__ x, const double *__restrict__ b,
                                                const double *__restrict__ invd, const double *__restrict__ sc,
                                                double *__restrict__ r64, float *__restrict__ r32,
                                                float *__restrict__ d32, double *part) {
  IoRes io{x, b, invd, sc, r64, r32, d32, mode, {0.0, 0.0, 0.0, 0.0}, buf_of(x, 8u * (uint32_t)n)};
  if (x_zero) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) io.row((int)i, 0.0);
  } else {
    auto cell = lattice_cell<DIM, P, KIND>(c, t);
    lattice_march<DIM, P>(g, lattice_block(g), cell, io, lattice_smem);
  }
  if (mode == kLatTrue) {
    double out[1] = {io.acc[0]};
    group_partials<1>(out, part);
  } else {
    group_partials<4>(io.acc, part);
  }
}

// A slot of the FP32 path: a CG pass, or one of a reliable update's two (state
// ru): the slot that finds an update due folds the increment into the FP64
// solution (x += S d, d = 0); the next one replaces r by the FP64 residual of
// the folded x (ru = 1); the one after tests it and takes the direction from it
// and the direction before last (ru = 2), which is still in the other set.
template <int DIM, int P, int KIND>
__global__ FEMHIP_LATTICE_BOUNDS(true) void k_lat_rf(Lattice g, CoefDev c, Q2Tab t, int32_t n, PairOf<float> r,
                                               PairOf<float> q, PairOf<float> p, float *d, double *__restrict__ x,
                                               const double *__restrict__ b, const double *__restrict__ sc, CgState *S,
                                               int par, const double *part_in, double *part_out, CgResult *R,
                                               CgResult *Rh) {
  double sums_in[kSums];   // after an update pass only the first two count
  group_begin<kSums>(part_in, (int)gridDim.x, sums_in);
  const CgState &cur = S[par];
  CgState &next = S[par ^ 1];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (cur.done) {   // keep `done` sticky in both parity slots
    if (lead) {
      next.done = 1;
      if (Rh) *Rh = *R;
    }
    return;
  }
  const int set = cur.set;
  const uint32_t b4 = 4u * (uint32_t)n, b8 = 8u * (uint32_t)n;
  if (cur.ru == 1) {
    if (lead) {
      next = cur;
      next.ru = 2;
      if (Rh) *Rh = *R;
    }
    IoRes io{x, b, nullptr, sc, nullptr, r.v[set], nullptr, kLatUpdate, {0.0, 0.0, 0.0, 0.0}, buf_of(x, b8)};
    auto cell = lattice_cell<DIM, P, KIND>(c, t);
    lattice_march<DIM, P>(g, lattice_block(g), cell, io, lattice_smem);
    double out[2] = {io.acc[0], io.acc[1]};
    group_partials<2>(out, part_out);
    return;
  }
  int act = kRfGo;
  auto begin = [&](double &alpha, double &beta) {
    act = rf_begin(cur, next, lead, sums_in, R, alpha, beta);
    if (lead && Rh) *Rh = *R;
    return act == kRfGo;
  };
  const uint32_t old = cur.first == 1 ? 0 : b4;
  IoRf<decltype(begin)> io{buf_of(r.v[set], b4), buf_of(q.v[set], cur.ru == 2 ? 0 : old), buf_of(sc, sc ? b8 : 0),
                           buf_of(p.v[set], old), buf_of(r.v[set ^ 1], b4), buf_of(q.v[set ^ 1], b4),
                           buf_of(p.v[set ^ 1], b4), buf_of(d, b4), sc != nullptr, begin, 0.0f, 0.0f,
                           {0.0, 0.0, 0.0, 0.0, 0.0, 0.0}};
  auto cell = lattice_cell<DIM, P, KIND>(c, t);
  if (!lattice_march<DIM, P>(g, lattice_block(g), cell, io, lattice_smem)) io.ready();   // no cells: the decision all the same
  if (act == kRfFold) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
      x[i] = new_x(x[i], d[i], sc, i);
      d[i] = 0.0f;
    }
  }
  if (act != kRfGo) return;
  group_partials<kSums>(io.sum, part_out);
}

// ---- two launches an iteration ----

struct IoCgA {
  static constexpr int kKeep = 1, kAhead3 = 1;
  struct Halo {
    double r, d, p;
  };
  struct Raw : Halo {
    double x;
  };
  const CgState &cur;
  CgState &next;
  const double *part_in;
  double *hist;
  CgResult *R, *Rh;
  BufRsrc r, invd, p, pn, x, q;   // p has no bytes in the first pass: reads as 0
  bool jac, done;
  int groups;
  double alpha, beta, pq, pp;
  __device__ __forceinline__ Halo halo(uint32_t o) const {
    return Halo{buf_ld64(r, o), jac ? buf_ld64(invd, o) : 1.0, buf_ld64(p, o)};
  }
  __device__ __forceinline__ Raw fetch(uint32_t o) const { return Raw{halo(o), buf_ld64(x, o)}; }
  __device__ __forceinline__ bool ready() {
    const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
    alpha = beta = 0.0;
    if (cur.first) {   // p = M r
      if (lead) {
        next = cur;
        next.first = 0;
        if (Rh) *Rh = *R;
      }
      return true;
    }
    double red[2];
    group_reduce<2>(part_in, groups, red);
    alpha = cur.alpha;
    done = cg_decide(cur, red, lead, next, hist, R, Rh, beta);
    return !done;
  }
  __device__ __forceinline__ double halo_value(const Halo &w) const { return __builtin_fma(beta, w.p, w.d * w.r); }
  __device__ __forceinline__ double value(const Raw &w, uint32_t o, double (&keep)[kKeep]) const {
    const double u = halo_value(w);
    buf_st64(pn, o, u);
    buf_st64(x, o, __builtin_fma(alpha, w.p, w.x));
    keep[0] = u;
    return u;
  }
  template <bool FULL>
  __device__ __forceinline__ void out(uint32_t o, const double (&keep)[kKeep], double y) {
    buf_st64(q, o, y);
    const double u = o < kNoPlane ? keep[0] : 0.0;
    pq += u * y;
    pp += u * u;
  }
};

template <int DIM, int P, int KIND>
__global__ FEMHIP_LATTICE_BOUNDS(false) void k_lat_a(Lattice g, CoefDev c, Q2Tab t, int32_t n, const double *r,
                                              const double *invd, PairOf<double> p, double *x, double *q, CgState *S,
                                              int par, const double *part_b, int gb, double *part, double *hist,
                                              CgResult *R, CgResult *Rh) {
  const CgState &cur = S[par];
  if (cur.done) {   // keep `done` sticky in both parity slots
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      S[par ^ 1].done = 1;
      if (Rh) *Rh = *R;
    }
    return;
  }
  const uint32_t bytes = 8u * (uint32_t)n;
  IoCgA io{cur, S[par ^ 1], part_b, hist, R, Rh, buf_of(r, bytes), buf_of(invd, invd ? bytes : 0),
           buf_of(p.v[par], cur.first ? 0 : bytes), buf_of(p.v[par ^ 1], bytes), buf_of(x, bytes), buf_of(q, bytes),
           invd != nullptr, false, gb, 0.0, 0.0, 0.0, 0.0};
  auto cell = lattice_cell<DIM, P, KIND>(c, t);
  if (!lattice_march<DIM, P>(g, lattice_block(g), cell, io, lattice_smem)) io.ready();   // no cells: the decision all the same
  if (io.done) {   // the last iteration: x += alpha p
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const double *pold = p.v[par];
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
      x[i] = __builtin_fma(cur.alpha, pold[i], x[i]);
    return;
  }
  double out[2] = {io.pq, io.pp};
  group_partials<2>(out, part);
}

// r -= alpha q (two rows a load); partials <r,z>, ||r||^2
__global__ __launch_bounds__(kThreads) void k_lat_b(int32_t n, double *__restrict__ r, const double *__restrict__ q,
                                                    const double *__restrict__ invd, CgState *S, int par,
                                                    const double *part_a, int ga, double *part) {
  double red[2];
  partials_begin<2>(part_a, ga, red);
  if (S[par].done) return;
  constexpr int K = 4;   // pairs a thread loads before it reduces the partials
  const int64_t i0 = (int64_t)blockIdx.x * kThreads + threadIdx.x, stride = (int64_t)gridDim.x * kThreads;
  const int64_t np = n / 2;
  double2 rv[K], qv[K], dv[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int64_t i = i0 + k * stride;
    if (i < np) {
      rv[k] = reinterpret_cast<const double2 *>(r)[i];
      qv[k] = reinterpret_cast<const double2 *>(q)[i];
      dv[k] = invd ? reinterpret_cast<const double2 *>(invd)[i] : double2{1.0, 1.0};
    }
  }
  partials_end<2>(red);
  const double alpha = (red[0] != 0.0) ? S[par].rz / red[0] : 0.0;   // cg.f90:195-199
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    S[par].alpha = alpha;
    S[par].pap = red[0];
    S[par].pp = red[1];
  }
  double rz = 0.0, rr = 0.0;
  auto one = [&](double r0, double qi, double di) {
    const double ri = __builtin_fma(-alpha, qi, r0);
    rz += ri * (di * ri);
    rr += ri * ri;
    return ri;
  };
  auto pair = [&](int64_t i, const double2 &a, const double2 &b, const double2 &d) {
    reinterpret_cast<double2 *>(r)[i] = double2{one(a.x, b.x, d.x), one(a.y, b.y, d.y)};
  };
#pragma unroll
  for (int k = 0; k < K; ++k)
    if (i0 + k * stride < np) pair(i0 + k * stride, rv[k], qv[k], dv[k]);
  for (int64_t i = i0 + K * stride; i < np; i += stride)
    pair(i, reinterpret_cast<const double2 *>(r)[i], reinterpret_cast<const double2 *>(q)[i],
         invd ? reinterpret_cast<const double2 *>(invd)[i] : double2{1.0, 1.0});
  if ((n & 1) && i0 == 0) r[n - 1] = one(r[n - 1], q[n - 1], invd ? invd[n - 1] : 1.0);
  double out[2] = {rz, rr};
  group_partials<2>(out, part);
}

// FP32: p and r are those of the scaled system S A S (sc = S in FP64, null:
// S = I), d the increment in its variables.
struct IoRfA {
  static constexpr int kKeep = 2, kAhead3 = 1;
  struct Halo {
    double s;
    float r, p;
  };
  struct Raw : Halo {
    float d;
  };
  BufRsrc r, sc, p, pn, d, q;   // p has no bytes in the first pass: reads as 0
  float alpha, beta;            // alpha 0 where d does not move
  bool jac;
  double pq;
  __device__ __forceinline__ bool ready() const { return true; }
  __device__ __forceinline__ Halo halo(uint32_t o) const {
    return Halo{jac ? buf_ld64(sc, o) : 1.0, buf_ld32(r, o), buf_ld32(p, o)};
  }
  __device__ __forceinline__ Raw fetch(uint32_t o) const { return Raw{halo(o), buf_ld32(d, o)}; }
  __device__ __forceinline__ double halo_value(const Halo &w) const {
    return w.s * (double)dir_value(beta, w.p, w.r);
  }
  __device__ __forceinline__ double value(const Raw &w, uint32_t o, double (&keep)[kKeep]) const {
    const float pn_ = dir_value(beta, w.p, w.r);
    buf_st32(pn, o, pn_);
    buf_st32(d, o, w.d + alpha * w.p);
    keep[0] = w.s * (double)pn_;
    keep[1] = w.s;
    return keep[0];
  }
  template <bool FULL>
  __device__ __forceinline__ void out(uint32_t o, const double (&keep)[kKeep], double y) {
    const double si = FULL ? keep[1] : jac ? buf_ld64(sc, o) : 1.0;
    buf_st32(q, o, (float)(si * y));
    pq += (o < kNoPlane ? keep[0] : 0.0) * y;
  }
};

template <int DIM, int P, int KIND>
__global__ FEMHIP_LATTICE_BOUNDS(false) void k_lat_rf_a(Lattice g, CoefDev c, Q2Tab t, int32_t n, const float *r,
                                                 const double *sc, PairOf<float> p, float *d, float *q, double *x,
                                                 CgState *S, int par, const double *part_b, int gb, double *part,
                                                 CgResult *R, CgResult *Rh) {
  const CgState &cur = S[par];
  const bool lead = blockIdx.x == 0 && threadIdx.x == 0;
  if (cur.done) {   // keep `done` sticky in both parity slots
    if (lead) {
      S[par ^ 1].done = 1;
      if (Rh) *Rh = *R;
    }
    return;
  }
  double red[2] = {0.0, 0.0};
  if (!cur.first) group_reduce<2>(part_b, gb, red);
  const RfStep step = rf_decide(cur, red, lead, S[par ^ 1], R);
  if (lead && Rh) *Rh = *R;
  if (step.done) return;
  const float a = (float)cur.alpha;
  const float *pold = p.v[par];
  if (step.fold) {   // the next slot B recomputes the residual of the new x; p moves to the other vector
    float *pnew = p.v[par ^ 1];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
      const float pi = pold[i];
      x[i] = new_x(x[i], d[i] + a * pi, sc, i);
      d[i] = 0.0f;
      pnew[i] = pi;
    }
    return;
  }
  const uint32_t b4 = 4u * (uint32_t)n;
  IoRfA io{buf_of(r, b4), buf_of(sc, sc ? 2 * b4 : 0), buf_of(pold, cur.first ? 0 : b4), buf_of(p.v[par ^ 1], b4),
           buf_of(d, b4), buf_of(q, b4), step.upd_d ? a : 0.0f, (float)step.beta, sc != nullptr, 0.0};
  auto cell = lattice_cell<DIM, P, KIND>(c, t);
  lattice_march<DIM, P>(g, lattice_block(g), cell, io, lattice_smem);
  double out[1] = {io.pq};
  group_partials<1>(out, part);
}

// FP32 slot B: r -= alpha q (four rows a load), or after a fold the FP64 residual of the folded x
template <int DIM, int P, int KIND>
__global__ FEMHIP_LATTICE_BOUNDS(false) void k_lat_rf_b(Lattice g, CoefDev c, Q2Tab t, int32_t n, float *__restrict__ r,
                                                 const float *__restrict__ q, const double *__restrict__ sc,
                                                 const double *__restrict__ b, const double *__restrict__ x, CgState *S,
                                                 int par, const double *part_a, int ga, double *part) {
  CgState &st = S[par];
  if (st.done) return;
  if (st.ru) {
    IoRes io{x, b, nullptr, sc, nullptr, r, nullptr, kLatUpdate, {0.0, 0.0, 0.0, 0.0}, buf_of(x, 8u * (uint32_t)n)};
    auto cell = lattice_cell<DIM, P, KIND>(c, t);
    lattice_march<DIM, P>(g, lattice_block(g), cell, io, lattice_smem);
    double out[2] = {io.acc[0], io.acc[1]};
    group_partials<2>(out, part);
    return;
  }
  constexpr int K = 4;
  const int64_t i0 = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t)gridDim.x * blockDim.x;
  const int64_t np = n / 4;
  float4 rv[K], qv[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {   // in flight while the partials are reduced
    const int64_t i = i0 + k * stride;
    if (i < np) {
      rv[k] = reinterpret_cast<const float4 *>(r)[i];
      qv[k] = reinterpret_cast<const float4 *>(q)[i];
    }
  }
  double red[1];
  group_reduce<1>(part_a, ga, red);
  const double alpha = (red[0] != 0.0) ? st.rz / red[0] : 0.0;   // cg.f90:195-199
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st.alpha = alpha;
    st.pap = red[0];
  }
  const float a = (float)alpha;
  double rr = 0.0;
  auto one = [&](float r0, float qi) {
    const float ri = r0 + (-a) * qi;
    rr += (double)ri * (double)ri;
    return ri;
  };
  auto quad = [&](int64_t i, const float4 &u, const float4 &v) {
    reinterpret_cast<float4 *>(r)[i] = float4{one(u.x, v.x), one(u.y, v.y), one(u.z, v.z), one(u.w, v.w)};
  };
#pragma unroll
  for (int k = 0; k < K; ++k)
    if (i0 + k * stride < np) quad(i0 + k * stride, rv[k], qv[k]);
  for (int64_t i = i0 + K * stride; i < np; i += stride)
    quad(i, reinterpret_cast<const float4 *>(r)[i], reinterpret_cast<const float4 *>(q)[i]);
  if (i0 < n - 4 * np) r[4 * np + i0] = one(r[4 * np + i0], q[4 * np + i0]);
  double out[2] = {rr, 0.0};
  group_partials<2>(out, part);
}

// k_jacobi into lattice order (perm null: the operator's rows are the lattice's)
__global__ void k_lat_jacobi(int32_t n, const int32_t *__restrict__ rowptr, const int32_t *__restrict__ col,
                             const double *__restrict__ val, const int32_t *__restrict__ perm,
                             double *__restrict__ out, int root, int *flag) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int32_t lo = rowptr[i], hi = rowptr[i + 1] - 1;
  double d = 0.0;
  while (lo <= hi) {
    const int32_t mid = (lo + hi) >> 1;
    const int32_t c = col[mid];
    if (c == i) {
      d = val[mid];
      break;
    }
    if (c < i) lo = mid + 1;
    else hi = mid - 1;
  }
  jacobi_store(d, root, out, perm ? perm[i] : i, flag);
}

// the same from a diagonal held as such (operators without a CSR)
__global__ void k_jacobi_diag(int32_t n, const double *__restrict__ diag, double *__restrict__ out, int root,
                              int *flag) {
  const int32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) jacobi_store(diag[i], root, out, i, flag);
}

struct LatticeKernels {
  decltype(&k_lat_a<3, 1, 0>) a;
  decltype(&k_lat_rf_a<3, 1, 0>) rf_a;
  decltype(&k_lat_rf_b<3, 1, 0>) rf_b;
  decltype(&k_lat_cg<3, 1, 0>) cg;
  decltype(&k_lat_rf<3, 1, 0>) rf;
  decltype(&k_lat_res<3, 1, 0>) res;
};
template <int DIM, int P, int KIND>
constexpr LatticeKernels lattice_kernels_of() {
  return {k_lat_a<DIM, P, KIND>, k_lat_rf_a<DIM, P, KIND>, k_lat_rf_b<DIM, P, KIND>, k_lat_cg<DIM, P, KIND>, k_lat_rf<DIM, P, KIND>, k_lat_res<DIM, P, KIND>};
}
template <int DIM, int P>
LatticeKernels lattice_kernels_by_kind(int kind) {
  return kind == kCoefCell ? lattice_kernels_of<DIM, P, kCoefCell>()
         : kind == kCoefSin3 ? lattice_kernels_of<DIM, P, kCoefSin3>() : lattice_kernels_of<DIM, P, kCoefPoint>();
}
LatticeKernels lattice_kernels(int dim, int order, int kind) {
  if (kind == kElastic) return lattice_kernels_of<3, 1, kElastic>();
  if (dim == 2) return order == 1 ? lattice_kernels_by_kind<2, 1>(kind) : lattice_kernels_by_kind<2, 2>(kind);
  return order == 1 ? lattice_kernels_by_kind<3, 1>(kind) : lattice_kernels_by_kind<3, 2>(kind);
}
