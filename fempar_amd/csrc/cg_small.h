// cg_small.h -- CG iterations of small systems in one workgroup; included by
// cg.hip inside its namespaces.
//
// Up to kSmallMaxRows rows an iteration in three launches is launch latency
// (14 us, whatever the product costs).  One workgroup holds such a system: the
// direction, x and M in LDS, r in registers, and the values of a symmetric
// stencil in registers too where they fit (R rows a thread, KP stored
// diagonals).  8 waves then: each repeats an iteration's two workgroup sums and
// its scalars (250 of 350 instructions at 961 rows), but fewer leave the LDS
// latency open (us an iteration at 961 / 3969 rows of 9 values with 4, 8 and 16
// waves: 2.1 / 8, 1.8 / 3.6, 2.2 / 4.4).  Other layouts are streamed from the L2
// each iteration, by 16 waves for the loads in flight.  A launch runs up to
// `count` iterations.  Products sum a row's terms in the order of slice_rows, so
// rows round as in k_spmv.  32 x 32 Q1 with assembly and download: 0.93 ms, now
// 0.26.

constexpr int32_t kSmallMaxRows = 4096;
constexpr int kSmallChunk = 1024;                     // iterations a launch

// Row `lane` of slice s as in slice_rows, its terms in the same order, x in LDS
// (without that one's special cases, which hold more loads than fit here).
__device__ __forceinline__ double small_row(const SlicedDev &m, const double *__restrict__ v, const double *x, int s, int lane) {
  const int hi = m.n - 1;
  int row = s * kSlice + lane;
  asm volatile("" : "+v"(row));
  double acc = 0.0;
  if (m.sym) {
    const double *vv = v + row;
#pragma unroll 14
    for (int k = 0; k < m.kplus; ++k) acc += vv[(int64_t)k * m.stride] * x[min(row + m.soffs[k], hi)];
#pragma unroll 13
    for (int k = 1; k < m.kplus; ++k) {
      const int rr = row - m.soffs[k], rc = min(max(rr, 0), hi);
      const double a = v[sym_at(k, rc, m.stride, m.kplus)];
      acc += (rr < 0 ? 0.0 : a) * x[rc];
    }
    return acc;
  }
  const int meta = m.meta[s], K = meta & 0x0fffffff;
  const double *vv = v + m.base[s] + lane;
  if (!(meta >> 30)) {
    const int32_t *off = m.offs + m.aux[s];
#pragma unroll 8
    for (int k = 0; k < K; ++k) acc += vv[k * kSlice] * x[min(max(row + off[k], 0), hi)];
  } else {
    const int32_t *ec = m.ecol + m.aux[s] + lane;
#pragma unroll 8
    for (int k = 0; k < K; ++k) acc += vv[k * kSlice] * x[ec[k * kSlice]];
  }
  return acc;
}

// LDS: p between two margins of zeros (KP > 0: the largest offset; columns past
// the ends need no clamping, their values are 0), x, M.
__host__ __device__ constexpr size_t small_lds(int32_t n, int32_t margin) { return sizeof(double) * ((size_t)3 * n + 2 * (size_t)margin); }

template <int T, int R, int KP>
__global__ __launch_bounds__(T) void k_cg_small(SlicedDev m, const double *__restrict__ v,
                                                            double *__restrict__ gr, double *__restrict__ gx,
                                                            double *__restrict__ gp, const double *__restrict__ invd,
                                                            CgState *S, int margin, int count, double *hist,
                                                            CgResult *Res, CgResult *Rh) {
  extern __shared__ double small_mem[];
  __shared__ double sums[4][T / 64];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), n = m.n;
  const bool lead = tid == 0;
  double *p = small_mem + margin, *x = p + n + margin, *d = x + n;
  constexpr int KC = KP > 0 ? KP : 1;
  int o[KC];
  double up[R][KC], low[R][KC], r[R];
  int row[R];
  CgState cur;   // every thread's, the same; field by field, so that it stays in registers
  cur.rz = S->rz;
  cur.rnrm_m = S->rnrm_m;
  cur.alpha = cur.pap = cur.pp = cur.beta = 0.0;
  cur.rhs_test = S->rhs_test;
  cur.rhs_extra = S->rhs_extra;
  cur.est = S->est;
  cur.rnorm = S->rnorm;
  cur.rtol = S->rtol;
  cur.atol = S->atol;
  cur.iter = S->iter;
  cur.done = S->done;
  cur.converged = S->converged;
  cur.maxit = S->maxit;
  cur.crit = S->crit;
  for (int i = tid; i < margin; i += T) p[-1 - i] = p[n + i] = 0.0;
  if constexpr (KP > 0)
#pragma unroll
    for (int k = 0; k < KP; ++k) o[k] = m.soffs[k];
#pragma unroll
  for (int j = 0; j < R; ++j) {
    const int s = w + j * (T / 64);
    row[j] = s < m.ns ? slice_row_index(m, s, lane) : n;
    const bool on = row[j] < n;
    const int i = on ? row[j] : 0;
    r[j] = on ? gr[i] : 0.0;
    if (on) {
      p[i] = gp[i];
      x[i] = gx[i];
      d[i] = invd ? invd[i] : 1.0;
    }
    if constexpr (KP > 0)
#pragma unroll
      for (int k = 0; k < KP; ++k) {
        up[j][k] = on ? v[sym_at(k, i, m.stride, KP)] : 0.0;
        low[j][k] = on && i >= o[k] ? v[sym_at(k, i - o[k], m.stride, KP)] : 0.0;
      }
  }
  __syncthreads();
  for (int c = 0; c < count; ++c) {
    if (__builtin_amdgcn_readfirstlane(cur.done)) break;
    if constexpr (KP > 0)
#pragma unroll
      for (int k = 0; k < KP; ++k) asm volatile("" : "+s"(o[k]));   // no address is kept from pass to pass: registers
    double q[R], a2[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < R; ++j) {
      q[j] = 0.0;
      const int s = w + j * (T / 64);
      if (s >= m.ns) continue;
      double y = 0.0;
      const bool on = row[j] < n;
      const int i = on ? row[j] : 0;
      if constexpr (KP > 0) {
#pragma unroll
        for (int k = 0; k < KP; ++k) y += up[j][k] * p[i + o[k]];
#pragma unroll
        for (int k = 1; k < KP; ++k) y += low[j][k] * p[i - o[k]];
      } else {
        y = small_row(m, v, p, s, lane);
      }
      if (on) {
        q[j] = y;
        const double pi = p[i];
        a2[0] += pi * y;
        a2[1] += pi * pi;
      }
    }
    block_sums<T / 64>(a2, sums);
    const double alpha = a2[0] != 0.0 ? cur.rz / a2[0] : 0.0;   // cg.f90:195-199
    cur.alpha = alpha;
    cur.pap = a2[0];
    cur.pp = a2[1];
    double b2[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (row[j] < n) {
        r[j] = r[j] + (-alpha) * q[j];
        b2[0] += r[j] * (d[row[j]] * r[j]);
        b2[1] += r[j] * r[j];
      }
    block_sums<T / 64>(b2, sums + 2);
    const double rnorm = sqrt(b2[1]), beta = (1.0 / cur.rz) * b2[0];
    double est, rhs_test;
    cur.converged = cg_test(cur, ++cur.iter, b2, rnorm, est, rhs_test);
    cur.est = est;
    cur.rhs_test = rhs_test;
    cur.rnorm = rnorm;
    cur.done = cur.converged || cur.iter >= cur.maxit;
    cur.beta = beta;
    cur.rz = b2[0];
    cur.rnrm_m = sqrt(b2[0]);
    if (lead && hist) hist[cur.iter - 1] = est;
    const int done = __builtin_amdgcn_readfirstlane(cur.done);
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (row[j] < n) {
        const double pi = p[row[j]];
        x[row[j]] = x[row[j]] + alpha * pi;
        if (!done) p[row[j]] = d[row[j]] * r[j] + beta * pi;
      }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (row[j] < n) {
      gr[row[j]] = r[j];
      gx[row[j]] = x[row[j]];
      gp[row[j]] = p[row[j]];
    }
  if (lead) {
    if (cur.iter > 0) {
      S->rz = cur.rz;
      S->rnrm_m = cur.rnrm_m;
      S->est = cur.est;
      S->rhs_test = cur.rhs_test;
      S->rnorm = cur.rnorm;
      S->iter = cur.iter;
      S->done = cur.done;
      S->converged = cur.converged;
      Res->iter = cur.iter;
      Res->est = cur.est;
      Res->rhs_test = cur.rhs_test;
      Res->rnorm = cur.rnorm;
      Res->converged = cur.converged;
      Res->done = cur.done;
      Res->prog = cur.est;
      Res->prog_it = cur.iter;
    }
    if (Rh) *Rh = *Res;
  }
}

// Values an iteration may stream: one CU reads about 12 an ns.  Sliced layouts:
// 12 against 39 us an iteration at 22,000 values (3-D Q2), 13 against 25 at 71,000
// (elasticity), 26 each at 157,000.  Symmetric stencils read every value twice, with an
// address of its own: 11.3 against 14.5 us at 48,000, 18 against 15 at 94,000.
constexpr int64_t kSmallEntries = 110000, kSmallEntriesSym = 65000;
using SmallKernel = void (*)(SlicedDev, const double *, double *, double *, double *, const double *, CgState *, int, int,
                             double *, CgResult *, CgResult *);
// The kernel and its launch for a layout of n rows; fn is null where the
// three-launch iterations are faster.
struct SmallCg {
  SmallKernel fn = nullptr;
  int threads = 0, margin = 0;
  size_t lds = 0;
};
inline SmallCg small_cg(const Sliced &sl, int32_t n) {
  SmallCg c;
  if (n < 1 || n > kSmallMaxRows) return c;
  constexpr int T = 512;
  const int r = (sl.ns + T / 64 - 1) / (T / 64);   // rows a thread
  if (sl.sym && sl.kplus == 5)
    c.fn = r <= 1 ? k_cg_small<T, 1, 5> : r <= 2 ? k_cg_small<T, 2, 5> : r <= 4 ? k_cg_small<T, 4, 5> : k_cg_small<T, 8, 5>;
  else if (sl.sym && sl.kplus == 14 && r <= 4)
    c.fn = r <= 1 ? k_cg_small<T, 1, 14> : r <= 2 ? k_cg_small<T, 2, 14> : k_cg_small<T, 4, 14>;
  if (c.fn) {
    c.threads = T;
    c.margin = sl.h_soffs.back();
    c.lds = small_lds(n, c.margin);
    if (c.lds <= 150 * 1024) return c;
  }
  c = SmallCg{};
  if (sl.sym ? 2 * sl.entries > kSmallEntriesSym : sl.entries > kSmallEntries) return c;
  c.fn = sl.ns <= 16 ? k_cg_small<1024, 1, 0> : sl.ns <= 32 ? k_cg_small<1024, 2, 0> : k_cg_small<1024, 4, 0>;
  c.threads = 1024;
  c.lds = small_lds(n, 0);
  return c;
}
