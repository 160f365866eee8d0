// Jacobi-preconditioned CG (hmholtz.f:611-846 CGGO) and its helpers
// (hmholtz.f:527-609 CHKTCG1, :380-524 SETPREC), all data resident on the GPU.
//
// One CG iteration of the reference,
//     z = r*d ; rtz1 = (z,r)_mult ; rbn2 = sqrt((r,r)_{binv*mult}/vol)
//     exit test ; beta ; p = z + beta p ; w = A p ; dssum(w) ; w *= mask
//     rho = (w,p)_mult ; alpha ; x += alpha p ; r -= alpha w
// runs as three launches:
//     k_cg_update_dots : x/r update of the previous iteration + both dots;
//                        in its last block the exit test and beta
//     axhelm (MODE 1)  : p update fused in, w = A_L p, rho = sum p.w
//     gs_assemble_step : w <- mask * dssum(w); in a block of its own alpha
// (With the two scalar steps as kernels of their own 336 elements, lx1 8, took
// 420 us a solve, now 347; 1.68e7 nodes 7250, now 7180.)
// rho is taken before the assembly: with p continuous and zero where the
// mask is, and mult summing to one over each group of shared nodes,
// (mask*QQ^T w, p)_mult = sum_l p_l w_l exactly in exact arithmetic.  The
// solve checks those conditions once and otherwise runs the unfused
// sequence (axhelm, dssum, mask, dot).
// Scalars stay on the device (CgState); the kernel of the exit test reports
// them to the host.  Kernels past the exit return immediately.
#include <cmath>
#include <cstring>
#include <vector>

#include "nekamd_internal.h"
#include "tails.h"

namespace nekamd {

namespace {

constexpr int kMaxCg = kMaxCgIter;

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_down(v, o, 64);
  return v;
}

// Sum of `count` partials by one block of kScalThreads threads in a fixed
// order.  Result valid on thread 0.
constexpr int kScalThreads = 1024;
__device__ double block_sum_array(const double *__restrict__ part, int count) {
  return block_sum_partials(part, count);
}

__device__ __forceinline__ void block_store2(double a, double b, double *pa, double *pb) {
  __shared__ double sa[4], sbb[4];
  a = wave_sum(a);
  b = wave_sum(b);
  if ((threadIdx.x & 63) == 0) {
    sa[threadIdx.x >> 6] = a;
    sbb[threadIdx.x >> 6] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    leave(pa + blockIdx.x, ((sa[0] + sa[1]) + sa[2]) + sa[3]);
    leave(pb + blockIdx.x, ((sbb[0] + sbb[1]) + sbb[2]) + sbb[3]);
  }
}

// last_block's counters of a solve
static_assert(kCounterDoubles <= kRedBlocks, "their place in red");
inline int *counters(double *red) { return reinterpret_cast<int *>(red + kRedCount); }

// Grid of the update-and-dots kernels: about 2048 nodes per block, at most
// kUpdBlocks -- a launch costs about 10 ns per block, which dominates small
// fields at a fixed large grid.  One partial sum per block.
inline int upd_blocks(int64_t n) {
  int64_t b = (n + 2047) / 2048;
  return (int)(b < 64 ? 64 : (b > kUpdBlocks ? kUpdBlocks : b));
}

// ---- what a solve has to know of its arrays (SolveFacts) -------------------
// One pass over h1, h2, mask, mult, f and, where asked, binv (the sums of
// chktcg1), another mask and the count codes of mult; f masked in place where
// asked.  Bound by its streams (6 to 9 words per node: 149 us, 5.4 TB/s, on
// 32,768 elements at lx1 = 8, where one reduction after another, each with
// its own host wait, took 0.5 ms; on 336 elements 10 us).  kNF results per block, fixed grid; the sums by
// one block in a fixed order.
enum { kF_h1min, kF_h1max, kF_h2min, kF_h2max, kF_fmax, kF_fmasked, kF_skmin, kF_inner, kF_mgdiff,
       kF_nocode, kF_rr, kF_bc1, kF_bc2, kNF };
__host__ __device__ constexpr int fact_op(int q) {  // 0 sum, 1 min, 2 max
  return (q == kF_h1min || q == kF_h2min || q == kF_skmin) ? 1 : (q >= kF_rr ? 0 : 2);
}
__device__ __forceinline__ double fact_join(int op, double a, double b) {
  return op == 0 ? a + b : (op == 1 ? fmin(a, b) : fmax(a, b));
}
__device__ __forceinline__ double fact_start(int op) {
  return op == 0 ? 0.0 : (op == 1 ? INFINITY : -INFINITY);
}

__global__ void __launch_bounds__(256)
    k_facts(const double *__restrict__ h1, const double *__restrict__ h2,
            const double *__restrict__ mask, const double *__restrict__ mult, double *f,
            int mask_f, const double *__restrict__ binv, const double *__restrict__ other,
            uint8_t *__restrict__ code, int64_t n, int np, double *__restrict__ part,
            double *__restrict__ groups, int *__restrict__ left) {
  __shared__ double sb[4][kNF];
  __shared__ uint8_t s_in[kMaxNP * kMaxNP * kMaxNP];
  const int np3 = np * np * np;
  for (int q = threadIdx.x; q < np3; q += 256) {
    const int i = q % np, j = (q / np) % np, k = q / (np * np);
    s_in[q] = i > 0 && i < np - 1 && j > 0 && j < np - 1 && k > 0 && k < np - 1;
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) {  // for the kernels after this one
    *groups = 0.0;
    *left = kNF;
  }
  __syncthreads();
  double v[kNF];
#pragma unroll
  for (int q = 0; q < kNF; ++q) v[q] = fact_start(fact_op(q));
  v[kF_fmax] = v[kF_fmasked] = v[kF_inner] = v[kF_mgdiff] = v[kF_nocode] = 0.0;
  const int64_t i0 = blockIdx.x * (int64_t)256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
  int at = (int)(i0 % np3);
  const int step = (int)(stride % np3);
  for (int64_t i = i0; i < n; i += stride) {
    const double a1 = h1[i], a2 = h2[i], m = mask[i], u = mult[i];
    v[kF_h1min] = fmin(v[kF_h1min], a1);
    v[kF_h1max] = fmax(v[kF_h1max], a1);
    v[kF_h2min] = fmin(v[kF_h2min], a2);
    v[kF_h2max] = fmax(v[kF_h2max], a2);
    v[kF_skmin] = fmin(v[kF_skmin], m);
    if (s_in[at]) v[kF_inner] = fmax(v[kF_inner], fmax(fabs(m - 1.0), fabs(u - 1.0)));
    at += step;
    at -= at >= np3 ? np3 : 0;
    double fi = 0.0;
    if (f) {
      fi = f[i];
      if (mask_f) {
        fi = fi * m;
        f[i] = fi;
      }
      v[kF_fmax] = fmax(v[kF_fmax], fabs(fi));
      if (m == 0.0) v[kF_fmasked] = fmax(v[kF_fmasked], fabs(fi));
    }
    if (binv) {
      v[kF_rr] += ((binv[i] * fi) * fi) * u;
      v[kF_bc1] += m * u;
      v[kF_bc2] += u;
    }
    if (other && other[i] != m) v[kF_mgdiff] = 1.0;
    if (code) {
      const double c = u > 0.0 ? rint(1.0 / u) : 0.0;
      const bool ok = c >= 1.0 && c <= 255.0 && 1.0 / c == u;
      code[i] = ok ? (uint8_t)c : (uint8_t)0;
      if (!ok) v[kF_nocode] = 1.0;
    }
  }
#pragma unroll
  for (int q = 0; q < kNF; ++q) {
    for (int o = 32; o > 0; o >>= 1)
      v[q] = fact_join(fact_op(q), v[q], __shfl_down(v[q], o, 64));
    if ((threadIdx.x & 63) == 0) sb[threadIdx.x >> 6][q] = v[q];
  }
  __syncthreads();
  if (threadIdx.x < kNF) {
    const int q = threadIdx.x, op = fact_op(q);
    double t = sb[0][q];
    for (int w = 1; w < 4; ++w) t = fact_join(op, t, sb[w][q]);
    part[(int64_t)q * kRedBlocks + blockIdx.x] = t;
  }
}

// block q: result q over the count partials; the last block to end reports
// the results and the group check to the host (left counts the blocks to go)
__global__ void __launch_bounds__(256)
    k_facts_final(const double *__restrict__ part, int count, double *__restrict__ out,
                  int *__restrict__ left, BoxRef rep) {
  __shared__ double sb[4];
  const int q = blockIdx.x, op = fact_op(q);
  double v = fact_start(op);
  for (int t = threadIdx.x; t < count; t += 256)
    v = fact_join(op, v, part[(int64_t)q * kRedBlocks + t]);
  for (int o = 32; o > 0; o >>= 1) v = fact_join(op, v, __shfl_down(v, o, 64));
  if ((threadIdx.x & 63) == 0) sb[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = sb[0];
    for (int w = 1; w < 4; ++w) t = fact_join(op, t, sb[w]);
    out[q] = t;
    if (rep.b) {
      rep.b->v[q] = t;
      if (q == 0) rep.b->v[kNF] = out[kNF];
      __threadfence_system();
      if (atomicSub(left, 1) == 1) box_report(rep);
    }
  }
}

// partial sums of a*a*b
__global__ void __launch_bounds__(256)
    k_sq_sum(const double *__restrict__ a, const double *__restrict__ b, int64_t n,
             double *__restrict__ part) {
  __shared__ double sb[4];
  double v = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    v += (a[i] * a[i]) * b[i];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sb[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = ((sb[0] + sb[1]) + sb[2]) + sb[3];
}
__global__ void __launch_bounds__(1024)
    k_sum_final(const double *__restrict__ part, int count, double *__restrict__ out) {
  const double t = block_sum_array(part, count);
  if (threadIdx.x == 0) *out = t;
}

// ---- elementwise ----------------------------------------------------------
__global__ void k_fill(double *__restrict__ a, double v, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    a[i] = v;
}
__global__ void k_mul(double *__restrict__ a, const double *__restrict__ b, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    a[i] = a[i] * b[i];
}
__global__ void k_inv(double *__restrict__ a, int64_t n) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    a[i] = 1.0 / a[i];
}
// d = 1/d (the assembled diagonal); r = f, x = 0; dm = d*mult; bm = binv*mult
// (or mult when param18=1); and the first iteration's partial sums (those of
// k_cg_update_dots without an update)
__global__ void __launch_bounds__(256)
    k_cg_init(double *__restrict__ x, double *__restrict__ r, const double *__restrict__ f,
              double *__restrict__ d, const double *__restrict__ mult,
              const double *__restrict__ binv, double *__restrict__ dm,
              double *__restrict__ bm, int plain_norm, int64_t n, double *__restrict__ part1,
              double *__restrict__ part2, CgState init, CgState *__restrict__ st,
              int *__restrict__ cnt) {
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) *st = init;
    clear_counters(cnt);
  }
  double s1 = 0.0, s2 = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double di = 1.0 / d[i], mu = mult[i], fi = f[i];
    const double a = di * mu, b = plain_norm ? mu : binv[i] * mu;
    d[i] = di;
    r[i] = fi;
    x[i] = 0.0;
    dm[i] = a;
    bm[i] = b;
    const double rr = fi * fi;
    s1 += a * rr;
    s2 += b * rr;
  }
  block_store2(s1, s2, part1, part2);
}

// the state to the host (a solve that is done changes it no more)
__device__ __forceinline__ void state_report(const CgState *st, const BoxRef &rep) {
  if (!rep.b) return;
  *reinterpret_cast<CgState *>(rep.b->v) = *st;
  box_report(rep);
}
// (of a mixed solve: the iteration's state, and whether a refresh is due)
constexpr int kBoxDue = (int)(sizeof(HostBox::v) / sizeof(double)) - 1;
static_assert(sizeof(CgState) <= sizeof(double) * kBoxDue, "a report holds a state");

__device__ void cg_scalars1(CgState *st, double s1, double s2, double *hist) {
  const int iter = st->iter + 1;
  st->iter = iter;
  if (iter > st->maxit) {  // loop exhausted (hmholtz.f:817: niter = iter-1)
    st->done = 1;
    st->niter = st->maxit;
    return;
  }
  st->rtz2 = st->rtz1;
  st->rtz1 = s1;
  const double rbn2 = sqrt(s2 / st->vol);
  st->rbn2 = rbn2;
  if (iter == 1) st->rbn0 = rbn2;
  if (st->param22 < 0) st->tol = fabs(st->param22) * st->rbn0;
  if (st->tin < 0) st->tol = fabs(st->tin) * st->rbn0;
  if (hist) {
    hist[5 * (iter - 1) + 0] = rbn2;
    hist[5 * (iter - 1) + 1] = s1;
  }
  if (rbn2 <= st->tol && (iter > 1 || st->istep <= 5)) {
    st->done = 1;
    st->converged = 1;
    st->niter = iter - 1;
    return;
  }
  st->beta = (iter == 1) ? 0.0 : st->rtz1 / st->rtz2;
}

// x += alpha p ; r -= alpha w (the update of the previous iteration) ; partial
// sums of (d*r)*r*mult and binv*mult*r*r (vlsc3 / vlsc32, hmholtz.f:754-759).
// VEC: 16-byte loads of node pairs (all six arrays 16-byte aligned).  The last
// block makes the iteration's exit test and beta and reports to the host.
template <bool VEC>
__global__ void __launch_bounds__(256)
    k_cg_update_dots(double *__restrict__ x, double *__restrict__ r,
                     const double *__restrict__ p, const double *__restrict__ w,
                     const double *__restrict__ dm, const double *__restrict__ bm, int64_t n,
                     CgState *st, double *part1, double *part2, int *cnt, double *hist,
                     BoxRef rep) {
  if (st->done) return;
  const double alpha = st->alpha;
  double s1 = 0.0, s2 = 0.0;
  const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  int64_t done_upto = 0;
  if constexpr (VEC) {
    // node pairs as native 2-vectors, streamed with nontemporal hints
    typedef double v2 __attribute__((ext_vector_type(2)));
    const int64_t n2 = n >> 1;
    v2 *x2 = reinterpret_cast<v2 *>(x);
    v2 *r2 = reinterpret_cast<v2 *>(r);
    const v2 *p2 = reinterpret_cast<const v2 *>(p);
    const v2 *w2 = reinterpret_cast<const v2 *>(w);
    const v2 *dm2 = reinterpret_cast<const v2 *>(dm);
    const v2 *bm2 = reinterpret_cast<const v2 *>(bm);
    for (int64_t i = tid; i < n2; i += stride) {
      v2 ri = __builtin_nontemporal_load(r2 + i);
      v2 xi = __builtin_nontemporal_load(x2 + i);
      const v2 pi = __builtin_nontemporal_load(p2 + i), wi = __builtin_nontemporal_load(w2 + i);
      xi.x = xi.x + alpha * pi.x;
      xi.y = xi.y + alpha * pi.y;
      ri.x = ri.x + (-alpha) * wi.x;
      ri.y = ri.y + (-alpha) * wi.y;
      __builtin_nontemporal_store(xi, x2 + i);
      __builtin_nontemporal_store(ri, r2 + i);
      const v2 d = __builtin_nontemporal_load(dm2 + i), b = __builtin_nontemporal_load(bm2 + i);
      const double rr0 = ri.x * ri.x, rr1 = ri.y * ri.y;
      s1 += d.x * rr0;
      s2 += b.x * rr0;
      s1 += d.y * rr1;
      s2 += b.y * rr1;
    }
    done_upto = n2 * 2;
  }
  for (int64_t i = done_upto + tid; i < n; i += stride) {
    x[i] = x[i] + alpha * p[i];
    const double ri = r[i] + (-alpha) * w[i];
    r[i] = ri;
    const double rr = ri * ri;
    s1 += dm[i] * rr;
    s2 += bm[i] * rr;
  }
  block_store2(s1, s2, part1, part2);
  if (!last_block(cnt, gridDim.x)) return;
  double t[2];
  sum_left(part1, part2 - part1, gridDim.x, t);
  if (threadIdx.x != 0) return;
  cg_scalars1(st, t[0], t[1], hist);
  state_report(st, rep);
}

// the first iteration's, after k_cg_init
__global__ void __launch_bounds__(kScalThreads)
    k_cg_scalars1(CgState *__restrict__ st, const double *__restrict__ part1,
                  const double *__restrict__ part2, int nparts, double *__restrict__ hist,
                  BoxRef rep) {
  if (st->done) return;
  double t[2];
  sum_left(part1, part2 - part1, nparts, t);
  if (threadIdx.x != 0) return;
  cg_scalars1(st, t[0], t[1], hist);
  state_report(st, rep);
}

// rho and alpha (the general path; the fused one has them in the assembly)
__global__ void __launch_bounds__(kScalThreads)
    k_cg_scalars2(CgState *__restrict__ st, StepLength step) {
  if (!st->done) step_length(step);
}
// rho = the count partials of the operator, alpha = rtz1 / rho
inline StepLength step_of(CgState *st, const double *part, int count, double *hist) {
  return StepLength{part, count, &st->rtz1, &st->rho, &st->alpha, hist, &st->beta, &st->iter};
}

// rho over all nodes (used when ids are not zero exactly at interiors):
// part[b] = sum w*p*mult over the block's nodes
__global__ void __launch_bounds__(256)
    k_dot3_guarded(const double *__restrict__ a, const double *__restrict__ b,
                   const double *__restrict__ c, int64_t n, const CgState *__restrict__ st,
                   double *__restrict__ part) {
  __shared__ double sb[4];
  if (st->done) return;
  double v = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    v += a[i] * b[i] * c[i];
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sb[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = ((sb[0] + sb[1]) + sb[2]) + sb[3];
}

__global__ void k_mask_guarded(double *__restrict__ w, const double *__restrict__ mask,
                               int64_t n, const CgState *__restrict__ st) {
  if (st->done) return;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    w[i] = w[i] * mask[i];
}

// ---- mixed precision: FP32 iteration, FP64 solution and true residual ----
// The Jacobi PCG iterates in single precision (r, p, w, the correction xs
// accumulated since the last refresh, the preconditioner; FP32 operator),
// with every inner product accumulated in FP64.  A refresh -- x += xs in
// FP64, r = f - mask*QQ^T A_L x in FP64 (FP64 axhelm and assembly), the
// iterated residual replaced by it -- runs when the iterated residual has
// fallen by kRefresh since the last one, when it meets the tolerance (the
// solve ends only if the FP64 residual meets it too) and when maxit is
// reached.  The search direction survives a refresh (reliable updates:
// Sleijpen & van der Vorst 1996; Clark et al. 2010 for single/double CG).
struct McgState {
  CgState cg;    // the iteration (read back by the host as a CgState)
  CgState gate;  // beta, and done: no operator now (the solve ended, or due)
  int due;       // a refresh is asked for
  double rmax;   // largest iterated residual norm since the last refresh
  int final;     // 1: iterated residual met the tolerance; 2: maxit reached
  int nrefresh;
};
// Refresh when the iterated residual has fallen by this factor since the
// last refresh.  The FP32 recurrence stays within a few FP32 roundings of
// the residual it started from, so a drop of 1e4 still leaves the iterated
// residual accurate to about 1e-3 relative; a factor of 0.1 refreshed every
// second iteration of a fast solve (8 decades in 16 iterations), costing an
// FP64 operator apply each time.  Measured on five time-step solves of 10-32
// iterations: 0.1 -> 1.07x over FP64, 1e-2 -> 1.24x, 1e-3 -> 1.32x,
// 1e-4 -> 1.40x with unchanged iteration counts and FP64 residuals; 1e-5
// and 1e-6 gain nothing more and let the solution drift further (up to
// 9e-9 relative from the FP64 solve at 1e-6, 4e-11 at 1e-4).
constexpr double kRefresh = 1e-4;
__device__ __forceinline__ void state_report(const McgState *ms, const BoxRef &rep) {
  if (!rep.b) return;
  rep.b->v[kBoxDue] = ms->due;
  state_report(&ms->cg, rep);
}

// as cg_scalars1, but a refresh of the residual is requested instead of
// ending the solve or when the iterated residual fell by kRefresh
__device__ void mcg_scalars1(McgState *ms, double s1, double s2, double *hist) {
  CgState *st = &ms->cg;
  const int iter = st->iter + 1;
  st->iter = iter;
  if (iter > st->maxit) {  // loop exhausted: fold the correction into x
    ms->final = 2;
    ms->due = ms->gate.done = 1;
    return;
  }
  st->rtz2 = st->rtz1;
  st->rtz1 = s1;
  const double rbn2 = sqrt(s2 / st->vol);
  st->rbn2 = rbn2;
  if (iter == 1) {
    st->rbn0 = rbn2;
    ms->rmax = rbn2;
  }
  if (st->param22 < 0) st->tol = fabs(st->param22) * st->rbn0;
  if (st->tin < 0) st->tol = fabs(st->tin) * st->rbn0;
  if (hist) {
    hist[5 * (iter - 1) + 0] = rbn2;
    hist[5 * (iter - 1) + 1] = s1;
  }
  if (rbn2 <= st->tol && (iter > 1 || st->istep <= 5)) {
    ms->final = 1;
    ms->due = ms->gate.done = 1;
    return;
  }
  if (rbn2 < kRefresh * ms->rmax) {
    ms->final = 0;
    ms->due = ms->gate.done = 1;
    return;
  }
  if (rbn2 > ms->rmax) ms->rmax = rbn2;
  ms->gate.beta = st->beta = (iter == 1) ? 0.0 : st->rtz1 / st->rtz2;
}

// xs += alpha p ; r -= alpha w (FP32) ; FP64 partials of dm*r*r and bm*r*r;
// the iteration's tests in the last block
template <bool VEC>
__global__ void __launch_bounds__(256)
    k_mcg_update_dots(float *__restrict__ xs, float *__restrict__ r,
                      const float *__restrict__ p, const float *__restrict__ w,
                      const float *__restrict__ dm, const float *__restrict__ bm, int64_t n,
                      McgState *ms, double *part1, double *part2, int *cnt, double *hist,
                      BoxRef rep) {
  CgState *st = &ms->cg;
  if (st->done) return;
  const float alpha = (float)st->alpha;
  double s1 = 0.0, s2 = 0.0;
  const int64_t tid = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  int64_t done_upto = 0;
  if constexpr (VEC) {
    typedef float v4 __attribute__((ext_vector_type(4)));
    const int64_t n4 = n >> 2;
    v4 *x4 = reinterpret_cast<v4 *>(xs);
    v4 *r4 = reinterpret_cast<v4 *>(r);
    const v4 *p4 = reinterpret_cast<const v4 *>(p);
    const v4 *w4 = reinterpret_cast<const v4 *>(w);
    const v4 *d4 = reinterpret_cast<const v4 *>(dm);
    const v4 *b4 = reinterpret_cast<const v4 *>(bm);
    for (int64_t i = tid; i < n4; i += stride) {
      v4 ri = __builtin_nontemporal_load(r4 + i);
      v4 xi = __builtin_nontemporal_load(x4 + i);
      const v4 pi = __builtin_nontemporal_load(p4 + i), wi = __builtin_nontemporal_load(w4 + i);
      xi.x += alpha * pi.x;
      xi.y += alpha * pi.y;
      xi.z += alpha * pi.z;
      xi.w += alpha * pi.w;
      ri.x -= alpha * wi.x;
      ri.y -= alpha * wi.y;
      ri.z -= alpha * wi.z;
      ri.w -= alpha * wi.w;
      __builtin_nontemporal_store(xi, x4 + i);
      __builtin_nontemporal_store(ri, r4 + i);
      const v4 d = __builtin_nontemporal_load(d4 + i), b = __builtin_nontemporal_load(b4 + i);
      const double q0 = (double)ri.x * ri.x, q1 = (double)ri.y * ri.y,
                   q2 = (double)ri.z * ri.z, q3 = (double)ri.w * ri.w;
      s1 += d.x * q0 + d.y * q1 + d.z * q2 + d.w * q3;
      s2 += b.x * q0 + b.y * q1 + b.z * q2 + b.w * q3;
    }
    done_upto = n4 * 4;
  }
  for (int64_t i = done_upto + tid; i < n; i += stride) {
    xs[i] = xs[i] + alpha * p[i];
    const float ri = r[i] - alpha * w[i];
    r[i] = ri;
    const double q = (double)ri * ri;
    s1 += dm[i] * q;
    s2 += bm[i] * q;
  }
  block_store2(s1, s2, part1, part2);
  if (!last_block(cnt, gridDim.x)) return;
  double t[2];
  sum_left(part1, part2 - part1, gridDim.x, t);
  if (threadIdx.x != 0) return;
  mcg_scalars1(ms, t[0], t[1], hist);
  state_report(ms, rep);
}

// the first iteration's, after k_mcg_init
__global__ void __launch_bounds__(kScalThreads)
    k_mcg_scalars1(McgState *__restrict__ ms, const double *__restrict__ part1,
                   const double *__restrict__ part2, int nparts, double *__restrict__ hist,
                   BoxRef rep) {
  if (ms->cg.done) return;
  double t[2];
  sum_left(part1, part2 - part1, nparts, t);
  if (threadIdx.x != 0) return;
  mcg_scalars1(ms, t[0], t[1], hist);
  state_report(ms, rep);
}

// refresh, part 1: x += xs (FP64), xs = 0
__global__ void k_mcg_fold(double *__restrict__ x, float *__restrict__ xs, int64_t n) {
#pragma unroll 4
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    x[i] = x[i] + (double)xs[i];
    xs[i] = 0.0f;
  }
}

// refresh, part 3: the true residual's norm decides the exit; otherwise the
// iteration continues from it with the same search direction
__device__ void mcg_scalars1b(McgState *ms, double s1, double s2, double *hist) {
  CgState *st = &ms->cg;
  ms->due = 0;
  ms->nrefresh += 1;
  const double rbn2 = sqrt(s2 / st->vol);
  st->rbn2 = rbn2;
  if (ms->final == 2) {
    st->done = 1;
    st->niter = st->maxit;
    return;
  }
  const int iter = st->iter;
  st->rtz1 = s1;
  if (hist) {
    hist[5 * (iter - 1) + 0] = rbn2;
    hist[5 * (iter - 1) + 1] = s1;
  }
  if (ms->final == 1 && rbn2 <= st->tol) {
    st->done = 1;
    st->converged = 1;
    st->niter = iter - 1;
    return;
  }
  ms->final = 0;
  ms->rmax = rbn2;
  ms->gate.done = 0;
  ms->gate.beta = st->beta = (iter == 1) ? 0.0 : st->rtz1 / st->rtz2;
}

// refresh, part 2 (after ax = mask*QQ^T A_L x): r = f - ax in FP64, stored
// rounded; partials of dm*r32^2 (the iteration's rtz) and bm*r^2 (FP64 norm);
// part 3 and the report in the last block.
__global__ void __launch_bounds__(256)
    k_mcg_resid(float *__restrict__ r32, const double *__restrict__ f,
                const double *__restrict__ ax, const float *__restrict__ dm,
                const float *__restrict__ bm, int64_t n, McgState *ms, double *part1,
                double *part2, int *cnt, double *hist, BoxRef rep) {
  double s1 = 0.0, s2 = 0.0;
#pragma unroll 4
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double ri = f[i] - ax[i];
    const float rf = (float)ri;
    r32[i] = rf;
    s1 += dm[i] * ((double)rf * rf);
    s2 += bm[i] * (ri * ri);
  }
  block_store2(s1, s2, part1, part2);
  if (!last_block(cnt, gridDim.x)) return;
  double t[2];
  sum_left(part1, part2 - part1, gridDim.x, t);
  if (threadIdx.x != 0) return;
  mcg_scalars1b(ms, t[0], t[1], hist);
  state_report(ms, rep);
}

// x = 0, xs = 0, r = f (rounded), and 1/d (d the assembled diagonal), its
// product with mult and binv*mult (or mult) in FP32; the first iteration's
// partial sums
__global__ void __launch_bounds__(256)
    k_mcg_init(double *__restrict__ x, float *__restrict__ xs, float *__restrict__ r,
               float *__restrict__ d32, float *__restrict__ dm, float *__restrict__ bm,
               const double *__restrict__ f, const double *__restrict__ d,
               const double *__restrict__ mult, const double *__restrict__ binv, int plain_norm,
               int64_t n, double *__restrict__ part1, double *__restrict__ part2, McgState init,
               McgState *__restrict__ ms, int *__restrict__ cnt) {
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) *ms = init;
    clear_counters(cnt);
  }
  double s1 = 0.0, s2 = 0.0;
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const double di = 1.0 / d[i], mu = mult[i];
    const float a = (float)(di * mu), b = (float)(plain_norm ? mu : binv[i] * mu);
    const float ri = (float)f[i];
    x[i] = 0.0;
    xs[i] = 0.0f;
    r[i] = ri;
    d32[i] = (float)di;
    dm[i] = a;
    bm[i] = b;
    const double q = (double)ri * ri;
    s1 += a * q;
    s2 += b * q;
  }
  block_store2(s1, s2, part1, part2);
}

int grid_for(int64_t n) {
  int64_t g = (n + 255) / 256;
  if (g > 8192) g = 8192;
  if (g < 1) g = 1;
  return (int)g;
}

}  // namespace

int ensure_small(Mesh &m) {
  // room for the mixed-precision solve's state (a CgState first)
  if (!m.st) NK_HIP(hipMalloc(&m.st, sizeof(McgState)));
  if (!m.red) NK_HIP(hipMalloc(&m.red, sizeof(double) * kRedSize));
  if (m.reports && !m.box) NK_TRY(box_alloc(&m.box));
  return NKH_OK;
}

int box_alloc(HostBox **b) {
  NK_HIP(hipHostMalloc(reinterpret_cast<void **>(b), sizeof(HostBox),
                       hipHostMallocMapped | hipHostMallocCoherent));
  std::memset(static_cast<void *>(*b), 0, sizeof(HostBox));
  return NKH_OK;
}

namespace {
__global__ void k_box_report(BoxRef r) { box_report(r); }
}  // namespace

int box_join(const BoxRef &r, hipStream_t s) {
  hipLaunchKernelGGL(k_box_report, dim3(1), dim3(1), 0, s, r);
  NK_HIP(hipGetLastError());
  return box_wait(r, s);
}

int box_wait(const BoxRef &r, hipStream_t s) {
  for (int64_t spin = 1;; ++spin) {
    if (__atomic_load_n(&r.b->seq, __ATOMIC_ACQUIRE) >= r.seq) return NKH_OK;
    if (spin % 8192 == 0) {  // every 50 us or so
      const hipError_t e = hipStreamQuery(s);
      if (e == hipErrorNotReady) continue;
      NK_HIP(e);
      NK_CHECK(__atomic_load_n(&r.b->seq, __ATOMIC_ACQUIRE) >= r.seq, NKH_ERR_STATE,
               "a solve's kernels ended without their report");
      return NKH_OK;
    }
    __builtin_ia32_pause();
  }
}

int ensure_workspace(Mesh &m) {
  NK_TRY(ensure_small(m));
  const size_t need = cg_ws_doubles(m.n);
  if (m.ws && m.ws_doubles >= need) return NKH_OK;
  if (m.ws) (void)hipFree(m.ws);
  m.ws = nullptr;
  if (hipMalloc(&m.ws, sizeof(double) * need) != hipSuccess) {
    set_error("workspace allocation of %zu doubles failed", need);
    return NKH_ERR_NOMEM;
  }
  m.ws_doubles = need;
  return NKH_OK;
}

// The passes of gather_facts on s: partial sums in red, the kNF + 1 results
// at red + kRedOut, the group flags of mask in flag.
static int enqueue_facts(Mesh &m, const double *h1, const double *h2, const double *mask,
                         const double *mult, double *f, const FactsAsk &ask, double *red,
                         uint8_t *flag, const BoxRef &rep, hipStream_t s) {
  static_assert(kNF * kRedBlocks <= kRedCount, "the partial sums take the dots' place");
  double *part = red + kRedPart1, *res = red + kRedOut;
  int *left = reinterpret_cast<int *>(res + kNF + 1);
  const int64_t per = 1024;  // nodes per block, up to the fixed grid
  const int nb = (int)std::min<int64_t>(std::max<int64_t>((m.n + per - 1) / per, 1), kRedBlocks);
  hipLaunchKernelGGL(k_facts, dim3(nb), dim3(256), 0, s, h1, h2, mask, mult, f,
                     ask.mask_f ? 1 : 0, ask.chk ? m.binv : nullptr, ask.other_mask, ask.code,
                     m.n, m.np, part, res + kNF, left);
  NK_TRY(gs_prepare(m.gs, mask, mult, flag, res + kNF, s));
  hipLaunchKernelGGL(k_facts_final, dim3(kNF), dim3(256), 0, s, part, nb, res, left, rep);
  NK_HIP(hipGetLastError());
  return NKH_OK;
}

// the facts from the kNF + 1 results (on the host)
static SolveFacts read_facts(const Mesh &m, const double *h1, const double *h2, const double *h) {
  SolveFacts o;
  o.h1min = h[kF_h1min];
  o.h1max = h[kF_h1max];
  o.h2min = h[kF_h2min];
  o.h2max = h[kF_h2max];
  o.fmax = h[kF_fmax];
  o.fmasked = h[kF_fmasked];
  o.skmin = h[kF_skmin];
  o.inner = h[kF_inner];
  o.mgdiff = h[kF_mgdiff];
  o.nocode = h[kF_nocode];
  o.rr = h[kF_rr];
  o.bcneu1 = h[kF_bc1];
  o.bcneu2 = h[kF_bc2];
  o.groups = m.gs.ngroups > 0 ? h[kNF] : 1.0;  // no ids at all: never fused
  o.h1 = h1;
  o.h2 = h2;
  o.interior_zero = m.gs.interior_zero;
  return o;
}

int gather_facts(Mesh &m, const double *h1, const double *h2, const double *mask,
                 const double *mult, double *f, const FactsAsk &ask, SolveFacts *out,
                 hipStream_t s) {
  NK_TRY(ensure_small(m));
  if (!m.gs.flag && m.gs.ngroups > 0) NK_HIP(hipMalloc(&m.gs.flag, (size_t)m.gs.ngroups));
  const BoxRef rep = m.next_report();
  NK_TRY(enqueue_facts(m, h1, h2, mask, mult, f, ask, m.red, m.gs.flag, rep, s));
  if (rep.b) {
    NK_TRY(box_wait(rep, s));
    *out = read_facts(m, h1, h2, rep.b->v);
    return NKH_OK;
  }
  double h[kNF + 1];
  NK_HIP(hipMemcpyAsync(h, m.red + kRedOut, sizeof(h), hipMemcpyDeviceToHost, s));
  NK_HIP(hipStreamSynchronize(s));
  *out = read_facts(m, h1, h2, h);
  return NKH_OK;
}

int mul_inplace(double *a, const double *b, int64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_mul, dim3(grid_for(n)), dim3(256), 0, s, a, b, n);
  NK_HIP(hipGetLastError());
  return NKH_OK;
}

// the assembled Jacobi diagonal, not inverted
static int setprec_sum(Mesh &m, double *d, Coef h1, Coef h2, hipStream_t s) {
  NK_TRY(launch_setprec(m, d, h1, h2, s));
  return gs_op(m.gs, d, 0, s);
}

int run_setprec(Mesh &m, double *d, Coef h1, Coef h2, hipStream_t s) {
  NK_TRY(setprec_sum(m, d, h1, h2, s));
  hipLaunchKernelGGL(k_inv, dim3(grid_for(m.n)), dim3(256), 0, s, d, m.n);
  NK_HIP(hipGetLastError());
  return NKH_OK;
}

int run_chktcg1(Mesh &m, double *tol, const SolveFacts &facts) {
  hipStream_t s = cur_stream();
  const int64_t n = m.n;
  const double eps = 1.0e-13, acondno = 10.0;
  // rinit = sqrt(glsc3(binv*res, res, mult)/vol)
  const double rinit = std::sqrt(facts.rr / m.vol);
  const double rmin = eps * rinit;
  if (*tol < rmin) *tol = rmin;
  const double bctest = std::fabs(facts.bcneu1 - facts.bcneu2);
  // the operator's action on constants matters where no node is masked
  if (!(bctest < 0.1)) return NKH_OK;
  NK_TRY(ensure_workspace(m));
  double *w1 = m.ws, *w2 = m.ws + n;
  hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(256), 0, s, w1, 1.0, n);
  NK_TRY(launch_axhelm(m, w2, w1, facts.c1(), facts.c2(), s));
  hipLaunchKernelGGL(k_sq_sum, dim3(kRedBlocks), dim3(256), 0, s, w2, m.bm1, n,
                     m.red + kRedScratch);
  hipLaunchKernelGGL(k_sum_final, dim3(1), dim3(1024), 0, s, m.red + kRedScratch, kRedBlocks,
                     m.red + kRedOut);
  NK_HIP(hipGetLastError());
  double sq;
  NK_HIP(hipMemcpyAsync(&sq, m.red + kRedOut, sizeof(double), hipMemcpyDeviceToHost, s));
  NK_HIP(hipStreamSynchronize(s));
  const double bcrob = std::sqrt(sq / m.vol);
  if (bcrob < eps * acondno) {
    const double tolmin = rinit * eps * 10.0;
    if (*tol < tolmin) *tol = tolmin;
  }
  return NKH_OK;
}

// One Jacobi-PCG solve whose iterations can be enqueued one at a time (the
// single solve below, and the batch of solves).
struct CgRun {
  Mesh *m = nullptr;
  double *x = nullptr, *r = nullptr, *w = nullptr, *p = nullptr, *d = nullptr, *dm = nullptr,
         *bm = nullptr;
  double *red = nullptr;
  CgState *st = nullptr;
  const uint8_t *flag = nullptr;  // gs group flags for this solve's mask/mult
  Coef h1, h2;
  const double *mask = nullptr, *mult = nullptr;
  bool fused = false, vec_ok = false, trivial = false;
  int niter = 0, launched = 0, ax_grid_parts = 0;
  double *hist = nullptr;
  // An iteration reports its state after the exit test.  The test that ends
  // the solve is not its end: of the kernels behind it, which return at once,
  // any block that starts late still reads the state (and the next solve in
  // this work space, on another stream perhaps, sets it anew).  So the host
  // then waits for everything enqueued.
  Reports reports;
  BoxRef rep;  // the last one asked for
  int wait(CgState *hs, hipStream_t s) {
    NK_TRY(box_wait(rep, s));
    std::memcpy(hs, rep.b->v, sizeof(CgState));
    return hs->done ? box_join(reports.next(), s) : NKH_OK;
  }

  // hmholtz.f:611-720 up to the loop: preconditioner, r = f, null-space check,
  // choice of the fused iteration, device state.  ws: 6 n doubles, red:
  // kRedSize doubles, st: the state; all on stream s (host waits).
  int begin(Mesh &mesh, double *ws, double *red_, CgState *st_, double *x_, const double *f,
            const SolveFacts &facts, const double *mask_, const double *mult_, double tin,
            int maxit, const nkh_params &prm, bool want_hist, hipStream_t s) {
    m = &mesh;
    const int64_t n = mesh.n;
    x = x_;
    r = ws;
    w = ws + n;
    p = ws + 2 * n;
    d = ws + 3 * n;
    dm = ws + 4 * n;
    bm = ws + 5 * n;
    red = red_;
    st = st_;
    h1 = facts.c1();
    h2 = facts.c2();
    mask = mask_;
    mult = mult_;
    double tol = std::fabs(tin);
    if (prm.restol != 0.0) tol = prm.restol;
    if (tin < 0) tol = std::fabs(tin);
    niter = maxit < kMaxCg ? maxit : kMaxCg;
    trivial = facts.fmax == 0.0;
    if (trivial) {
      hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(256), 0, s, x, 0.0, n);
      NK_HIP(hipGetLastError());
      return NKH_OK;
    }
    // null-space check (hmholtz.f:705-720): pure Neumann with h2 == 0
    NK_CHECK(!(facts.skmin > 0 && facts.h2max == 0), NKH_ERR_UNSUPPORTED,
             "cggo: pure-Neumann mean correction (ifmcor) is not implemented");
    // the operator's kernel choice for this order (w is scratch until then)
    NK_TRY(axhelm_autotune(mesh, w, f, h1, h2, s));
    NK_TRY(setprec_sum(mesh, d, h1, h2, s));
    CgState h{};
    h.rtz1 = 1.0;
    h.tol = tol;
    h.tin = tin;
    h.vol = mesh.vol;
    h.param22 = prm.param22;
    h.maxit = niter;
    h.istep = prm.istep;
    h.param18 = prm.param18;
    hipLaunchKernelGGL(k_cg_init, dim3(upd_blocks(n)), dim3(256), 0, s, x, r, f, d, mult,
                       mesh.binv, dm, bm, prm.param18 == 1 ? 1 : 0, n, red + kRedPart1,
                       red + kRedPart2, h, st, counters(red));
    NK_HIP(hipGetLastError());
    // Fused iteration (rho inside axhelm, mask inside the assembly) when its
    // conditions hold and f is zero where masked.
    fused = facts.fused() && facts.fmasked == 0.0;
    flag = mesh.gs.flag;
    ax_grid_parts = axhelm_cg_grid(mesh);
    auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    vec_ok = al16(x) && al16(r) && al16(p) && al16(w) && al16(dm) && al16(bm);
    hist = nullptr;
    if (want_hist) {
      hist = red + kRedHist;
      hipLaunchKernelGGL(k_fill, dim3(grid_for(5 * kMaxCg)), dim3(256), 0, s, hist, 0.0,
                         (int64_t)5 * kMaxCg);
    }
    NK_HIP(hipGetLastError());
    return NKH_OK;
  }

  template <class Ev>
  int go_on(hipStream_t s, Ev &&ev) {
    return enqueue(s, ev(launched));
  }

  // one iteration's launches on s; ev (optional, 3 events) brackets axhelm
  // and the assembly
  int enqueue(hipStream_t s, hipEvent_t *ev = nullptr) {
    const int64_t n = m->n;
    double *part1 = red + kRedPart1, *part2 = red + kRedPart2, *rho1 = red + kRedRho1;
    const int ub = upd_blocks(n);
    rep = reports.next();
    if (launched > 0)
      hipLaunchKernelGGL((vec_ok ? k_cg_update_dots<true> : k_cg_update_dots<false>), dim3(ub),
                         dim3(256), 0, s, x, r, p, w, dm, bm, n, st, part1, part2,
                         counters(red), hist, rep);
    else  // (the first iteration's sums come from k_cg_init)
      hipLaunchKernelGGL(k_cg_scalars1, dim3(1), dim3(kScalThreads), 0, s, st, part1, part2, ub,
                         hist, rep);
    if (fused) {
      if (ev) NK_HIP(hipEventRecord(ev[0], s));
      NK_TRY(launch_axhelm_cg(*m, w, p, r, d, h1, h2, mult, st, rho1, s));
      if (ev) NK_HIP(hipEventRecord(ev[1], s));
      NK_TRY(gs_assemble_step(m->gs, w, st, s, flag, step_of(st, rho1, ax_grid_parts, hist)));
      if (ev) NK_HIP(hipEventRecord(ev[2], s));
    } else {
      NK_TRY(launch_axhelm_cg(*m, w, p, r, d, h1, h2, mult, st, nullptr, s));
      NK_TRY(gs_op(m->gs, w, 0, s));
      hipLaunchKernelGGL(k_mask_guarded, dim3(grid_for(n)), dim3(256), 0, s, w, mask, n, st);
      hipLaunchKernelGGL(k_dot3_guarded, dim3(kRedBlocks), dim3(256), 0, s, w, p, mult, n, st,
                         rho1);
      hipLaunchKernelGGL(k_cg_scalars2, dim3(1), dim3(kScalThreads), 0, s, st,
                         step_of(st, rho1, kRedBlocks, hist));
    }
    NK_HIP(hipGetLastError());
    ++launched;
    return NKH_OK;
  }

  void result(const CgState &hs, nkh_result *res) const {
    nkh_result out{};
    if (!trivial) {
      out.niter = hs.niter;
      out.converged = hs.converged;
      out.rbn0 = hs.rbn0;
      out.rbn2 = hs.rbn2;
      out.tol = hs.tol;
    }
    if (res) *res = out;
  }
};

// The mixed-precision Jacobi PCG (see McgState), enqueued like CgRun.
// Work space (cg_ws_doubles): ax (n doubles, FP64 refresh and set-up
// scratch), then seven FP32 vectors r, p, w, xs, d, d*mult, bm at 256-byte
// aligned offsets.  Needs uniform h1/h2 and the fused iteration's conditions.
struct McgRun {
  Mesh *m = nullptr;
  double *x = nullptr, *ax = nullptr;
  const double *f = nullptr;
  float *r = nullptr, *p = nullptr, *w = nullptr, *xs = nullptr, *d = nullptr, *dm = nullptr,
        *bm = nullptr;
  double *red = nullptr;
  McgState *ms = nullptr;
  CgState *st = nullptr;  // &ms->cg
  const uint8_t *flag = nullptr;
  Coef h1, h2;
  bool trivial = false, vec_ok = false, fused = true;
  int niter = 0, launched = 0, ax_grid_parts = 0;
  double *hist = nullptr;
  // the reports and the end of a solve as in CgRun
  Reports reports;
  BoxRef rep;
  bool due = false;  // the last report asked for a refresh
  int wait(CgState *hs, hipStream_t s) {
    NK_TRY(box_wait(rep, s));
    std::memcpy(hs, rep.b->v, sizeof(CgState));
    due = rep.b->v[kBoxDue] != 0.0;
    return hs->done ? box_join(reports.next(), s) : NKH_OK;
  }

  int begin(Mesh &mesh, double *ws, double *red_, void *st_, double *x_, const double *f_,
            const SolveFacts &facts, const double *mask, const double *mult, double tin,
            int maxit, const nkh_params &prm, bool want_hist, hipStream_t s) {
    m = &mesh;
    const int64_t n = mesh.n;
    h1 = facts.c1();
    h2 = facts.c2();
    NK_CHECK(h1.uniform() && h2.uniform(), NKH_ERR_UNSUPPORTED,
             "mixed-precision cggo: h1 and h2 must be uniform");
    x = x_;
    f = f_;
    ax = ws;
    const int64_t nn = (n + 63) / 64 * 64;
    float *base = reinterpret_cast<float *>(ws + (n + 31) / 32 * 32);
    r = base;
    p = base + nn;
    w = base + 2 * nn;
    xs = base + 3 * nn;
    d = base + 4 * nn;
    dm = base + 5 * nn;
    bm = base + 6 * nn;
    red = red_;
    ms = static_cast<McgState *>(st_);
    st = &ms->cg;
    double tol = std::fabs(tin);
    if (prm.restol != 0.0) tol = prm.restol;
    if (tin < 0) tol = std::fabs(tin);
    niter = maxit < kMaxCg ? maxit : kMaxCg;
    trivial = facts.fmax == 0.0;
    if (trivial) {
      hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(256), 0, s, x, 0.0, n);
      NK_HIP(hipGetLastError());
      return NKH_OK;
    }
    NK_CHECK(!(facts.skmin > 0 && h2.s == 0.0), NKH_ERR_UNSUPPORTED,
             "cggo: pure-Neumann mean correction (ifmcor) is not implemented");
    NK_CHECK(facts.fused() && facts.fmasked == 0.0, NKH_ERR_UNSUPPORTED,
             "mixed-precision cggo: needs ids zero at element interiors, 0/1 masks and "
             "mult summing to 1 per group");
    flag = mesh.gs.flag;
    NK_TRY(axhelm_autotune(mesh, ax, f, h1, h2, s));  // the refreshes' operator
    NK_TRY(setprec_sum(mesh, ax, h1, h2, s));  // the diagonal (FP64) in the ax slot
    McgState h{};
    h.cg.rtz1 = 1.0;
    h.cg.tol = tol;
    h.cg.tin = tin;
    h.cg.vol = mesh.vol;
    h.cg.param22 = prm.param22;
    h.cg.maxit = niter;
    h.cg.istep = prm.istep;
    h.cg.param18 = prm.param18;
    hipLaunchKernelGGL(k_mcg_init, dim3(upd_blocks(n)), dim3(256), 0, s, x, xs, r, d, dm, bm, f,
                       ax, mult, mesh.binv, prm.param18 == 1 ? 1 : 0, n, red + kRedPart1,
                       red + kRedPart2, h, ms, counters(red));
    NK_HIP(hipGetLastError());
    NK_TRY(ensure_geom32(mesh, s));
    ax_grid_parts = axhelm_cg_grid(mesh);
    auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    vec_ok = al16(r) && al16(p) && al16(w) && al16(xs) && al16(dm) && al16(bm);
    hist = nullptr;
    if (want_hist) {
      hist = red + kRedHist;
      hipLaunchKernelGGL(k_fill, dim3(grid_for(5 * kMaxCg)), dim3(256), 0, s, hist, 0.0,
                         (int64_t)5 * kMaxCg);
    }
    NK_HIP(hipGetLastError());
    return NKH_OK;
  }

  // what follows the last report: a refresh if it asked for one, or the next
  // iteration; ev(k): the events of iteration k
  template <class Ev>
  int go_on(hipStream_t s, Ev &&ev) {
    return due ? refresh(s, ev(launched - 1)) : enqueue(s, ev(launched));
  }

  // One iteration's launches on s.  Its operator returns at once when the
  // tests of the iteration ask for a refresh: the host, told so, enqueues that
  // and the operator again (refresh()).
  int enqueue(hipStream_t s, hipEvent_t *ev = nullptr) {
    const int64_t n = m->n;
    double *part1 = red + kRedPart1, *part2 = red + kRedPart2;
    const int ub = upd_blocks(n);
    rep = reports.next();
    if (launched > 0)
      hipLaunchKernelGGL((vec_ok ? k_mcg_update_dots<true> : k_mcg_update_dots<false>), dim3(ub),
                         dim3(256), 0, s, xs, r, p, w, dm, bm, n, ms, part1, part2,
                         counters(red), hist, rep);
    else  // (the first iteration's sums come from k_mcg_init)
      hipLaunchKernelGGL(k_mcg_scalars1, dim3(1), dim3(kScalThreads), 0, s, ms, part1, part2, ub,
                         hist, rep);
    NK_TRY(enqueue_operator(s, ev));
    ++launched;
    return NKH_OK;
  }

  // The refresh that the last report asked for, and that iteration's operator.
  // (With the refresh in every iteration, its kernels returning at once on
  // small grids where none was due, a solve of 12 iterations with 2 refreshes
  // on 9e6 nodes, lx1 8, took 3340 us, now 2830.)
  int refresh(hipStream_t s, hipEvent_t *ev = nullptr) {
    const int64_t n = m->n;
    rep = reports.next();
    hipLaunchKernelGGL(k_mcg_fold, dim3(upd_blocks(n)), dim3(256), 0, s, x, xs, n);
    NK_TRY(launch_axhelm(*m, ax, x, h1, h2, s));
    NK_TRY(gs_assemble(m->gs, ax, nullptr, s, flag));
    hipLaunchKernelGGL(k_mcg_resid, dim3(upd_blocks(n)), dim3(256), 0, s, r, f, ax, dm, bm, n, ms,
                       red + kRedPart1, red + kRedPart2, counters(red), hist, rep);
    return enqueue_operator(s, ev);
  }

  int enqueue_operator(hipStream_t s, hipEvent_t *ev) {
    double *rho1 = red + kRedRho1;
    if (ev) NK_HIP(hipEventRecord(ev[0], s));
    NK_TRY(launch_axhelm32_jac(*m, w, p, r, d, (float)h1.s, (float)h2.s, &ms->gate, rho1, s));
    if (ev) NK_HIP(hipEventRecord(ev[1], s));
    NK_TRY(gs_assemble_step(m->gs, w, &ms->gate, s, flag, step_of(st, rho1, ax_grid_parts, hist)));
    if (ev) NK_HIP(hipEventRecord(ev[2], s));
    NK_HIP(hipGetLastError());
    return NKH_OK;
  }

  void result(const CgState &hs, nkh_result *res) const {
    nkh_result out{};
    if (!trivial) {
      out.niter = hs.niter;
      out.converged = hs.converged;
      out.rbn0 = hs.rbn0;
      out.rbn2 = hs.rbn2;
      out.tol = hs.tol;
    }
    if (res) *res = out;
  }
};

size_t cg_ws_doubles(int64_t n) {
  const size_t mixed = (size_t)((n + 31) / 32 * 32) + (size_t)(7 * ((n + 63) / 64 * 64) + 1) / 2;
  return std::max((size_t)6 * (size_t)n, mixed);
}

namespace {

template <class Run>
int drive_cggo(Mesh &m, double *x, const double *f, const SolveFacts &facts,
               const double *mask, const double *mult, double tin, int maxit,
               const nkh_params &prm, nkh_result *res, double *history_host,
               bool allow_timers = true) {
  hipStream_t s = cur_stream();
  NK_TRY(ensure_workspace(m));
  Run run;
  NK_TRY(run.begin(m, m.ws, m.red, m.st, x, f, facts, mask, mult, tin, maxit, prm,
                   history_host != nullptr, s));
  if (run.trivial) {  // x = 0 is enqueued: returned when it is there, as any solution
    run.result(CgState{}, res);
    if (m.box) return box_join(m.next_report(), s);
    NK_HIP(hipStreamSynchronize(s));
    return NKH_OK;
  }
  CgState hs{};
  run.reports = Reports{m.box, &m.box_seq};
  // CTIMER mirror: event pairs around axhelm and gs of every launched iteration
  const bool timed = allow_timers && timers().on;
  const int niter = run.niter;
  std::vector<hipEvent_t> ev;
  if (timed) {
    ev.resize((size_t)4 * (niter + 1));
    for (auto &e : ev) NK_HIP(hipEventCreate(&e));
  }
  hipEvent_t t_solve0 = nullptr, t_solve1 = nullptr;
  if (timed) {
    NK_HIP(hipEventCreate(&t_solve0));
    NK_HIP(hipEventCreate(&t_solve1));
    NK_HIP(hipEventRecord(t_solve0, s));
  }
  // Each iteration's exit test reports to the host, which enqueues the next
  // iteration while the operator of this one runs.  Without a report (the
  // allocation-free solve) the state is copied back, later on every fourth
  // iteration.
  auto iterate = [&]() -> int {
    while (true) {
      NK_TRY(run.go_on(s, [&](int k) { return timed ? &ev[4 * k] : nullptr; }));
      if (run.reports.box) {
        NK_TRY(run.wait(&hs, s));
      } else if (run.launched < 8 || run.launched % 4 == 0 || run.launched > niter) {
        NK_HIP(hipMemcpyAsync(&hs, run.st, sizeof(CgState), hipMemcpyDeviceToHost, s));
        NK_HIP(hipStreamSynchronize(s));
      }
      if (hs.done) return NKH_OK;
      NK_CHECK(run.launched <= niter + 1, NKH_ERR_STATE, "cggo: state machine did not terminate");
    }
  };
  const int rc = iterate();
  if (rc != NKH_OK) (void)hipStreamSynchronize(s);  // an error leaves work in flight
  NK_TRY(rc);
  if (timed) {
    NK_HIP(hipEventRecord(t_solve1, s));
    NK_HIP(hipEventSynchronize(t_solve1));
    float ms = 0.f;
    // axhelm and gs did work in launches 1..niter (later ones returned at once)
    for (int it = 0; it < hs.niter && run.fused; ++it) {
      NK_HIP(hipEventElapsedTime(&ms, ev[4 * it + 0], ev[4 * it + 1]));
      timers().taxhm += ms * 1e-3;
      timers().naxhm += 1;
      NK_HIP(hipEventElapsedTime(&ms, ev[4 * it + 1], ev[4 * it + 2]));
      timers().tdsum += ms * 1e-3;
      timers().ndsum += 1;
    }
    NK_HIP(hipEventElapsedTime(&ms, t_solve0, t_solve1));
    timers().thmhz += ms * 1e-3;
    timers().nhmhz += 1;
    for (auto &e : ev) (void)hipEventDestroy(e);
    (void)hipEventDestroy(t_solve0);
    (void)hipEventDestroy(t_solve1);
  }
  run.result(hs, res);
  if (history_host) {
    NK_HIP(hipMemcpyAsync(history_host, run.hist, sizeof(double) * 5 * kMaxCg,
                          hipMemcpyDeviceToHost, s));
    NK_HIP(hipStreamSynchronize(s));
  }
  return NKH_OK;
}

}  // namespace

int run_cggo(Mesh &m, double *x, const double *f, const SolveFacts &facts, const double *mask,
             const double *mult, double tin, int maxit, const nkh_params &prm,
             nkh_result *res, double *history_host) {
  if (prm.precision == 2)
    return drive_cggo<McgRun>(m, x, f, facts, mask, mult, tin, maxit, prm, res, history_host);
  return drive_cggo<CgRun>(m, x, f, facts, mask, mult, tin, maxit, prm, res, history_host);
}

// ---------------------------------------------------------------------------
// Allocation-free FP64 Jacobi PCG (nkd_cggo_noalloc), for callers that may
// not allocate device memory.  The solve's vectors (r, w, p, d, d*mult,
// bm), its partial sums and history, its device state and the gs group
// flags of its mask/mult live in `scratch`, one file-scope device array per
// GPU, sized for meshes of at most kNoAllocMaxN local nodes.  Host code
// reaches the array only through the address hipGetSymbolAddress returns
// for the current device (noalloc_scratch).  Every call on a GPU uses the
// same array: calls that overlap on one GPU race.  Nothing in it needs to
// start at zero (each solve writes its state, partial sums, flags and
// vectors before reading them); the last call's contents stay behind.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocWs = 6 * (size_t)kNoAllocMaxN;                         // doubles
constexpr size_t kNoAllocRed = ((size_t)kRedSize + 31) / 32 * 32;               // doubles
constexpr size_t kNoAllocState = (sizeof(McgState) + 255) / 256 * 32;           // doubles
constexpr size_t kNoAllocFlag = ((size_t)kNoAllocMaxN + 255) / 256 * 32;        // doubles
constexpr size_t kNoAllocDoubles = kNoAllocWs + kNoAllocRed + kNoAllocState + kNoAllocFlag;
static_assert(kNoAllocMaxN < ((int64_t)1 << 20),
              "the axhelm autotuner (which allocates) runs on meshes of 2^20 nodes and up");

static __device__ __align__(256) double scratch[kNoAllocDoubles];

namespace {
constexpr int kNoAllocDevices = 64;
double *g_scratch_dev[kNoAllocDevices] = {};
}  // namespace

int noalloc_scratch(double **out) {
  int dev = 0;
  NK_HIP(hipGetDevice(&dev));
  NK_CHECK(dev >= 0 && dev < kNoAllocDevices, NKH_ERR_ARG, "noalloc scratch: device %d", dev);
  if (!g_scratch_dev[dev]) {
    void *p = nullptr;
    NK_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    NK_CHECK(p != nullptr, NKH_ERR_HIP, "noalloc scratch: no device address");
    g_scratch_dev[dev] = static_cast<double *>(p);
  }
  if (out) *out = g_scratch_dev[dev];
  return NKH_OK;
}

int run_cggo_noalloc(Mesh &m, double *x, const double *f, const double *h1, const double *h2,
                     const double *mask, const double *mult, double tin, int maxit,
                     const nkh_params &prm, nkh_result *res, double *history_host) {
  NK_CHECK(m.n <= kNoAllocMaxN, NKH_ERR_ARG,
           "nkd_cggo_noalloc: %lld local nodes exceed its static scratch (at most %lld)",
           (long long)m.n, (long long)kNoAllocMaxN);
  NK_CHECK(m.gs.ngroups <= kNoAllocMaxN, NKH_ERR_ARG, "nkd_cggo_noalloc: %lld gs groups",
           (long long)m.gs.ngroups);
  double *sp = nullptr;
  NK_TRY(noalloc_scratch(&sp));
  // a view of the mesh whose solve buffers are the scratch: the geometry
  // and gather-scatter map are the mesh's own, nothing of it is changed.
  // Without a box: the state is copied back.
  Mesh v = m;
  v.reports = false;
  v.box = nullptr;
  v.ws = sp;
  v.ws_doubles = kNoAllocWs;
  v.red = sp + kNoAllocWs;
  v.st = reinterpret_cast<CgState *>(sp + kNoAllocWs + kNoAllocRed);
  v.gs.flag = reinterpret_cast<uint8_t *>(sp + kNoAllocWs + kNoAllocRed + kNoAllocState);
  SolveFacts facts;
  NK_TRY(gather_facts(v, h1, h2, mask, mult, const_cast<double *>(f), FactsAsk(), &facts,
                      cur_stream()));
  return drive_cggo<CgRun>(v, x, f, facts, mask, mult, tin, maxit, prm, res, history_host,
                           false);
}

// ---------------------------------------------------------------------------
// Batched Jacobi-PCG: several hmholtz solves (different meshes, h1/h2,
// masks, sizes; the same lx1 or not) iterate together, each with its own work
// space, state, gs group flags and stream.  The host takes the open solves in
// turn, waits for the report of one's exit test and enqueues its next
// iteration: they run side by side, in step with the slowest of them.  (A
// captured graph of eight iterations of all of them, built on every call, took
// longer to build than small solves take to run: five solves of 560 to 1,320
// elements 3.3 ms a call with it, 1.7 so; 64 of 336 elements 54 and 13 ms, one
// solve after another 23.)
// ---------------------------------------------------------------------------
struct CgBatch {
  int nb = 0;
  std::vector<int> mesh;
  std::vector<double *> ws, red;
  std::vector<CgState *> st;
  std::vector<uint8_t *> flag;
  std::vector<int64_t> nflag;
  std::vector<hipStream_t> streams;
  std::vector<hipEvent_t> ev;  // fork + one join per solve
  std::vector<HostBox *> box;
  std::vector<unsigned long long> seq;  // reports so far
  void release() {
    for (HostBox *q : box)
      if (q) (void)hipHostFree(q);
    box.clear();
    for (double *q : ws) (void)hipFree(q);
    for (double *q : red) (void)hipFree(q);
    for (CgState *q : st) (void)hipFree(q);
    for (uint8_t *q : flag) (void)hipFree(q);
    for (hipStream_t q : streams) (void)hipStreamDestroy(q);
    for (hipEvent_t q : ev) (void)hipEventDestroy(q);
    ws.clear();
    red.clear();
    st.clear();
    flag.clear();
    streams.clear();
    ev.clear();
  }
};

namespace {
std::vector<CgBatch *> g_batches;
}

int batch_create(int nb, const int *meshes, int *id) {
  NK_CHECK(nb >= 1 && nb <= 64 && meshes && id, NKH_ERR_ARG, "nkh_batch_create: bad arguments");
  CgBatch *B = new CgBatch();
  B->nb = nb;
  auto fail = [&](int rc) {
    B->release();
    delete B;
    return rc;
  };
  for (int k = 0; k < nb; ++k) {
    Mesh *m = get_mesh(meshes[k]);
    if (!m || !m->has_geom || !m->has_gs) {
      set_error("nkh_batch_create: mesh %d is not ready", meshes[k]);
      return fail(NKH_ERR_STATE);
    }
    NK_TRY(ensure_small(*m));
    double *w = nullptr, *r = nullptr;
    CgState *c = nullptr;
    uint8_t *fl = nullptr;
    hipStream_t q = nullptr;
    if (hipMalloc(&w, sizeof(double) * cg_ws_doubles(m->n)) != hipSuccess ||
        hipMalloc(&r, sizeof(double) * kRedSize) != hipSuccess ||
        hipMalloc(&c, sizeof(McgState)) != hipSuccess ||
        hipMalloc(&fl, (size_t)std::max<int64_t>(m->gs.ngroups, 1)) != hipSuccess ||
        hipStreamCreateWithFlags(&q, hipStreamNonBlocking) != hipSuccess) {
      (void)hipGetLastError();
      for (void *v : {(void *)w, (void *)r, (void *)c, (void *)fl}) (void)hipFree(v);
      if (q) (void)hipStreamDestroy(q);
      set_error("nkh_batch_create: out of device memory");
      return fail(NKH_ERR_NOMEM);
    }
    B->mesh.push_back(meshes[k]);
    B->ws.push_back(w);
    B->red.push_back(r);
    B->st.push_back(c);
    B->flag.push_back(fl);
    B->nflag.push_back(m->gs.ngroups);
    B->streams.push_back(q);
    B->box.push_back(nullptr);
    B->seq.push_back(0);
    const int rc = box_alloc(&B->box.back());
    if (rc != NKH_OK) return fail(rc);
  }
  for (int k = 0; k <= nb; ++k) {
    hipEvent_t e;
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      set_error("nkh_batch_create: event creation failed");
      return fail(NKH_ERR_HIP);
    }
    B->ev.push_back(e);
  }
  g_batches.push_back(B);
  *id = (int)g_batches.size() - 1;
  return NKH_OK;
}

int batch_meshes(int id, std::vector<int> *meshes) {
  NK_CHECK(id >= 0 && id < (int)g_batches.size() && g_batches[(size_t)id], NKH_ERR_ARG,
           "batch: bad handle %d", id);
  *meshes = g_batches[(size_t)id]->mesh;
  return NKH_OK;
}

int batch_destroy(int id) {
  NK_CHECK(id >= 0 && id < (int)g_batches.size() && g_batches[(size_t)id], NKH_ERR_ARG,
           "nkh_batch_destroy: bad handle %d", id);
  (void)hipDeviceSynchronize();
  g_batches[(size_t)id]->release();
  delete g_batches[(size_t)id];
  g_batches[(size_t)id] = nullptr;
  return NKH_OK;
}

int batch_facts(int id, const nkh_batch_solve *solves, bool chk, SolveFacts *out,
                hipStream_t s) {
  NK_CHECK(id >= 0 && id < (int)g_batches.size() && g_batches[(size_t)id], NKH_ERR_ARG,
           "batch: bad handle %d", id);
  CgBatch &B = *g_batches[(size_t)id];
  std::vector<BoxRef> rep((size_t)B.nb);
  FactsAsk ask;
  ask.mask_f = true;
  ask.chk = chk;
  for (int k = 0; k < B.nb; ++k) {
    Mesh *m = get_mesh(B.mesh[(size_t)k]);
    NK_CHECK(m && m->n > 0, NKH_ERR_STATE, "batch: mesh of solve %d is gone", k);
    NK_CHECK(m->gs.ngroups == B.nflag[(size_t)k], NKH_ERR_STATE,
             "batch: the gather-scatter map of solve %d changed", k);
    const nkh_batch_solve &q = solves[k];
    rep[(size_t)k] = Reports{B.box[(size_t)k], &B.seq[(size_t)k]}.next();
    NK_TRY(enqueue_facts(*m, q.h1, q.h2, q.mask, q.mult, q.rhs, ask, B.red[(size_t)k],
                         B.flag[(size_t)k], rep[(size_t)k], s));
  }
  for (int k = 0; k < B.nb; ++k) {
    NK_TRY(box_wait(rep[(size_t)k], s));
    out[k] = read_facts(*get_mesh(B.mesh[(size_t)k]), solves[k].h1, solves[k].h2,
                        B.box[(size_t)k]->v);
  }
  return NKH_OK;
}

namespace {

template <class Run>
int batch_drive(CgBatch &B, const double *const *x, const double *const *f,
                const SolveFacts *facts, const double *const *mask, const double *const *mult,
                const double *tin, int maxit, const nkh_params &prm, nkh_result *res,
                int *launches_out) {
  hipStream_t s = cur_stream();
  std::vector<Run> runs((size_t)B.nb);
  std::vector<int> active;
  for (int k = 0; k < B.nb; ++k) {
    Mesh *m = get_mesh(B.mesh[(size_t)k]);
    NK_CHECK(m && m->n > 0, NKH_ERR_STATE, "batch: mesh of solve %d is gone", k);
    // set-up of solve k on s
    NK_TRY(runs[(size_t)k].begin(*m, B.ws[(size_t)k], B.red[(size_t)k], B.st[(size_t)k],
                                 const_cast<double *>(x[k]), f[k], facts[k], mask[k], mult[k],
                                 tin[k], maxit, prm, false, s));
    if (runs[(size_t)k].trivial) continue;
    if (m->gs.ngroups > 0) runs[(size_t)k].flag = B.flag[(size_t)k];
    active.push_back(k);
  }
  // every solve on its own stream, after the set-up on s
  int launches = 0;
  if (!active.empty()) {
    NK_HIP(hipEventRecord(B.ev[0], s));
    int rc = NKH_OK;
    std::vector<int> open;
    auto no_events = [](int) -> hipEvent_t * { return nullptr; };
    for (int k : active) {
      Run &run = runs[(size_t)k];
      run.reports = Reports{B.box[(size_t)k], &B.seq[(size_t)k]};
      if (rc == NKH_OK && hipStreamWaitEvent(B.streams[(size_t)k], B.ev[0], 0) != hipSuccess) {
        set_error("batch: a solve's stream cannot wait for its set-up");
        rc = NKH_ERR_HIP;
      }
      if (rc == NKH_OK) rc = run.go_on(B.streams[(size_t)k], no_events);
      open.push_back(k);
    }
    // round robin over the solves that have not ended: their report is read,
    // then their next iteration enqueued
    while (rc == NKH_OK && !open.empty()) {
      std::vector<int> next;
      for (int k : open) {
        Run &run = runs[(size_t)k];
        hipStream_t q = B.streams[(size_t)k];
        CgState hs;
        if ((rc = run.wait(&hs, q)) != NKH_OK) break;
        if (hs.done) {
          run.result(hs, &res[k]);
          continue;
        }
        if (run.launched > run.niter + 1) {
          set_error("batch: a state machine did not terminate");
          rc = NKH_ERR_STATE;
          break;
        }
        if ((rc = run.go_on(q, no_events)) != NKH_OK) break;
        next.push_back(k);
      }
      open.swap(next);
    }
    // the caller's stream goes on after every solve's, also after an error
    // (which leaves work in flight)
    for (int k : active) {
      if (rc != NKH_OK) (void)hipStreamSynchronize(B.streams[(size_t)k]);
      launches = std::max(launches, runs[(size_t)k].launched);
      (void)hipEventRecord(B.ev[(size_t)k + 1], B.streams[(size_t)k]);
      (void)hipStreamWaitEvent(s, B.ev[(size_t)k + 1], 0);
    }
    NK_TRY(rc);
  }
  int zero = -1;  // a solve whose x = 0 is enqueued on s
  for (int k = 0; k < B.nb; ++k)
    if (runs[(size_t)k].trivial) {
      runs[(size_t)k].result(CgState{}, &res[k]);
      zero = k;
    }
  if (zero >= 0)
    NK_TRY(box_join(Reports{B.box[(size_t)zero], &B.seq[(size_t)zero]}.next(), s));
  if (launches_out) *launches_out = launches;
  return NKH_OK;
}

}  // namespace

int run_cggo_batch(int id, const double *const *x, const double *const *f,
                   const SolveFacts *facts, const double *const *mask,
                   const double *const *mult, const double *tin, int maxit,
                   const nkh_params &prm, nkh_result *res, int *launches_out) {
  NK_CHECK(id >= 0 && id < (int)g_batches.size() && g_batches[(size_t)id], NKH_ERR_ARG,
           "batch: bad handle %d", id);
  CgBatch &B = *g_batches[(size_t)id];
  if (prm.precision == 2)
    return batch_drive<McgRun>(B, x, f, facts, mask, mult, tin, maxit, prm, res, launches_out);
  return batch_drive<CgRun>(B, x, f, facts, mask, mult, tin, maxit, prm, res, launches_out);
}

}  // namespace nekamd
