// Right-preconditioned restarted GMRES with the h1mg V-cycle (gmres.f:304-545
// hmh_gmres), the reference's default pressure solver (param(42) = 0).
//
// Krylov vectors V (m+1) and preconditioned vectors Z (m) stay in HBM; the
// small Hessenberg problem (Givens rotations, back substitution) runs on the
// host from the Gram-Schmidt coefficients each step reports.  Dots are
// fixed-grid partial sums reduced in a fixed order.  ml = mu = 1 in the
// reference (uzawa_gmres_split, gmres.f:252-271), so there is no scaling.
#include <algorithm>
#include <cmath>
#include <vector>

#include "hsmg.h"
#include "tails.h"

namespace nekamd {

namespace {

constexpr int kGmBlocks = 2048;  // room for the partials of one sum (dot_blocks)
constexpr int kDotChunk = 8;
// last_block's counters: a set for each chunk of products, one for the norms
constexpr int kCounters = (kGmresM + kDotChunk - 1) / kDotChunk + 1;
constexpr int kCounterInts = 2 * kCounterDoubles;

#define NK_LOOP(i, n)                                                          \
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < (n); \
       i += (int64_t)gridDim.x * blockDim.x)

// *out = the sum over the grid of a, and in the last block that and the nh
// doubles h before it to the host
__device__ __forceinline__ void norm_and_report(double a, double *part, int *cnt, double *out,
                                                const double *h, int nh, const BoxRef &rep) {
  __shared__ double sa[4];
  for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
  if ((threadIdx.x & 63) == 0) sa[threadIdx.x >> 6] = a;
  __syncthreads();
  if (threadIdx.x == 0) leave(part + blockIdx.x, ((sa[0] + sa[1]) + sa[2]) + sa[3]);
  if (!last_block(cnt, gridDim.x)) return;
  double t[1];
  sum_left(part, 0, gridDim.x, t);
  if (threadIdx.x != 0) return;
  *out = t[0];
  for (int i = 0; i < nh; ++i) rep.b->v[i] = h[i];
  rep.b->v[nh] = t[0];
  box_report(rep);
}
static_assert(kGmresM + 1 <= (int)(sizeof(HostBox::v) / sizeof(double)), "a report holds a step");

// r = res - mask*w; *a2 = sum r*r*wt, reported   (r = res - A x with ax's mask)
__global__ void __launch_bounds__(256)
    k_gm_resid(double *__restrict__ r, const double *__restrict__ res,
               const double *__restrict__ w, const double *__restrict__ mask,
               const double *__restrict__ wt, int64_t n, int first, double *part, int *cnt,
               double *a2, BoxRef rep) {
  double a = 0.0;
  NK_LOOP(i, n) {
    const double ri = first ? res[i] : res[i] - w[i] * mask[i];
    r[i] = ri;
    a += (ri * ri) * wt[i];
  }
  norm_and_report(a, part, cnt, a2, nullptr, 0, rep);
}

// h_c = sum (mask*w v_c)*wt for the C vectors v at V (vlsc3, gmres.f:466)
template <int C>
__device__ __forceinline__ void gm_dots(const double *__restrict__ w,
                                        const double *__restrict__ mask,
                                        const double *__restrict__ V, int64_t n,
                                        const double *__restrict__ wt, double *part, int *cnt,
                                        double *h, double (*sw)[4]) {
  double acc[C] = {};
  NK_LOOP(q, n) {
    double v[C];
#pragma unroll
    for (int c = 0; c < C; ++c) v[c] = V[(int64_t)c * n + q];
    const double wq = w[q] * mask[q], wv = wt[q];
#pragma unroll
    for (int c = 0; c < C; ++c) acc[c] += (wq * v[c]) * wv;
  }
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    double a = acc[c];
    for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
    if (lane == 0) sw[c][wave] = a;
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t < C)
    leave(part + (int64_t)t * kGmBlocks + blockIdx.x, ((sw[t][0] + sw[t][1]) + sw[t][2]) + sw[t][3]);
  if (!last_block(cnt, gridDim.x)) return;
  for (int c = wave; c < C; c += 4) {
    const double *p = part + (int64_t)c * kGmBlocks;
    double b[4] = {};
    int q = lane;
    for (; q + 192 < (int)gridDim.x; q += 256) {
      double l[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) l[u] = left(p + q + 64 * u);
#pragma unroll
      for (int u = 0; u < 4; ++u) b[u] += l[u];
    }
    for (; q < (int)gridDim.x; q += 64) b[0] += left(p + q);
    double a = (b[0] + b[1]) + (b[2] + b[3]);
    for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
    if (lane == 0) h[c] = a;
  }
}

// Chunk blockIdx.y of the j products, kDotChunk of them a chunk (each reads w,
// mask and wt once); cnt: a set of counters a chunk.  The last block of a chunk adds
// up its products, a wavefront each.
__global__ void __launch_bounds__(256)
    k_gm_dots(const double *__restrict__ w, const double *__restrict__ mask,
              const double *__restrict__ V, int64_t n, int j, const double *__restrict__ wt,
              double *part, int *cnt, double *h) {
  __shared__ double sw[kDotChunk][4];
  const int i0 = blockIdx.y * kDotChunk;
  V += (int64_t)i0 * n;
  part += (int64_t)i0 * kGmBlocks;
  h += i0;
  cnt += blockIdx.y * kCounterInts;
  switch (j - i0) {
    case 1: return gm_dots<1>(w, mask, V, n, wt, part, cnt, h, sw);
    case 2: return gm_dots<2>(w, mask, V, n, wt, part, cnt, h, sw);
    case 3: return gm_dots<3>(w, mask, V, n, wt, part, cnt, h, sw);
    case 4: return gm_dots<4>(w, mask, V, n, wt, part, cnt, h, sw);
    case 5: return gm_dots<5>(w, mask, V, n, wt, part, cnt, h, sw);
    case 6: return gm_dots<6>(w, mask, V, n, wt, part, cnt, h, sw);
    case 7: return gm_dots<7>(w, mask, V, n, wt, part, cnt, h, sw);
    default: return gm_dots<8>(w, mask, V, n, wt, part, cnt, h, sw);
  }
}
static_assert(kDotChunk == 8, "the cases of k_gm_dots");

// w = mask*w - h_i v_i for i = 0..j-1 in order (add2s2), then *a2 = sum w*w*wt,
// reported with h
__global__ void __launch_bounds__(256)
    k_gm_orth(double *__restrict__ w, const double *__restrict__ mask,
              const double *__restrict__ V, const double *__restrict__ h, int j,
              const double *__restrict__ wt, int64_t n, double *part, int *cnt, double *a2,
              BoxRef rep) {
  double a = 0.0;
  NK_LOOP(q, n) {
    double wq = w[q] * mask[q];
    const double wv = wt[q];
    int i = 0;
    for (; i + 4 <= j; i += 4) {
      double v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = V[(int64_t)(i + u) * n + q];
#pragma unroll
      for (int u = 0; u < 4; ++u) wq = wq + (-h[i + u]) * v[u];
    }
    for (; i < j; ++i) wq = wq + (-h[i]) * V[(int64_t)i * n + q];
    w[q] = wq;
    a += (wq * wq) * wv;
  }
  norm_and_report(a, part, cnt, a2, h, j, rep);
}

// v = u / sqrt(*a2) (cmult2: the next Krylov vector), w = v * mgmask (the
// right-hand side that h1mg_solve masks in place).  It needs no host: the
// step's report is on its way meanwhile.
__global__ void __launch_bounds__(256)
    k_gm_next(double *__restrict__ v, double *w, const double *u, const double *__restrict__ a2,
              const double *__restrict__ mask, int64_t n) {
  const double s = 1.0 / sqrt(*a2);
  NK_LOOP(i, n) {
    const double vi = u[i] * s;
    v[i] = vi;
    w[i] = vi * mask[i];
  }
}

struct GmCoef {
  double c[kGmresM];
};
// x = x + c_i z_i for i = 0..j-1 in order
__global__ void k_gm_xupd(double *__restrict__ x, const double *__restrict__ Z, GmCoef c, int j,
                          int64_t n) {
  NK_LOOP(q, n) {
    double xq = x[q];
    for (int i = 0; i < j; ++i) xq = xq + c.c[i] * Z[(int64_t)i * n + q];
    x[q] = xq;
  }
}

// x = 0, and the counters of the kernels that end in last_block
__global__ void k_gm_zero(double *__restrict__ x, int64_t n, int *__restrict__ cnt) {
  if (blockIdx.x == 0)
    for (int k = 0; k < kCounters; ++k) clear_counters(cnt + k * kCounterInts);
  NK_LOOP(i, n) x[i] = 0.0;
}

}  // namespace

int run_gmres(Mesh &m, double *res, const SolveFacts &facts, const double *wt,
              const double *mask, int maxit, const nkh_params &prm, nkh_result *out,
              double *rnorm_history) {
  NK_CHECK(m.mg, NKH_ERR_STATE, "hmh_gmres needs the multigrid hierarchy (nkh_mg_setup)");
  NK_CHECK(prm.param40 == 0 || prm.param40 == 1, NKH_ERR_UNSUPPORTED,
           "hmh_gmres: coarse solver param40=%d (0 exact, 1 one AMG V-cycle)", prm.param40);
  Mg &mg = *m.mg;
  hipStream_t s = cur_stream();
  const Coef h1 = facts.c1(), h2 = facts.c2();
  const int64_t n = m.n;
  const int M = kGmresM;
  if (!mg.gV) {
    NK_TRY(mg_dalloc(&mg.gV, (int64_t)(M + 1) * n));
    NK_TRY(mg_dalloc(&mg.gZ, (int64_t)M * n));
    for (double **p : {&mg.gx, &mg.gr, &mg.gw}) NK_TRY(mg_dalloc(p, n));
    NK_TRY(mg_dalloc(&mg.gpart, (int64_t)(M + 2) * kGmBlocks));
    NK_TRY(mg_dalloc(&mg.gsm, 2 * (M + 2) + kCounters * kCounterDoubles));
  }
  double *V = mg.gV, *Z = mg.gZ, *x = mg.gx, *r = mg.gr, *w = mg.gw, *part = mg.gpart;
  // h(1..j), the squared norm after them, the counters
  double *dh = mg.gsm, *da2 = mg.gsm + (M + 2);
  int *cnt = reinterpret_cast<int *>(mg.gsm + 2 * (M + 2));
  int *ncnt = cnt + (kCounters - 1) * kCounterInts;
  NK_TRY(ensure_small(m));
  const double *mgmask = mg.lev[mg.lmax].mask;
  const dim3 G(dot_blocks(n)), B(256);
  const double norm_fac = 1.0 / std::sqrt(m.vol);
  const bool nullsp = mg_null_space_on(mg, h2);
  // hmholtz.f-style tolerance (gmres.f:352-356)
  double tolps = 0.0;
  NK_TRY(run_chktcg1(m, &tolps, facts));
  if (prm.param21 > 0 && tolps > std::fabs(prm.param21)) tolps = std::fabs(prm.param21);
  if (prm.istep == 0) tolps = 1.e-4;
  double tolpss = tolps;
  std::vector<double> H((size_t)M * M, 0.0), gam(M + 1, 0.0), c(M, 0.0), sn(M, 0.0);
  auto HH = [&](int i, int jj) -> double & { return H[(size_t)i + (size_t)M * jj]; };
  hipLaunchKernelGGL(k_gm_zero, dim3(mg_grid(n)), B, 0, s, x, n, cnt);
  double div0 = 0.0, rnorm = 0.0;
  int iter = 0, j = 0;
  bool iconv = false;
  while (!iconv) {
    // r = res (first) or res - A x
    if (iter > 0) {
      NK_TRY(launch_axhelm(m, w, x, h1, h2, s));
      NK_TRY(gs_op(m.gs, w, 0, s));
    }
    const BoxRef rep0 = m.next_report();
    hipLaunchKernelGGL(k_gm_resid, G, B, 0, s, r, res, w, mask, wt, n, iter == 0 ? 1 : 0, part,
                       ncnt, da2, rep0);
    hipLaunchKernelGGL(k_gm_next, dim3(mg_grid(n)), B, 0, s, V, w, r, da2, mgmask, n);
    NK_HIP(hipGetLastError());
    NK_TRY(box_wait(rep0, s));
    gam[0] = std::sqrt(rep0.b->v[0]);
    if (iter == 0) {
      div0 = gam[0] * norm_fac;
      if (prm.param21 < 0) tolpss = std::fabs(prm.param21) * div0;
    }
    rnorm = 0.0;
    if (gam[0] == 0.0) break;
    for (j = 1; j <= M; ++j) {
      iter += 1;
      double *zj = Z + (int64_t)(j - 1) * n;
      NK_TRY(mg_solve(m, zj, w, s, prm.param40, prm.precision));
      if (nullsp) NK_TRY(mg_ortho(mg, zj, n, s));  // gmres.f:427
      NK_TRY(launch_axhelm(m, w, zj, h1, h2, s));
      NK_TRY(gs_op(m.gs, w, 0, s));
      // classical Gram-Schmidt, one pass (gmres.f:464-474)
      hipLaunchKernelGGL(k_gm_dots, dim3(G.x, (j + kDotChunk - 1) / kDotChunk), B, 0, s, w, mask,
                         V, n, j, wt, part, cnt, dh);
      const BoxRef rep = m.next_report();
      hipLaunchKernelGGL(k_gm_orth, G, B, 0, s, w, mask, V, dh, j, wt, n, part, ncnt, da2, rep);
      if (j < M)  // (not read if this step is the last)
        hipLaunchKernelGGL(k_gm_next, dim3(mg_grid(n)), B, 0, s, V + (int64_t)j * n, w, w, da2,
                           mgmask, n);
      NK_HIP(hipGetLastError());
      NK_TRY(box_wait(rep, s));
      for (int i = 1; i <= j; ++i) HH(i - 1, j - 1) = rep.b->v[i - 1];
      const double a2 = rep.b->v[j];
      for (int i = 1; i <= j - 1; ++i) {  // previous Givens rotations
        const double temp = HH(i - 1, j - 1);
        HH(i - 1, j - 1) = c[i - 1] * temp + sn[i - 1] * HH(i, j - 1);
        HH(i, j - 1) = -sn[i - 1] * temp + c[i - 1] * HH(i, j - 1);
      }
      const double alpha = std::sqrt(a2);
      rnorm = 0.0;
      if (alpha == 0.0) {
        iconv = true;
        break;
      }
      const double l = std::sqrt(HH(j - 1, j - 1) * HH(j - 1, j - 1) + alpha * alpha);
      const double temp = 1.0 / l;
      c[j - 1] = HH(j - 1, j - 1) * temp;
      sn[j - 1] = alpha * temp;
      HH(j - 1, j - 1) = l;
      gam[j] = -sn[j - 1] * gam[j - 1];
      gam[j - 1] = c[j - 1] * gam[j - 1];
      rnorm = std::fabs(gam[j]) * norm_fac;
      if (rnorm_history) rnorm_history[iter - 1] = rnorm;
      if (iter + 1 > maxit || rnorm < tolpss) {
        iconv = true;
        break;
      }
      if (j == M) break;  // restart
    }
    if (j > M) j = M;
    // back substitution c = H^-1 gamma; x += sum c_i z_i (gmres.f:518-529)
    for (int k = j; k >= 1; --k) {
      double temp = gam[k - 1];
      for (int i = j; i >= k + 1; --i) temp = temp - HH(k - 1, i - 1) * c[i - 1];
      c[k - 1] = temp / HH(k - 1, k - 1);
    }
    GmCoef cj{};
    std::copy(c.begin(), c.begin() + j, cj.c);
    hipLaunchKernelGGL(k_gm_xupd, dim3(mg_grid(n)), B, 0, s, x, Z, cj, j, n);
    NK_HIP(hipGetLastError());
  }
  // res = x (copy, gmres.f:535), orthogonalised against the null space (:534)
  NK_HIP(hipMemcpyAsync(res, x, sizeof(double) * n, hipMemcpyDeviceToDevice, s));
  if (nullsp) NK_TRY(mg_ortho(mg, res, n, s));
  NK_TRY(box_join(m.next_report(), s));
  if (out) {
    out->niter = iter;
    out->converged = rnorm < tolpss || gam[0] == 0.0;
    out->rbn0 = div0;
    out->rbn2 = rnorm;
    out->tol = tolpss;
  }
  return NKH_OK;
}

}  // namespace nekamd
