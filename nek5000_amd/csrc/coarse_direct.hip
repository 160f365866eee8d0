// Direct solver of the coarse problem (the reference factors it exactly, with
// XXT: crs_xxt.c:922-960).
//
// The unknowns are dissected once: recursive bisection along the coordinates
// cuts them into np parts that touch each other only through a separator.  Of
// every part's block A_pp, and of the separator's Schur complement
// S = A_ss - sum_p A_sp A_pp^-1 A_ps, the explicit inverse is formed on the
// GPU and kept; the couplings stay sparse.  A solve is then
//   y_p = A_pp^-1 b_p                 k_dir_parts<false>
//   g   = b_s - sum_p A_sp y_p        k_dir_sep_rhs
//   x_s = S^-1 g                      k_dir_sep
//   x_p = A_pp^-1 (b_p - A_ps x_s)    k_dir_parts<true>
// four launches that stream the inverses, with no iteration, no reduction
// and no host wait.  Small problems are one part without a separator: a plain
// inverse, one launch.  The set-up measures the residuals of two solves, and has
// ill-conditioned problems (very stretched elements without a Dirichlet face)
// refined: k_dir_resid, the same launches on the residual, k_dir_add.
//
// Why: preconditioned CG on this problem is a serial chain of about 16
// iterations of 6 to 10 kernels, each 3 to 12 us long whatever the size.
// Measured on boxes of trilinear elements with varying coefficients, us per
// solve, AMG-PCG to 1e-13 -> direct (and direct with its matrices out of the
// caches): n = 1,320 652 -> 5 (15), 4,080 731 -> 20 (31), 7,980 773 -> 26
// (48), 24,360 1,085 -> 118 (185), 46,620 1,411 -> 295 (359).  Relative
// residuals 5e-16 to 5e-15 against the PCG's 1e-14 to 9e-14; with one
// unknown held (no Dirichlet face) 2e-13 to 3e-12 against 4e-13 to 2e-12.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "coarse_direct.h"

namespace nekamd {

namespace {

constexpr int kTile = 64;  // tile of the inversion, and padding of its matrices
// The bytes of inverses one solve may stream.  A cube-like problem reaches
// them at about 60,000 unknowns, where the solve still takes a third of the
// PCG's time; the set-up (2 n^3 flops of the separator) then takes 0.3 s and
// grows with n^2, which few solves would pay for much further on.  More than
// kMaxUnknowns are not dissected at all.
constexpr double kMaxStream = 2.2e9;
constexpr int kMaxUnknowns = 100000;
// The least share of its matrix's diagonal entry that a pivot may be: a second
// region without a Dirichlet face leaves pivots of -2e-14 to 3e-14.
constexpr double kPivotMin = 1e-13;
// Relative residuals that the set-up measures (refine_to).  The inversion's
// grow with the square of the condition number and reach what rounding allows
// by one to three steps of refinement, which a solve takes above kGoodResidual.
// Above kMaxResidual, refined, the inverses are not used.  Measured on boxes of
// 1,320 to 54,834 unknowns, and in brackets the AMG-PCG (of at most 500
// iterations) on the same right-hand sides: Dirichlet faces, elements up to
// 1:1,000, 2e-15 to 9e-14 (1e-14 to 2e-10).  Neumann faces only: cubes 1e-13
// to 1e-12 (5e-14 to 3e-13), 1:10 3e-12 to 2e-11 (4e-12 to 3e-11), 1:100 4e-10
// to 3e-9 (5e-4 to 5e-2), rods of 1:1,000 4e-7 to 8e-7, refined 8e-9 to 7e-8
// (5e-8 to 29), plates of 1:1,000 3e-8 to 3e-5, refined 1e-8 to 7e-8 (0.1 to
// 28), of 1:10,000 3e-6 to 2e-1, refined 1e-6 to 7e-6 (40 to 850).
constexpr double kGoodResidual = 1e-8, kMaxResidual = 1e-4;
constexpr int kMaxRefine = 3;
// a part's right-hand side is staged in LDS
constexpr int kMaxPart = 4096;
// Cost model of a dissection, fitted to solves with the matrices out of the
// caches, as the rest of a V-cycle leaves them: streaming rate, and what one
// launch and the four launches take besides.  A plain inverse up to about
// 2,200 unknowns (n = 1,320: 15 us against 23 in parts; 3,600: 55 against 29).
constexpr double kStreamRate = 3.0e12, kPlainTime = 11e-6, kPartsTime = 20e-6;

int pad_up(int v) { return (v + kTile - 1) / kTile * kTile; }

// ---------------------------------------------------------------------------
// dissection (host)
// ---------------------------------------------------------------------------
struct Dissection {
  std::vector<std::vector<int32_t>> part;
  std::vector<int32_t> sep;
  double bytes() const {  // streamed by one solve
    int k = 0;
    for (const auto &p : part) k = std::max(k, (int)p.size());
    const double kp = pad_up(k), sp = sep.size();
    return 8.0 * ((part.size() > 1 ? 2.0 : 1.0) * (double)part.size() * kp * kp + sp * sp);
  }
  double seconds() const {
    return bytes() / kStreamRate + (part.size() > 1 ? kPartsTime : kPlainTime);
  }
};

// Split every part in two halves by the coordinate whose cut leaves the
// smallest separator; the separator is the upper half's unknowns next to the
// lower half.
Dissection bisect(const Dissection &d, const std::vector<int32_t> &rp,
                  const std::vector<int32_t> &ci, const std::vector<double> &xyz) {
  Dissection out;
  out.sep = d.sep;
  const int n = (int)rp.size() - 1;
  std::vector<int8_t> side((size_t)n, 0);  // 1 lower half, 2 upper half of the part at hand
  for (const auto &p : d.part) {
    std::vector<int32_t> best_lo, best_hi, best_sep;
    for (int dir = 0; dir < 3; ++dir) {
      std::vector<int32_t> q(p);
      const size_t h = q.size() / 2;
      std::nth_element(q.begin(), q.begin() + (std::ptrdiff_t)h, q.end(),
                       [&](int32_t a, int32_t b) {
                         const double xa = xyz[3 * (size_t)a + dir], xb = xyz[3 * (size_t)b + dir];
                         return xa != xb ? xa < xb : a < b;
                       });
      for (size_t t = 0; t < q.size(); ++t) side[(size_t)q[t]] = t < h ? 1 : 2;
      std::vector<int32_t> hi, sp;
      for (size_t t = h; t < q.size(); ++t) {
        const int32_t i = q[t];
        bool cut = false;
        for (int32_t e = rp[i]; e < rp[i + 1] && !cut; ++e) cut = side[(size_t)ci[e]] == 1;
        (cut ? sp : hi).push_back(i);
      }
      for (int32_t i : q) side[(size_t)i] = 0;
      if (dir == 0 || sp.size() < best_sep.size()) {
        best_lo.assign(q.begin(), q.begin() + (std::ptrdiff_t)h);
        best_hi.swap(hi);
        best_sep.swap(sp);
      }
    }
    if (!best_lo.empty()) out.part.push_back(std::move(best_lo));
    if (!best_hi.empty()) out.part.push_back(std::move(best_hi));
    out.sep.insert(out.sep.end(), best_sep.begin(), best_sep.end());
  }
  return out;
}

// ---------------------------------------------------------------------------
// inversion (device): blocked Gauss-Jordan in place, without pivoting (the
// matrices are symmetric positive definite), nb matrices of K x K at once
// (blockIdx.z).  Per block column: the pivot tile is inverted in LDS, the
// block row and the block column are set aside, and every other tile gets
// its rank-64 update on the FP64 matrix cores.
// ---------------------------------------------------------------------------
typedef double nk_dd4 __attribute__((ext_vector_type(4)));

// dg: the diagonals before the elimination, K per matrix; a pivot of less than
// kPivotMin of its own is rounding
__global__ void __launch_bounds__(256)
    k_gj_pivot(const double *__restrict__ A, int K, int kb, const double *__restrict__ dg,
               double *__restrict__ P, int *bad) {
  __shared__ double a[kTile][kTile + 1];
  dg += (int64_t)blockIdx.z * K + kb * kTile;
  const double *Ab = A + (int64_t)blockIdx.z * K * K + (int64_t)kb * kTile * K + kb * kTile;
  for (int t = threadIdx.x; t < kTile * kTile; t += 256)
    a[t / kTile][t % kTile] = Ab[(int64_t)(t / kTile) * K + t % kTile];
  __syncthreads();
  const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
  for (int j = 0; j < kTile; ++j) {
    const double pj = a[j][j];
    if (threadIdx.x == 0 && !(pj > 0.0 && pj > kPivotMin * dg[j] && pj < 1e300))
      atomicOr(bad, 1);
    const double pv = 1.0 / pj;
    const double rj = (c == j ? 1.0 : a[j][c]) * pv;  // scaled pivot row
    double f[kTile / 4];
#pragma unroll
    for (int q = 0; q < kTile / 4; ++q) f[q] = a[r0 + 4 * q][j];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kTile / 4; ++q) {
      const int r = r0 + 4 * q;
      if (r == j) a[r][c] = rj;
      else a[r][c] = (c == j ? 0.0 : a[r][c]) - f[q] * rj;
    }
    __syncthreads();
  }
  double *Pb = P + (int64_t)blockIdx.z * kTile * kTile;
  for (int t = threadIdx.x; t < kTile * kTile; t += 256) Pb[t] = a[t / kTile][t % kTile];
}

// acc = (16 rows of X from row 16 w) * Y for one wavefront w of four: X 64 x
// 64 at row pitch xp in global memory, Y in LDS; acc[t] holds the 16 x 16 tile
// of columns 16 t (row 4 v + l/16 and column l%16 in register v of lane l)
__device__ __forceinline__ void tile_product(const double *__restrict__ X, int64_t xp,
                                             const double (*Y)[kTile + 1], nk_dd4 acc[4]) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
  double x[kTile / 4];
#pragma unroll
  for (int c = 0; c < kTile / 4; ++c) x[c] = X[(int64_t)(16 * w + lr) * xp + 4 * c + lg];
#pragma unroll
  for (int t = 0; t < 4; ++t) acc[t] = nk_dd4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < kTile / 4; ++c)
#pragma unroll
    for (int t = 0; t < 4; ++t)
      acc[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[c], Y[4 * c + lg][16 * t + lr], acc[t], 0,
                                                    0, 0);
}

// R = P * (block row kb), and C = (block column kb), for tile blockIdx.x
__global__ void __launch_bounds__(256)
    k_gj_panel(const double *__restrict__ A, int K, int kb, const double *__restrict__ P,
               double *__restrict__ R, double *__restrict__ C) {
  __shared__ double Y[kTile][kTile + 1];
  const int jt = blockIdx.x;
  const double *Am = A + (int64_t)blockIdx.z * K * K;
  if (blockIdx.y == 1) {
    double *Cb = C + (int64_t)blockIdx.z * K * kTile;
    for (int t = threadIdx.x; t < kTile * kTile; t += 256) {
      const int64_t r = (int64_t)jt * kTile + t / kTile;
      Cb[r * kTile + t % kTile] = Am[r * K + kb * kTile + t % kTile];
    }
    return;
  }
  for (int t = threadIdx.x; t < kTile * kTile; t += 256)
    Y[t / kTile][t % kTile] = Am[((int64_t)kb * kTile + t / kTile) * K + jt * kTile + t % kTile];
  __syncthreads();
  nk_dd4 acc[4];
  tile_product(P + (int64_t)blockIdx.z * kTile * kTile, kTile, Y, acc);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
  double *Rb = R + (int64_t)blockIdx.z * K * kTile;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v)
      Rb[(int64_t)(16 * w + 4 * v + lg) * K + jt * kTile + 16 * t + lr] = acc[t][v];
}

__global__ void __launch_bounds__(256)
    k_gj_update(double *__restrict__ A, int K, int kb, const double *__restrict__ P,
                const double *__restrict__ R, const double *__restrict__ C) {
  __shared__ double Y[kTile][kTile + 1];
  const int jt = blockIdx.x, it = blockIdx.y;
  double *At = A + (int64_t)blockIdx.z * K * K + (int64_t)it * kTile * K + jt * kTile;
  const double *Pb = P + (int64_t)blockIdx.z * kTile * kTile;
  const double *Rb = R + (int64_t)blockIdx.z * K * kTile;
  if (it == kb) {  // the block row: P in the pivot tile, R elsewhere
    for (int t = threadIdx.x; t < kTile * kTile; t += 256)
      At[(int64_t)(t / kTile) * K + t % kTile] =
          jt == kb ? Pb[t] : Rb[(int64_t)(t / kTile) * K + jt * kTile + t % kTile];
    return;
  }
  for (int t = threadIdx.x; t < kTile * kTile; t += 256)
    Y[t / kTile][t % kTile] =
        jt == kb ? Pb[t] : Rb[(int64_t)(t / kTile) * K + jt * kTile + t % kTile];
  __syncthreads();
  nk_dd4 acc[4];
  tile_product(C + (int64_t)blockIdx.z * K * kTile + (int64_t)it * kTile * kTile, kTile, Y, acc);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, lr = lane & 15, lg = lane >> 4;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      double *a = At + (int64_t)(16 * w + 4 * v + lg) * K + 16 * t + lr;
      *a = (jt == kb ? 0.0 : *a) - acc[t][v];
    }
}

// identity, nb matrices of K x K
__global__ void k_dir_eye(double *__restrict__ A, int K, int64_t total) {
  const int64_t kk = (int64_t)K * K;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t t = q % kk;
    A[q] = (t / K == t % K) ? 1.0 : 0.0;
  }
}

// dg = the diagonals, nb matrices of K x K
__global__ void k_dir_diag(const double *__restrict__ A, int K, int nb, double *__restrict__ dg) {
  for (int q = blockIdx.x * 256 + threadIdx.x; q < nb * K; q += gridDim.x * 256)
    dg[q] = A[(int64_t)(q / K) * K * K + (int64_t)(q % K) * K + q % K];
}

// A[at[q]] = v[q]
__global__ void k_dir_put(double *__restrict__ A, const int64_t *__restrict__ at,
                          const double *__restrict__ v, int64_t cnt) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < cnt;
       q += (int64_t)gridDim.x * blockDim.x)
    A[at[q]] = v[q];
}

// One part's share of the Schur complement.  Its nb neighbouring separator
// rows bl[0..nb); entries [cp[q], cp[q+1]) of column q: local rows cr of the
// part with A(row, q) = cv and A(q, row) = rv.
// T(row, q) = sum_c inv(row, c) A(c, q)
__global__ void __launch_bounds__(256)
    k_dir_schur_t(double *__restrict__ T, const double *__restrict__ inv, int kld, int k, int nb,
                  const int32_t *__restrict__ cp, const int32_t *__restrict__ cr,
                  const double *__restrict__ cv) {
  const int q = blockIdx.x * 64 + (threadIdx.x & 63);
  const int row = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (q >= nb || row >= k) return;
  double a = 0.0;
  for (int e = cp[q]; e < cp[q + 1]; ++e) a += inv[(int64_t)row * kld + cr[e]] * cv[e];
  T[(int64_t)row * nb + q] = a;
}
// S(p, q) -= sum_r A(p, r) T(r, q)
__global__ void __launch_bounds__(256)
    k_dir_schur_s(double *__restrict__ S, int64_t sld, const double *__restrict__ T, int nb,
                  const int32_t *__restrict__ bl, const int32_t *__restrict__ cp,
                  const int32_t *__restrict__ cr, const double *__restrict__ rv) {
  const int q = blockIdx.x * 64 + (threadIdx.x & 63);
  const int p = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (q >= nb || p >= nb) return;
  double a = 0.0;
  for (int e = cp[p]; e < cp[p + 1]; ++e) a += rv[e] * T[(int64_t)cr[e] * nb + q];
  S[bl[p] * sld + bl[q]] -= a;
}

// ---------------------------------------------------------------------------
// the solve (device)
// ---------------------------------------------------------------------------
typedef double nk_dd2 __attribute__((ext_vector_type(2)));

// NR consecutive rows of a row-major matrix (pitch ld, even) times v[0..len),
// len even and v readable to there: the sums on every lane of the wavefront
template <int NR>
__device__ __forceinline__ void row_products(const double *__restrict__ m, int64_t ld, int len,
                                             const double *v, double (&sum)[NR]) {
  const int lane = threadIdx.x & 63;
  double a[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) a[r] = 0.0;
#pragma unroll 2
  for (int j = 2 * lane; j < len; j += 128) {
    const nk_dd2 x = *reinterpret_cast<const nk_dd2 *>(v + j);
#pragma unroll
    for (int r = 0; r < NR; ++r) {
      const nk_dd2 t = *reinterpret_cast<const nk_dd2 *>(m + r * ld + j);
      a[r] += t.x * x.x;
      a[r] += t.y * x.y;
    }
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) {
    for (int o = 32; o > 0; o >>= 1) a[r] += __shfl_xor(a[r], o, 64);
    sum[r] = a[r];
  }
}

constexpr int kRows = 4;  // rows per wavefront
// at most this many rows in all: one row per wavefront, to fill the chip
constexpr int kFewRows = 4096;

// Part blockIdx.y, rows 4 NR blockIdx.x ...: BACK false, y = inv b; true, x =
// inv (b - A_ps x_s) into the unknowns' own order.  Bound by the stream of
// inv; each block stages the part's right-hand side in LDS and reuses each of
// its values for NR rows per load.
template <bool BACK, int NR>
__global__ void __launch_bounds__(256)
    k_dir_parts(const double *__restrict__ inv, int kld, const int32_t *__restrict__ prow,
                const double *__restrict__ b, double *__restrict__ y,
                const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                const double *__restrict__ cv, const double *__restrict__ xs,
                double *__restrict__ x) {
  extern __shared__ double v[];
  const int64_t p0 = (int64_t)blockIdx.y * kld;
  const int32_t *pr = prow + p0;
  const int r0 = blockIdx.x * 4 * NR;
  if (pr[r0] < 0) return;  // padding follows the part's rows
  for (int j = threadIdx.x; j < kld; j += 256) {
    const int u = pr[j];
    double t = u >= 0 ? b[u] : 0.0;
    if constexpr (BACK) {
      if (u >= 0)
        for (int e = rp[p0 + j]; e < rp[p0 + j + 1]; ++e) t -= cv[e] * xs[ci[e]];
    }
    v[j] = t;
  }
  __syncthreads();
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = r0 + w * NR;
  double s[NR];
  row_products<NR>(inv + (p0 + r) * kld, kld, kld, v, s);
  if (lane < NR) {
    double t = s[0];
#pragma unroll
    for (int q = 1; q < NR; ++q) t = lane == q ? s[q] : t;
    if constexpr (BACK) {
      const int u = pr[r + lane];
      if (u >= 0) x[u] = t;
    } else {
      y[p0 + r + lane] = t;
    }
  }
}

// g = b_s - A_sp y, eight lanes per row
__global__ void __launch_bounds__(256)
    k_dir_sep_rhs(double *__restrict__ g, const double *__restrict__ b,
                  const int32_t *__restrict__ srow, const int32_t *__restrict__ rp,
                  const int32_t *__restrict__ ci, const double *__restrict__ cv,
                  const double *__restrict__ y, int ns) {
  const int i = (blockIdx.x * 256 + threadIdx.x) >> 3, l = threadIdx.x & 7;
  double a = 0.0;
  if (i < ns)
    for (int e = rp[i] + l; e < rp[i + 1]; e += 8) a += cv[e] * y[ci[e]];
  for (int o = 4; o > 0; o >>= 1) a += __shfl_xor(a, o, 8);
  if (i < ns && l == 0) g[i] = b[srow[i]] - a;
}

// x_s = S^-1 g, four rows per wavefront (the last group of rows reads into
// the padding, which is there)
__global__ void __launch_bounds__(256)
    k_dir_sep(const double *__restrict__ sinv, int sld, const double *__restrict__ g,
              const int32_t *__restrict__ srow, double *__restrict__ xs,
              double *__restrict__ x, int ns) {
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = (blockIdx.x * 4 + w) * kRows;
  if (r >= ns) return;
  double s[kRows];
  row_products<kRows>(sinv + (int64_t)r * sld, sld, (ns + 1) & ~1, g, s);
  if (lane < kRows && r + lane < ns) {
    double t = s[0];
#pragma unroll
    for (int q = 1; q < kRows; ++q) t = lane == q ? s[q] : t;
    xs[r + lane] = t;
    x[srow[r + lane]] = t;
  }
}

// r = b - A x, eight lanes per row; x += d (the refinement of a solve)
__global__ void __launch_bounds__(256)
    k_dir_resid(double *__restrict__ r, const double *__restrict__ b, const double *__restrict__ x,
                const int32_t *__restrict__ rp, const int32_t *__restrict__ ci,
                const double *__restrict__ v, int n) {
  const int i = (blockIdx.x * 256 + threadIdx.x) >> 3, l = threadIdx.x & 7;
  double a = 0.0;
  if (i < n)
    for (int e = rp[i] + l; e < rp[i + 1]; e += 8) a += v[e] * x[ci[e]];
  for (int o = 4; o > 0; o >>= 1) a += __shfl_xor(a, o, 8);
  if (i < n && l == 0) r[i] = b[i] - a;
}
__global__ void __launch_bounds__(256)
    k_dir_add(double *__restrict__ x, const double *__restrict__ d, int n) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] += d[i];
}

template <typename T>
bool up(T **dst, const std::vector<T> &src) {
  if (hipMalloc(dst, sizeof(T) * std::max<size_t>(src.size(), 1)) != hipSuccess) return false;
  return src.empty() ||
         hipMemcpy(*dst, src.data(), sizeof(T) * src.size(), hipMemcpyHostToDevice) == hipSuccess;
}

// device scratch of the set-up
struct Scratch {
  std::vector<void *> p;
  template <typename T>
  bool get(T **q, size_t cnt) {
    if (hipMalloc(q, sizeof(T) * std::max<size_t>(cnt, 1)) != hipSuccess) return false;
    p.push_back(*q);
    return true;
  }
  template <typename T>
  bool put(T **q, const std::vector<T> &v) {
    return get(q, v.size()) &&
           (v.empty() ||
            hipMemcpy(*q, v.data(), sizeof(T) * v.size(), hipMemcpyHostToDevice) == hipSuccess);
  }
  ~Scratch() {
    for (void *q : p) (void)hipFree(q);
  }
};

// nb inverses in place; P, R and C hold nb of each panel, dg their diagonals
void invert(double *A, int K, int nb, const double *dg, double *P, double *R, double *C, int *bad,
            hipStream_t s) {
  const int kt = K / kTile;
  for (int kb = 0; kb < kt; ++kb) {
    hipLaunchKernelGGL(k_gj_pivot, dim3(1, 1, nb), dim3(256), 0, s, A, K, kb, dg, P, bad);
    hipLaunchKernelGGL(k_gj_panel, dim3(kt, 2, nb), dim3(256), 0, s, A, K, kb, P, R, C);
    hipLaunchKernelGGL(k_gj_update, dim3(kt, kt, nb), dim3(256), 0, s, A, K, kb, P, R, C);
  }
}

}  // namespace

void DirectCoarse::release() {
  for (void *q : {(void *)inv, (void *)sinv, (void *)prow, (void *)srow, (void *)is_rp,
                  (void *)is_ci, (void *)is_v, (void *)si_rp, (void *)si_ci, (void *)si_v,
                  (void *)y, (void *)g, (void *)xs, (void *)a_rp, (void *)a_ci, (void *)a_v,
                  (void *)rr, (void *)dd})
    if (q) (void)hipFree(q);
  *this = DirectCoarse();
}

int DirectCoarse::setup(const std::vector<int32_t> &rp, const std::vector<int32_t> &ci,
                        const std::vector<double> &v, const std::vector<double> &xyz,
                        hipStream_t s, bool *ok) {
  *ok = false;
  release();
  const int N = (int)rp.size() - 1;
  if (N <= 0 || N > kMaxUnknowns || xyz.size() != 3 * (size_t)N) return NKH_OK;
  // the fastest dissection by the cost model; bisection stops once the
  // separator alone costs more than the best so far
  Dissection best, d;
  d.part.resize(1);
  d.part[0].resize((size_t)N);
  for (int i = 0; i < N; ++i) d.part[0][(size_t)i] = i;
  auto fits = [](const Dissection &q) {
    size_t k = 0;
    for (const auto &p : q.part) k = std::max(k, p.size());
    return k <= (size_t)kMaxPart;
  };
  double t = INFINITY;
  for (int level = 0; level < 10; ++level) {
    if (level > 0) d = bisect(d, rp, ci, xyz);
    const double sb = (double)d.sep.size();
    if (8.0 * sb * sb > kMaxStream || 8.0 * sb * sb / kStreamRate > t) break;
    if (fits(d) && d.seconds() < t) {
      t = d.seconds();
      best = d;
    }
    if (d.part[0].size() < 2 * (size_t)kTile) break;
  }
  if (best.part.empty() || best.bytes() > kMaxStream) return NKH_OK;

  // local numbering: a part's row, or a separator's row
  np = (int)best.part.size();
  ns = (int)best.sep.size();
  int kmax = 0;
  for (const auto &p : best.part) kmax = std::max(kmax, (int)p.size());
  kld = pad_up(kmax);
  sld = pad_up(ns);
  std::vector<int32_t> hprow((size_t)np * kld, -1), at((size_t)N), of((size_t)N, -1);
  for (int p = 0; p < np; ++p)
    for (size_t j = 0; j < best.part[(size_t)p].size(); ++j) {
      const int32_t u = best.part[(size_t)p][j];
      hprow[(size_t)p * kld + j] = u;
      of[(size_t)u] = p;
      at[(size_t)u] = (int32_t)j;
    }
  for (int q = 0; q < ns; ++q) at[(size_t)best.sep[(size_t)q]] = q;
  // blocks and couplings
  std::vector<int64_t> pa, sa;
  std::vector<double> pv, sv;
  std::vector<int32_t> h_is_rp((size_t)np * kld + 1, 0), h_is_ci, h_si_rp((size_t)ns + 1, 0),
      h_si_ci;
  std::vector<double> h_is_v, h_si_v;
  for (int p = 0; p < np; ++p)
    for (int j = 0; j < kld; ++j) {
      const size_t row = (size_t)p * kld + j;
      const int32_t u = hprow[row];
      if (u >= 0)
        for (int32_t e = rp[u]; e < rp[u + 1]; ++e) {
          const int32_t c = ci[e];
          if (of[(size_t)c] < 0) {
            h_is_ci.push_back(at[(size_t)c]);
            h_is_v.push_back(v[e]);
          } else {  // the dissection leaves no coupling between two parts
            NK_CHECK(of[(size_t)c] == p, NKH_ERR_STATE, "coarse dissection: parts touch");
            pa.push_back((int64_t)row * kld + at[(size_t)c]);
            pv.push_back(v[e]);
          }
        }
      h_is_rp[row + 1] = (int32_t)h_is_ci.size();
    }
  // per part its neighbouring separator rows and, per such row, the part's
  // rows it couples to with both entries
  struct Side {
    std::vector<int32_t> bl, cp, cr;
    std::vector<double> cv, rv;
  };
  std::vector<Side> side((size_t)np);
  for (int q = 0; q < ns; ++q) {
    const int32_t u = best.sep[(size_t)q];
    for (int32_t e = rp[u]; e < rp[u + 1]; ++e) {
      const int32_t c = ci[e];
      const int p = of[(size_t)c];
      if (p < 0) {
        sa.push_back((int64_t)q * sld + at[(size_t)c]);
        sv.push_back(v[e]);
        continue;
      }
      h_si_ci.push_back((int32_t)(p * kld + at[(size_t)c]));
      h_si_v.push_back(v[e]);
      Side &S = side[(size_t)p];
      if (S.bl.empty() || S.bl.back() != q) {
        S.bl.push_back(q);
        S.cp.push_back((int32_t)S.cr.size());
      }
      S.cr.push_back(at[(size_t)c]);
      S.rv.push_back(v[e]);
      double back = 0.0;  // A(c, u)
      for (int32_t t2 = rp[c]; t2 < rp[c + 1]; ++t2)
        if (ci[t2] == u) back = v[t2];
      S.cv.push_back(back);
    }
    h_si_rp[(size_t)q + 1] = (int32_t)h_si_ci.size();
  }
  Side all;  // every part's, one after another
  std::vector<size_t> bl0((size_t)np), cp0((size_t)np), cr0((size_t)np);
  size_t nbmax = 0;
  for (int p = 0; p < np; ++p) {
    Side &S = side[(size_t)p];
    S.cp.push_back((int32_t)S.cr.size());
    nbmax = std::max(nbmax, S.bl.size());
    bl0[(size_t)p] = all.bl.size();
    cp0[(size_t)p] = all.cp.size();
    cr0[(size_t)p] = all.cr.size();
    all.bl.insert(all.bl.end(), S.bl.begin(), S.bl.end());
    all.cp.insert(all.cp.end(), S.cp.begin(), S.cp.end());
    all.cr.insert(all.cr.end(), S.cr.begin(), S.cr.end());
    all.cv.insert(all.cv.end(), S.cv.begin(), S.cv.end());
    all.rv.insert(all.rv.end(), S.rv.begin(), S.rv.end());
  }
  const size_t kk = (size_t)kld * kld;
  Scratch sc;
  int64_t *da = nullptr, *ds = nullptr;
  double *dv = nullptr, *dsv = nullptr, *P = nullptr, *R = nullptr, *C = nullptr, *T = nullptr,
         *dg = nullptr;
  int32_t *bl = nullptr, *cp = nullptr, *cr = nullptr;
  double *cv = nullptr, *rv = nullptr;
  int *bad = nullptr;
  const size_t panel = (size_t)std::max((int64_t)np * kld, (int64_t)sld) * kTile;
  int hbad = 0;
  bool good = hipMalloc(&inv, sizeof(double) * kk * np) == hipSuccess &&
              hipMalloc(&sinv, sizeof(double) * std::max<size_t>((size_t)sld * sld, 1)) ==
                  hipSuccess &&
              hipMalloc(&y, sizeof(double) * (size_t)np * kld) == hipSuccess &&
              hipMalloc(&g, sizeof(double) * std::max(sld, 1)) == hipSuccess &&
              hipMalloc(&xs, sizeof(double) * std::max(sld, 1)) == hipSuccess &&
              up(&prow, hprow) && up(&srow, best.sep) && up(&is_rp, h_is_rp) &&
              up(&is_ci, h_is_ci) && up(&is_v, h_is_v) && up(&si_rp, h_si_rp) &&
              up(&si_ci, h_si_ci) && up(&si_v, h_si_v) && sc.put(&da, pa) && sc.put(&dv, pv) &&
              sc.put(&ds, sa) && sc.put(&dsv, sv) && sc.get(&P, (size_t)np * kTile * kTile) &&
              sc.get(&R, panel) && sc.get(&C, panel) && sc.get(&T, (size_t)kld * nbmax) &&
              sc.get(&dg, (size_t)std::max((int64_t)np * kld, (int64_t)sld)) &&
              sc.put(&bl, all.bl) && sc.put(&cp, all.cp) && sc.put(&cr, all.cr) &&
              sc.put(&cv, all.cv) && sc.put(&rv, all.rv) && sc.put(&bad, std::vector<int>(1, 0));
  if (good) {
    auto grid = [](int64_t cnt) {
      return dim3((unsigned)std::max<int64_t>(1, std::min<int64_t>((cnt + 255) / 256, 65536)));
    };
    const dim3 B(256);
    hipLaunchKernelGGL(k_dir_eye, grid((int64_t)kk * np), B, 0, s, inv, kld, (int64_t)kk * np);
    hipLaunchKernelGGL(k_dir_put, grid((int64_t)pa.size()), B, 0, s, inv, da, dv,
                       (int64_t)pa.size());
    hipLaunchKernelGGL(k_dir_diag, grid((int64_t)np * kld), B, 0, s, inv, kld, np, dg);
    invert(inv, kld, np, dg, P, R, C, bad, s);
    if (ns > 0) {
      const int64_t ss = (int64_t)sld * sld;
      hipLaunchKernelGGL(k_dir_eye, grid(ss), B, 0, s, sinv, sld, ss);
      hipLaunchKernelGGL(k_dir_put, grid((int64_t)sa.size()), B, 0, s, sinv, ds, dsv,
                         (int64_t)sa.size());
      // (of the separator's own block: what the parts take from it is the
      // cancellation that a pivot is measured against)
      hipLaunchKernelGGL(k_dir_diag, grid(sld), B, 0, s, sinv, sld, 1, dg);
      // the last row product of an odd separator reads one value past it
      good = hipMemsetAsync(g, 0, sizeof(double) * (size_t)sld, s) == hipSuccess;
      for (int p = 0; p < np; ++p) {
        const int nb = (int)side[(size_t)p].bl.size(), k = (int)best.part[(size_t)p].size();
        if (nb == 0) continue;
        const int32_t *cpp = cp + cp0[(size_t)p], *crp = cr + cr0[(size_t)p];
        const unsigned gx = (unsigned)((nb + 63) / 64);
        hipLaunchKernelGGL(k_dir_schur_t, dim3(gx, (unsigned)((k + 3) / 4)), B, 0, s, T,
                           inv + kk * (size_t)p, kld, k, nb, cpp, crp, cv + cr0[(size_t)p]);
        hipLaunchKernelGGL(k_dir_schur_s, dim3(gx, (unsigned)((nb + 3) / 4)), B, 0, s, sinv,
                           (int64_t)sld, T, nb, bl + bl0[(size_t)p], cpp, crp,
                           rv + cr0[(size_t)p]);
      }
      invert(sinv, sld, 1, dg, P, R, C, bad, s);
    }
    good = good && hipGetLastError() == hipSuccess &&
           hipMemcpyAsync(&hbad, bad, sizeof(int), hipMemcpyDeviceToHost, s) == hipSuccess &&
           hipStreamSynchronize(s) == hipSuccess && hbad == 0;
  }
  if (good) {
    n = N;  // solve() is ready
    good = refine_to(rp, ci, v, xyz, s);
  }
  if (!good) {
    (void)hipStreamSynchronize(s);
    (void)hipGetLastError();
    release();
    return NKH_OK;
  }
  *ok = true;
  return NKH_OK;
}

// Set the refinement steps of a solve by the residuals of two: a rough
// right-hand side (numbers spread over [-1, 1)) and a smooth one (the sum of
// the coordinates), both less their means, as where one unknown of a problem
// with the constants in its null space is held.  False: not accurate enough,
// or out of memory.
bool DirectCoarse::refine_to(const std::vector<int32_t> &rp, const std::vector<int32_t> &ci,
                             const std::vector<double> &v, const std::vector<double> &xyz,
                             hipStream_t s) {
  Scratch sc;
  const size_t N = (size_t)n;
  std::vector<double> b[2], x(N);
  double *db = nullptr, *dx = nullptr;
  if (!sc.get(&db, N) || !sc.get(&dx, N)) return false;
  for (int kind = 0; kind < 2; ++kind) {
    uint32_t u = 1;
    double mean = 0.0;
    b[kind].resize(N);
    for (size_t i = 0; i < N; ++i) {
      u = u * 1664525u + 1013904223u;
      b[kind][i] = kind == 0 ? u * (1.0 / 2147483648.0) - 1.0
                             : xyz[3 * i] + xyz[3 * i + 1] + xyz[3 * i + 2];
      mean += b[kind][i];
    }
    for (double &t : b[kind]) t -= mean / (double)n;
  }
  auto residual = [&]() -> double {  // the larger |b - A x| / |b|
    double worst = 0.0;
    for (const std::vector<double> &bk : b) {
      if (hipMemcpyAsync(db, bk.data(), sizeof(double) * N, hipMemcpyHostToDevice, s) !=
              hipSuccess ||
          solve(dx, db, s) != NKH_OK ||
          hipMemcpyAsync(x.data(), dx, sizeof(double) * N, hipMemcpyDeviceToHost, s) !=
              hipSuccess ||
          hipStreamSynchronize(s) != hipSuccess)
        return INFINITY;
      double rr = 0.0, bb = 0.0;
      for (size_t i = 0; i < N; ++i) {
        double r = bk[i];
        for (int32_t e = rp[i]; e < rp[i + 1]; ++e) r -= v[(size_t)e] * x[(size_t)ci[(size_t)e]];
        rr += r * r;
        bb += bk[i] * bk[i];
      }
      if (bb == 0.0) continue;
      const double rel = std::sqrt(rr / bb);
      if (!(rel <= worst)) worst = std::isfinite(rel) ? rel : INFINITY;
    }
    return worst;
  };
  double res = residual();
  while (res > kGoodResidual && refine < kMaxRefine) {
    if (refine == 0 && !(up(&a_rp, rp) && up(&a_ci, ci) && up(&a_v, v) &&
                         hipMalloc(&rr, sizeof(double) * N) == hipSuccess &&
                         hipMalloc(&dd, sizeof(double) * N) == hipSuccess))
      return false;
    refine += 1;
    const double next = residual();
    if (!(next < 0.5 * res)) {  // nothing left to gain
      refine -= 1;
      break;
    }
    res = next;
  }
  return res <= kMaxResidual;
}

int DirectCoarse::solve(double *x, const double *b, hipStream_t s) const {
  NK_TRY(apply(x, b, s));
  const dim3 B(256);
  for (int k = 0; k < refine; ++k) {
    hipLaunchKernelGGL(k_dir_resid, dim3((unsigned)((n + 31) / 32)), B, 0, s, rr, b, x, a_rp, a_ci,
                       a_v, n);
    NK_TRY(apply(dd, rr, s));
    hipLaunchKernelGGL(k_dir_add, dim3((unsigned)((n + 255) / 256)), B, 0, s, x, dd, n);
    NK_HIP(hipGetLastError());
  }
  return NKH_OK;
}

int DirectCoarse::apply(double *x, const double *b, hipStream_t s) const {
  const dim3 B(256);
  const size_t lds = sizeof(double) * (size_t)kld;
  auto parts = [&](auto back_tag) {
    constexpr bool BACK = decltype(back_tag)::value;
    const bool few = (int64_t)np * kld <= kFewRows;
    const int rows = few ? 4 : 4 * kRows;
    hipLaunchKernelGGL((few ? k_dir_parts<BACK, 1> : k_dir_parts<BACK, kRows>),
                       dim3((unsigned)(kld / rows), (unsigned)np), B, lds, s, inv, kld, prow, b, y,
                       is_rp, is_ci, is_v, xs, x);
  };
  if (ns == 0) {  // separate parts: their inverses are the solve
    parts(std::true_type());
  } else {
    parts(std::false_type());
    hipLaunchKernelGGL(k_dir_sep_rhs, dim3((unsigned)((ns + 31) / 32)), B, 0, s, g, b, srow,
                       si_rp, si_ci, si_v, y, ns);
    hipLaunchKernelGGL(k_dir_sep, dim3((unsigned)((ns + 4 * kRows - 1) / (4 * kRows))), B, 0, s,
                       sinv, sld, g, srow, xs, x, ns);
    parts(std::true_type());
  }
  NK_HIP(hipGetLastError());
  return NKH_OK;
}

}  // namespace nekamd
