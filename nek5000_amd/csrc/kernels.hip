// Geometric factors and Jacobi diagonal kernels.
#include "element_kernels.h"

namespace nekamd {

// ---------------------------------------------------------------------------
// Geometric factors: coef.f:879-927 XYZRST (x_r = D x, x_s = x D^T per layer,
// x_t = x D^T over layers), coef.f:555-632 GLMAPM1 (Jacobian, cofactors via
// ascol5) and coef.f:633-785 GEODAT1 (G_ij = cof_i.cof_j / J * w3, bm1 = J*w3).
// ---------------------------------------------------------------------------
template <int NP>
__global__ void __launch_bounds__(NP * NP * epb<NP>())
    k_geom(DMat<NP> Dm, const double *__restrict__ Dg, const double *__restrict__ wg,
           const double *__restrict__ x, const double *__restrict__ y,
           const double *__restrict__ z, double *__restrict__ g, int64_t gstride,
           double *__restrict__ bm1, int64_t nel) {
  constexpr int NP2 = NP * NP, NP3 = NP2 * NP, EPB = epb<NP>();
  __shared__ double s_D[NP][NP + 1];
  __shared__ double s_x[EPB][3][NP3];
  const int tid = threadIdx.x;
  const int le = tid / NP2;
  const int ij = tid - le * NP2;
  const int i = ij % NP, j = ij / NP;
  for (int t = tid; t < NP2; t += blockDim.x) s_D[t % NP][t / NP] = Dg[t];
  for (int64_t eb = blockIdx.x; eb * EPB < nel; eb += gridDim.x) {
    const int64_t e = eb * EPB + le;
    const bool valid = (le < EPB) && (e < nel);
    const int64_t base = e * NP3 + ij;
    double cx[NP], cy[NP], cz[NP];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      double a = 0.0, b = 0.0, c = 0.0;
      if (valid) {
        a = x[base + k * NP2];
        b = y[base + k * NP2];
        c = z[base + k * NP2];
      }
      cx[k] = a;
      cy[k] = b;
      cz[k] = c;
      s_x[le][0][k * NP2 + ij] = a;
      s_x[le][1][k * NP2 + ij] = b;
      s_x[le][2][k * NP2 + ij] = c;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      double xr = 0, yr = 0, zr = 0, xs = 0, ys = 0, zs = 0, xt = 0, yt = 0, zt = 0;
#pragma unroll
      for (int m = 0; m < NP; ++m) {
        const double dr = s_D[i][m], ds = s_D[j][m], dt = Dm.d[k + NP * m];
        xr += dr * s_x[le][0][k * NP2 + j * NP + m];
        yr += dr * s_x[le][1][k * NP2 + j * NP + m];
        zr += dr * s_x[le][2][k * NP2 + j * NP + m];
        xs += ds * s_x[le][0][k * NP2 + m * NP + i];
        ys += ds * s_x[le][1][k * NP2 + m * NP + i];
        zs += ds * s_x[le][2][k * NP2 + m * NP + i];
        xt += dt * cx[m];
        yt += dt * cy[m];
        zt += dt * cz[m];
      }
      if (!valid) continue;
      double jac = 0.0;
      jac = jac + xr * ys * zt;
      jac = jac + xt * yr * zs;
      jac = jac + xs * yt * zr;
      jac = jac - xr * yt * zs;
      jac = jac - xs * yr * zt;
      jac = jac - xt * ys * zr;
      const double rx = ys * zt - yt * zs, ry = xt * zs - xs * zt, rz = xs * yt - xt * ys;
      const double sx = yt * zr - yr * zt, sy = xr * zt - xt * zr, sz = xt * yr - xr * yt;
      const double tx = yr * zs - ys * zr, ty = xs * zr - xr * zs, tz = xr * ys - xs * yr;
      const double wj = 1.0 / jac;
      const double w3 = wg[i] * wg[j] * wg[k];
      const int64_t l = base + k * NP2;
      g[l] = (rx * rx + ry * ry + rz * rz) * wj * w3;
      g[gstride + l] = (sx * sx + sy * sy + sz * sz) * wj * w3;
      g[2 * gstride + l] = (tx * tx + ty * ty + tz * tz) * wj * w3;
      g[3 * gstride + l] = (rx * sx + ry * sy + rz * sz) * wj * w3;
      g[4 * gstride + l] = (rx * tx + ry * ty + rz * tz) * wj * w3;
      g[5 * gstride + l] = (sx * tx + sy * ty + sz * tz) * wj * w3;
      bm1[l] = jac * w3;
    }
  }
}

template <int NP>
static int geom_dispatch(Mesh &m, const double *x, const double *y, const double *z,
                         hipStream_t s) {
  DMat<NP> Dm;
  for (int t = 0; t < NP * NP; ++t) Dm.d[t] = m.D[t];
  constexpr int EPB = epb<NP>();
  int64_t ngroups = (m.nel + EPB - 1) / EPB;
  int grid = (int)(ngroups < ((int64_t)1 << 20) ? ngroups : ((int64_t)1 << 20));
  if (grid < 1) grid = 1;
  // weights: stash after D in the device basis buffer
  hipLaunchKernelGGL((k_geom<NP>), dim3(grid), dim3(NP * NP * EPB), 0, s, Dm, m.Dd,
                     m.Dd + kMaxNP * kMaxNP, x, y, z, m.g, m.n, m.bm1, m.nel);
  NK_HIP(hipGetLastError());
  return NKH_OK;
}

int launch_geom(Mesh &m, const double *x, const double *y, const double *z, hipStream_t s) {
#define CALL(NP) geom_dispatch<NP>(m, x, y, z, s)
  NK_NP_SWITCH(m.np, CALL)
#undef CALL
}

// ---------------------------------------------------------------------------
// Jacobi diagonal, hmholtz.f:380-524 SETPREC (3-D, every element deformed):
//   d(ix,iy,iz) = sum_q g1(q,iy,iz) D(q,ix)^2 + g2(ix,q,iz) D(q,iy)^2
//               + g3(ix,iy,q) D(q,iz)^2
// plus the g4/g5/g6 cross terms the reference adds at the 8 element corners
// (loops 600/700/800 step by lx1-1), then d = d*h1 + h2*bm1.  The dssum and
// inversion that follow are done by the caller.
// The slab of the other element kernels: every thread's column of g1, g2 and
// g3 is loaded at once; g1 and g2 go through LDS one t-plane at a time (two
// buffers, one barrier per plane), g3 stays in registers.  Reads each factor
// once, 5 words per node: 362 -> 149 us (4.5 TB/s) on 32,768 elements at
// lx1 = 8, where one thread per node read its 3 NP factors from the caches.
// The sums run over g1, g2, g3 in that order, as in the reference.
// ---------------------------------------------------------------------------
template <int NP>
__global__ void __launch_bounds__(NP * NP * epb<NP>())
    k_setprec(DMat<NP> Dq, const double *__restrict__ Dg, const double *__restrict__ g,
              int64_t gstride, const double *__restrict__ h1f, double h1s,
              const double *__restrict__ h2f, double h2s, const double *__restrict__ bm1,
              double *__restrict__ d, int64_t nel) {
  constexpr int NP2 = NP * NP, NP3 = NP2 * NP, L = NP - 1, EPB = epb<NP>();
  __shared__ double s_q[NP][NP + 1];  // D(q, i)^2 at [i][q]
  __shared__ double s_g1[2][EPB][NP2];
  __shared__ double s_g2[2][EPB][NP2];
  const int tid = threadIdx.x;
  const int le = tid / NP2;
  const int ij = tid - le * NP2;
  const int ix = ij % NP, iy = ij / NP;
  for (int t = tid; t < NP2; t += blockDim.x) s_q[t / NP][t % NP] = Dg[t] * Dg[t];
  for (int64_t eb = blockIdx.x; eb * EPB < nel; eb += gridDim.x) {
    // a slab past the last element works on the block's first one, unstored
    const bool valid = EPB == 1 || eb * EPB + le < nel;
    const int64_t base = (eb * EPB + (valid ? le : 0)) * NP3 + ij;
    double r1[NP], r2[NP], r3[NP], rm[NP];
    if constexpr (NP & 1) __syncthreads();  // buffer 0 ends and starts an element
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int64_t l = base + k * NP2;
      r1[k] = ldnt(g + l);
      r2[k] = ldnt(g + gstride + l);
      r3[k] = ldnt(g + 2 * gstride + l);
      rm[k] = ldnt(bm1 + l);
    }
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int b = k & 1;
      // one plane at a time: the planes' LDS reads interleaved would fill the
      // registers (one wavefront per SIMD)
      __builtin_amdgcn_sched_barrier(0);
      s_g1[b][le][ij] = r1[k];
      s_g2[b][le][ij] = r2[k];
      __syncthreads();
      double v = 0.0;
#pragma unroll
      for (int q = 0; q < NP; ++q) v += s_g1[b][le][q + NP * iy] * s_q[ix][q];
#pragma unroll
      for (int q = 0; q < NP; ++q) v += s_g2[b][le][ix + NP * q] * s_q[iy][q];
#pragma unroll
      for (int q = 0; q < NP; ++q) v += r3[q] * Dq.d[q + NP * k];
      if (!valid) continue;
      const int64_t l = base + k * NP2;
      if ((k == 0 || k == L) && (ix == 0 || ix == L) && (iy == 0 || iy == L)) {
        // loop 600 (x-ends), 700 (y-ends), 800 (z-ends), in that order;
        // DXTM1(a,a) = D(a,a)
        const double g4 = g[3 * gstride + l], g5 = g[4 * gstride + l], g6 = g[5 * gstride + l];
        const double dx = Dg[ix == 0 ? 0 : NP2 - 1], dy = Dg[iy == 0 ? 0 : NP2 - 1],
                     dz = Dg[k == 0 ? 0 : NP2 - 1];
        v = v + g4 * dx * dy + g5 * dx * dz;
        v = v + g4 * dy * dx + g6 * dy * dz;
        v = v + g5 * dz * dx + g6 * dz * dy;
      }
      v = v * (h1f ? h1f[l] : h1s);
      v = v + (h2f ? h2f[l] : h2s) * rm[k];
      d[l] = v;
    }
  }
}

template <int NP>
static int setprec_dispatch(const Mesh &m, double *d, Coef h1, Coef h2, hipStream_t s) {
  DMat<NP> Dq;  // the squares, as the host forms them
  for (int t = 0; t < NP * NP; ++t) Dq.d[t] = m.D[t] * m.D[t];
  constexpr int EPB = epb<NP>();
  const int64_t ngroups = (m.nel + EPB - 1) / EPB;
  const int grid = (int)(ngroups < ((int64_t)1 << 20) ? ngroups : ((int64_t)1 << 20));
  hipLaunchKernelGGL((k_setprec<NP>), dim3(grid), dim3(NP * NP * EPB), 0, s, Dq, m.Dd, m.g, m.n,
                     h1.f, h1.s, h2.f, h2.s, m.bm1, d, m.nel);
  NK_HIP(hipGetLastError());
  return NKH_OK;
}

int launch_setprec(const Mesh &m, double *d, Coef h1, Coef h2, hipStream_t s) {
#define CALL(NP) setprec_dispatch<NP>(m, d, h1, h2, s)
  NK_NP_SWITCH(m.np, CALL)
#undef CALL
}

// Undeformed elements (genxyz.f:351-470 setdef; param(59) = 0): the
// reference's axhelm and setprec skip their cross terms g4..g6
// (hmholtz.f:188-218 fast path, `if (ifdfrm(e))`; :440-468), so they are
// held as zeros here, whatever sfastax (hmholtz.f:353-364) left in Nek's
// g4m1..g6m1.
__global__ void k_zero_cross(double *__restrict__ g, const uint8_t *__restrict__ undeformed,
                             int64_t npe, int64_t nel, int64_t n) {
  const int64_t total = 3 * n;
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < total;
       q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t l = q % n;
    if (undeformed[l / npe]) g[3 * n + q] = 0.0;
  }
}

int apply_undeformed(Mesh &m, hipStream_t s) {
  if (!m.undeformed || !m.g) return NKH_OK;
  const int64_t npe = (int64_t)m.np * m.np * m.np;
  int64_t grid = (3 * m.n + 255) / 256;
  if (grid > 65536) grid = 65536;
  hipLaunchKernelGGL(k_zero_cross, dim3((int)grid), dim3(256), 0, s, m.g, m.undeformed, npe,
                     m.nel, m.n);
  NK_HIP(hipGetLastError());
  return NKH_OK;
}

}  // namespace nekamd
