// Scalar work of the Krylov loops done by the kernels around it instead of by
// one-block kernels of their own, each of which cost 3 to 5 us and a gap of 4
// to 9 us between launches (MI355X).  Without them: Jacobi PCG on 336
// elements, lx1 8, 420 -> 347 us a solve, on 1.68e7 nodes 7250 -> 7180; batch
// of five 1810 -> 1660; GMRES lx1 6 2440 -> 2300; flexible CG in FP32 3640 -> 3490.
#pragma once
#include "nekamd_internal.h"

namespace nekamd {

// Blocks of a kernel that ends in last_block, two nodes per thread: 64 to
// 2048.
inline int dot_blocks(int64_t n) {
  const int64_t b = (n + 511) / 512;
  return (int)(b < 64 ? 64 : (b > 2048 ? 2048 : b));
}

// Results that a block leaves for the last block of its grid, wherever that
// runs: agent-scope stores and loads, which do not stay in an XCD's own L2.
// (A fence per block in their place writes that L2 back each time: the
// update-and-dots kernel on 1.68e7 nodes took 180 us without, 600 with it.)
__device__ __forceinline__ void leave(double *p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double left(const double *p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Counters of last_block: kSub of them and one over these, each in a cache
// line of its own.  Blocks that end together add to one counter at about 20
// ns each (507 blocks of an orthogonalisation: 9 us without the count, 20
// with one counter for all).
constexpr int kSub = 32, kLine = 32;                   // counters; ints a line
constexpr int kCounterDoubles = (kSub + 1) * kLine / 2;
// by the first 64 threads of one block, before the grids that count
__device__ __forceinline__ void clear_counters(int *cnt) {
  if (threadIdx.x <= kSub) cnt[kLine * threadIdx.x] = 0;
}

// True in the last of the grid's nb blocks to get here: every block's
// results, stored by leave() in its first wavefront, can then be read by
// left().  The wavefront counts its block only after its stores have reached
// the memory that the agent shares.  The counters start at 0 and are 0 again
// after the grid.  All threads must call it.
__device__ __forceinline__ bool last_block(int *cnt, int nb) {
  __shared__ int last;
  if (threadIdx.x < 64) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    if (threadIdx.x == 0) {
      const int b = blockIdx.x, g = b % kSub;
      int *c = cnt + kLine * g;
      last = 0;
      if (__hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
          (nb - g + kSub - 1) / kSub - 1) {  // the last of group g
        __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        c = cnt + kLine * kSub;
        if (__hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
            (nb < kSub ? nb : kSub) - 1) {
          __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          last = 1;
        }
      }
    }
  }
  __syncthreads();
  return last != 0;
}

// Sums of the N arrays (stride apart) of count results left by blocks, by one
// block (blockDim.x a multiple of 64, at most 1024) in a fixed order: four
// interleaved accumulators per thread, so that several loads are in flight,
// then the waves in order.  Valid on every thread.
template <int N>
__device__ __forceinline__ void sum_left(const double *p, int64_t stride, int count,
                                         double (&out)[N]) {
  __shared__ double sw[N][16];
  const int t = threadIdx.x, nt = blockDim.x;
  double v[N][4] = {};
  int q = t;
  for (; q + 3 * nt < count; q += 4 * nt) {
    double l[N][4];
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int u = 0; u < 4; ++u) l[k][u] = left(p + k * stride + q + u * nt);
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[k][u] += l[k][u];
  }
  for (; q < count; q += nt) {
#pragma unroll
    for (int k = 0; k < N; ++k) v[k][0] += left(p + k * stride + q);
  }
#pragma unroll
  for (int k = 0; k < N; ++k) {
    double a = (v[k][0] + v[k][1]) + (v[k][2] + v[k][3]);
    for (int o = 32; o > 0; o >>= 1) a += __shfl_down(a, o, 64);
    if ((t & 63) == 0) sw[k][t >> 6] = a;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < N; ++k) {
    double a = 0.0;
    for (int w = 0; w < (nt >> 6); ++w) a += sw[k][w];
    out[k] = a;
  }
  __syncthreads();
}

// The step length that an assembly leaves behind: *den = the sum of the count
// partials that the operator before it wrote, *alpha = *num / *den.
struct StepLength {
  const double *part;
  int count;
  const double *num;
  double *den, *alpha;
  // hist (may be null): rho, alpha and *beta of iteration *iter
  double *hist;
  const double *beta;
  const int *iter;
};
__device__ inline void step_length(const StepLength &a) {
  const double rho = block_sum_partials(a.part, a.count);
  if (threadIdx.x != 0) return;
  const double al = *a.num / rho;
  *a.den = rho;
  *a.alpha = al;
  if (a.hist) {
    double *h = a.hist + 5 * (*a.iter - 1);
    h[2] = rho;
    h[3] = al;
    h[4] = *a.beta;
  }
}

// gs_assemble, then a's step length; once st is done, neither.
int gs_assemble_step(const GsMap &gs, double *w, const CgState *st, hipStream_t s,
                     const uint8_t *flag, const StepLength &a);
int gs_assemble_step(const GsMap &gs, float *w, const CgState *st, hipStream_t s,
                     const uint8_t *flag, const StepLength &a);

}  // namespace nekamd
