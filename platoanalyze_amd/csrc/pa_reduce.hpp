// Fence-free grid reductions and XCD-aware persistent grids.
//
// A reduction kernel writes one partial per work-group; the kernel that needs the
// total (the next one in the stream) sums the partials in a fixed order in every
// work-group.  Kernel boundaries make the partials visible, so no work-group ever
// issues a device-scope fence (on a multi-XCD part such a fence writes back the
// issuing XCD's L2) and the result is deterministic run to run.
#pragma once
#include <hip/hip_runtime.h>

#include "pa_dpp.hpp"
#include "pa_kernels.hpp"

namespace pa {

// Work-groups of the persistent vector / reduction kernels (also the partial count);
// a multiple of the XCD count.
constexpr int kRedBlocks = 1024;

// Grid of a persistent kernel over `work` items handled `per_block` at a time.
inline int red_grid(size_t work, int per_block) {
  size_t g = (work + per_block - 1) / per_block;
  g = (g + kNumXcd - 1) / kNumXcd * kNumXcd;
  if (g < (size_t)kNumXcd) g = kNumXcd;
  if (g > (size_t)kRedBlocks) g = kRedBlocks;
  return (int)g;
}

// Sum over a wavefront, the same bits in every lane: DPP sums of the four 16-lane rows,
// then the rows' values through scalar registers (no LDS crossbar: six shuffles of a double
// were most of a small kernel's reduction time).
__device__ __forceinline__ double wave_sum(double v) {
  v = sum16(v);
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  double r[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, 16 * q);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), 16 * q);
    r[q] = __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
  }
  return (r[0] + r[1]) + (r[2] + r[3]);
}

// Sum of one value per thread over the work-group, returned in every thread
// (fixed order).  `sh` holds NT/64 doubles; safe to call repeatedly.  Every lane of the
// work-group takes part.
template <int NT>
__device__ __forceinline__ double block_reduce_all(double v, double* sh) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int q = 0; q < NT / 64; ++q) t += sh[q];
  return t;
}

// Two sums at once (one pair of barriers); `sh` holds 2 NT/64 doubles.
template <int NT>
__device__ __forceinline__ void block_reduce_two(double& a, double& b, double* sh) {
  a = wave_sum(a);
  b = wave_sum(b);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    sh[threadIdx.x >> 6] = a;
    sh[NT / 64 + (threadIdx.x >> 6)] = b;
  }
  __syncthreads();
  a = b = 0.0;
#pragma unroll
  for (int q = 0; q < NT / 64; ++q) {
    a += sh[q];
    b += sh[NT / 64 + q];
  }
}

// Fixed-order total of n partials written by an earlier kernel, in every thread.
template <int NT>
__device__ __forceinline__ double sum_partials_all(const double* p, int n, double* sh) {
  double v = 0.0;
  for (int i = threadIdx.x; i < n; i += NT) v += p[i];
  return block_reduce_all<NT>(v, sh);
}

// Totals of two partial arrays at once; `sh` holds 2 NT/64 doubles.
template <int NT>
__device__ __forceinline__ void sum_partials_two(const double* p, int np, const double* q, int nq, double* sh,
                                                 double& a, double& b) {
  a = b = 0.0;
  for (int i = threadIdx.x; i < np; i += NT) a += p[i];
  for (int i = threadIdx.x; i < nq; i += NT) b += q[i];
  block_reduce_two<NT>(a, b, sh);
}

// Same, with four independent accumulators per thread (for long partial arrays read by
// a single work-group: more loads in flight).  Fixed order, deterministic.
template <int NT>
__device__ __forceinline__ double sum_partials_wide(const double* p, int n, double* sh) {
  double a0 = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
  int i = threadIdx.x;
  for (; i + 3 * NT < n; i += 4 * NT) {
    a0 += p[i];
    a1 += p[i + NT];
    a2 += p[i + 2 * NT];
    a3 += p[i + 3 * NT];
  }
  for (; i < n; i += NT) a0 += p[i];
  return block_reduce_all<NT>((a0 + a1) + (a2 + a3), sh);
}

// Contiguous share [lo, hi) of n items for the XCD that runs this work-group
// (work-group b runs on XCD b % 8), and this group's rank j among the bx groups
// of that XCD.  Items close in index (Hilbert-ordered rows, chunks) stay in one L2.
struct XcdSpan {
  int lo, hi, j, bx;
};
__device__ __forceinline__ XcdSpan xcd_span(int n) {
  XcdSpan s;
  const int x = blockIdx.x % kNumXcd;
  s.j = blockIdx.x / kNumXcd;
  s.bx = gridDim.x / kNumXcd;
  const int per = (n + kNumXcd - 1) / kNumXcd;
  s.lo = min(n, x * per);
  s.hi = min(n, s.lo + per);
  return s;
}

}  // namespace pa
