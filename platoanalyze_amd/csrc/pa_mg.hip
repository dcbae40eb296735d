// Geometric multigrid kernels (see pa_mg.hpp).  Box node grids: node (i, j, k) of a
// level has grid index (i * ny + j) * nz + k; coarse node (I, J, K) sits on fine node
// (2I, 2J, 2K).  Trilinear prolongation: a fine coordinate 2I contributes weight 1 to
// coarse I, 2I +- 1 weight 1/2 to each neighbour; restriction is its transpose.
#include "pa_mg.hpp"
#include "pa_kernels.hpp"

#include <algorithm>

#include "pa_dpp.hpp"
#include "pa_reduce.hpp"
#include "pa_solver.hpp"
#include "pa_spmv.hpp"

namespace pa {

namespace {

constexpr int kT = 256;

int blocks_of(size_t n, int cap = 4096) {
  size_t g = (n + kT - 1) / kT;
  return (int)(g < 1 ? 1 : (g > (size_t)cap ? cap : g));
}

__device__ __forceinline__ void dinv3(const double* __restrict__ D, const double r[3], double z[3]) {
  z[0] = D[0] * r[0] + D[1] * r[1] + D[2] * r[2];
  z[1] = D[3] * r[0] + D[4] * r[1] + D[5] * r[2];
  z[2] = D[6] * r[0] + D[7] * r[1] + D[8] * r[2];
}

__device__ __forceinline__ void put_lattice(const MgLattice& L, int n, const double v[3]) {
  const int g = L.gpack[n];
  const uint32_t bm = L.bcmask[n];
  L.plat[((g & 1023) + 1) + (size_t)L.px * ((((g >> 10) & 1023) + 1) + (size_t)L.py * ((g >> 20) + 1))] = make_float4(
      (bm & 1u) ? 0.0f : (float)v[0], (bm & 2u) ? 0.0f : (float)v[1], (bm & 4u) ? 0.0f : (float)v[2], 0.0f);
}

// 8 lanes per coarse node, lane q the fine points q, q + 8, .. of its 27: two dependent
// gathers, so lanes in flight bound it.  One thread per node took 23.4 us for 128x64x64 ->
// 64x32x32 and 11.5, 10.1 and 7.7 us for the next three; now 12.0, 4.9, 4.6 and 4.4 us.
__global__ __launch_bounds__(kT) void k_mg_restrict(const double* __restrict__ rf, double* __restrict__ rc,
                                                    const int32_t* __restrict__ cgrid,
                                                    const int32_t* __restrict__ fnode, BoxDims fd,
                                                    const uint8_t* __restrict__ cbc, int ncn,
                                                    const double* __restrict__ cdinv, double inv_theta,
                                                    double* __restrict__ cx, double* __restrict__ cd) {
  const int q = threadIdx.x % 8;
  for (int c = (blockIdx.x * kT + threadIdx.x) / 8; c < ncn; c += gridDim.x * (kT / 8)) {
    const int I = cgrid[3 * c], J = cgrid[3 * c + 1], K = cgrid[3 * c + 2];
    const size_t o = 3 * (size_t)c;
    double D[3] = {0.0, 0.0, 0.0};  // lane i < 3: row i of the node's block
    if (cx && q < 3) {
#pragma unroll
      for (int i = 0; i < 3; ++i) D[i] = cdinv[3 * o + 3 * q + i];
    }
    const uint32_t bm = cbc[c];
    // branch-free: a point outside the fine grid (or past the 27) reads the coarse node's own
    // fine point with weight 0 (adds an exact zero), so all lookups issue at once
    double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      const int pt = q + 8 * m;
      const int a = pt / 9 - 1, b = pt / 3 % 3 - 1, e = pt % 3 - 1;
      const int i = 2 * I + a, j = 2 * J + b, k = 2 * K + e;
      const bool in = pt < 27 && (unsigned)i < (unsigned)fd.nx && (unsigned)j < (unsigned)fd.ny && (unsigned)k < (unsigned)fd.nz;
      const double w = in ? (a ? 0.5 : 1.0) * (b ? 0.5 : 1.0) * (e ? 0.5 : 1.0) : 0.0;
      const size_t f = 3 * (size_t)fnode[((size_t)(in ? i : 2 * I) * fd.ny + (in ? j : 2 * J)) * fd.nz + (in ? k : 2 * K)];
#pragma unroll
      for (int l = 0; l < 3; ++l) s[l] += w * rf[f + l];
    }
#pragma unroll
    for (int l = 0; l < 3; ++l) {  // every lane of the eight receives the sums
      s[l] += dpp_f64<kDppXor1>(s[l]);
      s[l] += dpp_f64<kDppXor2>(s[l]);
      s[l] += dpp_f64<kDppHalfMirror>(s[l]);
      if ((bm >> l) & 1u) s[l] = 0.0;
    }
    if (q < 3) {
      rc[o + q] = q == 0 ? s[0] : q == 1 ? s[1] : s[2];
      if (cx) {
        const double z = inv_theta * (D[0] * s[0] + D[1] * s[1] + D[2] * s[2]);
        cx[o + q] = z;
        cd[o + q] = z;
      }
    }
  }
}

__global__ __launch_bounds__(kT) void k_mg_prolong_add(const double* __restrict__ ec, double* __restrict__ xf,
                                                       const int32_t* __restrict__ fgrid,
                                                       const int32_t* __restrict__ cnode, BoxDims cd,
                                                       const uint8_t* __restrict__ fbc, int nfn, MgLattice lat) {
  for (int n = blockIdx.x * kT + threadIdx.x; n < nfn; n += gridDim.x * kT) {
    const int i = fgrid[3 * n], j = fgrid[3 * n + 1], k = fgrid[3 * n + 2];
    const int I0 = i >> 1, J0 = j >> 1, K0 = k >> 1;
    const int nI = (i & 1) ? 2 : 1, nJ = (j & 1) ? 2 : 1, nK = (k & 1) ? 2 : 1;
    const double wI = (i & 1) ? 0.5 : 1.0, wJ = (j & 1) ? 0.5 : 1.0, wK = (k & 1) ? 0.5 : 1.0;
    // branch-free over the 8 candidates: an absent one reads coarse point (I0, J0, K0) with
    // weight 0 (adds an exact zero)
    double s0 = 0.0, s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const bool in = a < nI && b < nJ && e < nK;
          const size_t c = 3 * (size_t)cnode[((size_t)(I0 + (in ? a : 0)) * cd.ny + (J0 + (in ? b : 0))) * cd.nz +
                                             (K0 + (in ? e : 0))];
          const double w = in ? wI * wJ * wK : 0.0;
          s0 += w * ec[c];
          s1 += w * ec[c + 1];
          s2 += w * ec[c + 2];
        }
    const uint32_t bm = fbc[n];
    const size_t d = 3 * (size_t)n;
    const double v[3] = {xf[d] + ((bm & 1u) ? 0.0 : s0), xf[d + 1] + ((bm & 2u) ? 0.0 : s1),
                         xf[d + 2] + ((bm & 4u) ? 0.0 : s2)};
#pragma unroll
    for (int l = 0; l < 3; ++l) xf[d + l] = v[l];
    if (lat.plat) put_lattice(lat, n, v);
  }
}

__global__ __launch_bounds__(kT) void k_mg_wrestrict(const double* __restrict__ wf, double* __restrict__ wc,
                                                     const int32_t* __restrict__ cgrid,
                                                     const int32_t* __restrict__ fnode, BoxDims fd, int ncn) {
  for (int c = blockIdx.x * kT + threadIdx.x; c < ncn; c += gridDim.x * kT) {
    const int I = cgrid[3 * c], J = cgrid[3 * c + 1], K = cgrid[3 * c + 2];
    double s = 0.0, ws = 0.0;
    for (int a = -1; a <= 1; ++a) {
      const int i = 2 * I + a;
      if (i < 0 || i >= fd.nx) continue;
      for (int b = -1; b <= 1; ++b) {
        const int j = 2 * J + b;
        if (j < 0 || j >= fd.ny) continue;
        for (int e = -1; e <= 1; ++e) {
          const int k = 2 * K + e;
          if (k < 0 || k >= fd.nz) continue;
          const double w = (a ? 0.5 : 1.0) * (b ? 0.5 : 1.0) * (e ? 0.5 : 1.0);
          s += w * wf[fnode[((size_t)i * fd.ny + j) * fd.nz + k]];
          ws += w;
        }
      }
    }
    wc[c] = s / ws;
  }
}

__global__ __launch_bounds__(kT) void k_simp_w(const double* z, double* w, int n, Material m) {
  for (int i = blockIdx.x * kT + threadIdx.x; i < n; i += gridDim.x * kT) w[i] = penalty_w(m, z[i]);
}

__global__ __launch_bounds__(kT) void k_cheb_first(double* __restrict__ x, double* __restrict__ d,
                                                   const double* __restrict__ r, const double* __restrict__ dinv,
                                                   double inv_theta, int nn, const double* __restrict__ t,
                                                   MgLattice lat) {
  for (int n = blockIdx.x * kT + threadIdx.x; n < nn; n += gridDim.x * kT) {
    const size_t o = 3 * (size_t)n;
    double rv[3] = {r[o], r[o + 1], r[o + 2]};
    if (t) {
#pragma unroll
      for (int i = 0; i < 3; ++i) rv[i] -= t[o + i];
    }
    double zv[3];
    dinv3(dinv + 9 * (size_t)n, rv, zv);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      zv[i] *= inv_theta;
      if (d) d[o + i] = zv[i];
      x[o + i] = zv[i];
    }
    if (lat.plat) put_lattice(lat, n, zv);
  }
}

__global__ __launch_bounds__(kT) void k_cheb_next(double* __restrict__ x, double* __restrict__ d,
                                                  const double* __restrict__ r, const double* __restrict__ Kx,
                                                  const double* __restrict__ dinv, double c1, double c2, int nn) {
  for (int n = blockIdx.x * kT + threadIdx.x; n < nn; n += gridDim.x * kT) {
    const size_t o = 3 * (size_t)n;
    const double rv[3] = {r[o] - Kx[o], r[o + 1] - Kx[o + 1], r[o + 2] - Kx[o + 2]};
    double zv[3];
    dinv3(dinv + 9 * (size_t)n, rv, zv);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double v = c1 * d[o + i] + c2 * zv[i];
      d[o + i] = v;
      x[o + i] += v;
    }
  }
}

__global__ __launch_bounds__(kT) void k_sub(double* out, const double* a, const double* b, size_t n) {
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) out[i] = a[i] - b[i];
}

__global__ __launch_bounds__(kT) void k_add(double* y, const double* x, size_t n) {
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) y[i] += x[i];
}

__global__ __launch_bounds__(kT) void k_add2(double* out, const double* a, const double* b, size_t n) {
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) out[i] = a[i] + b[i];
}

// one wavefront per row, fixed-order lane sums
__global__ __launch_bounds__(kT) void k_dense_gemv(const double* __restrict__ A, const double* __restrict__ x,
                                                   double* __restrict__ y, int n) {
  const int lane = threadIdx.x & 63;
  for (int row = (blockIdx.x * kT + threadIdx.x) / 64; row < n; row += gridDim.x * (kT / 64)) {
    double s = 0.0;
    for (int c = lane; c < n; c += 64) s += A[(size_t)row * n + c] * x[c];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
    if (lane == 0) y[row] = s;
  }
}

// x += alpha p, r -= alpha q, partials of r.r; with z also the V-cycle's start
// z = inv_theta D^-1 r and its lattice copy, while r is at hand
__global__ __launch_bounds__(kT) void k_mg_update(double* __restrict__ x, double* __restrict__ r,
                                                  const double* __restrict__ p, const double* __restrict__ q,
                                                  const double* __restrict__ scal, int nn, double* __restrict__ P_rr,
                                                  double* __restrict__ z, const double* __restrict__ dinv,
                                                  double inv_theta, MgLattice lat) {
  __shared__ double sh[kT / 64];
  const double alpha = scal[kAlpha];
  double rr = 0.0;
  const XcdSpan sp = xcd_span(nn);
  for (int n = sp.lo + sp.j * kT + threadIdx.x; n < sp.hi; n += sp.bx * kT) {
    const size_t d = 3 * (size_t)n;
    double rv[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      x[d + i] += alpha * p[d + i];
      rv[i] = r[d + i] - alpha * q[d + i];
      r[d + i] = rv[i];
      rr += rv[i] * rv[i];
    }
    if (z) {
      double zv[3];
      dinv3(dinv + 3 * d, rv, zv);
#pragma unroll
      for (int i = 0; i < 3; ++i) z[d + i] = zv[i] *= inv_theta;
      put_lattice(lat, n, zv);
    }
  }
  const double t = block_reduce_all<kT>(rr, sh);
  if (threadIdx.x == 0) P_rr[blockIdx.x] = t;
}

__global__ __launch_bounds__(kT) void k_mg_pupdate(double* __restrict__ p, const double* __restrict__ z,
                                                   const double* __restrict__ scal, int nn, int first, MgLattice lat) {
  const double beta = first ? 0.0 : scal[kBeta];
  for (int n = blockIdx.x * kT + threadIdx.x; n < nn; n += gridDim.x * kT) {
    const size_t d = 3 * (size_t)n;
    double v[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) p[d + i] = v[i] = first ? z[d + i] : fma(beta, p[d + i], z[d + i]);
    if (lat.plat) put_lattice(lat, n, v);
  }
}

// A row's epilogue operands are loaded by lanes 0..2 (one component each) before the
// product, so the row waits once instead of twice; with all of them loaded by lane 0 after
// the sums a smoothing step cost 16.6-20.0 us against 11.2 us for the residual alone (70785
// rows, 64x32x32 hexes).
template <int MODE, typename V>
__global__ __launch_bounds__(kT) void k_mg_rows(MgRowArgs A) {
  constexpr int kRows = kT / kLanesPerRow;
  constexpr bool kCheb = MODE == kMgCheb || MODE == kMgChebAdd;
  const int lane = threadIdx.x % kLanesPerRow;
  const XcdSpan sp = xcd_span(A.nrows);
  const double* __restrict__ x = A.x;
  const V* __restrict__ vals;
  if constexpr (sizeof(V) == 4) vals = A.vals32;
  else vals = A.vals;
  auto X = [&](int c, int j) { return x[3 * (size_t)c + j]; };
  for (int row = sp.lo + sp.j * kRows + threadIdx.x / kLanesPerRow; row < sp.hi; row += sp.bx * kRows) {
    const size_t o = 3 * (size_t)row;
    double rv[3], D[3], dv = 0.0, xv = 0.0, bv = 0.0;
    if (lane < 3) {
#pragma unroll
      for (int j = 0; j < 3; ++j) rv[j] = A.r[o + j];
      if constexpr (MODE != kMgRes) {
#pragma unroll
        for (int j = 0; j < 3; ++j) D[j] = A.dinv[3 * o + 3 * lane + j];
      }
      if constexpr (kCheb) {
        dv = A.d[o + lane];
        xv = x[o + lane];
      }
      if constexpr (MODE == kMgChebAdd) bv = A.base[o + lane];
    }
    double acc[3];
    spmv_row(vals, A.rowmap, A.col, row, lane, X, acc);
    if (lane < 3) {
      const double t[3] = {rv[0] - acc[0], rv[1] - acc[1], rv[2] - acc[2]};
      const double ti = lane == 0 ? t[0] : (lane == 1 ? t[1] : t[2]);
      if constexpr (MODE == kMgRes) {
        A.out[o + lane] = ti;
      } else {
        const double z = D[0] * t[0] + D[1] * t[1] + D[2] * t[2];
        if constexpr (MODE == kMgResCheb0) {
          A.out[o + lane] = ti;
          A.y[o + lane] = A.inv_theta * z;
          A.d[o + lane] = A.inv_theta * z;
        } else {
          const double dn = A.c1 * dv + A.c2 * z;
          A.d[o + lane] = dn;
          A.out[o + lane] = MODE == kMgCheb ? xv + dn : bv + xv + dn;
        }
      }
    }
  }
}

__global__ __launch_bounds__(kT) void k_to_f32(const double* __restrict__ a, float* __restrict__ b, size_t n) {
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) b[i] = (float)a[i];
}

// Spectral estimates (pa_mg.hpp).  What the host-driven form cost at 128x64x64 was the
// host: 16 steps x 5 levels x 2 dot products read back (160 round trips of ~20 us), plus a
// 13 MB start vector built and copied from the host; the kernels' own work is ~1 ms.
// So the scalars stay on the device (each consumer sums the level's partials itself, as in
// the PCG kernels) and one launch serves all levels: the coarse ones are a few work-groups
// each and would be launch-bound alone.
__device__ __forceinline__ int lz_level(const LzArgs& A) {
  int l = 0;
  while (l + 1 < A.nlev && (int)blockIdx.x >= A.L[l + 1].b0) ++l;
  return l;
}

__global__ __launch_bounds__(kT) void k_lz_init(LzArgs A) {
  __shared__ double sh[kT / 64];
  const LzLevel& L = A.L[lz_level(A)];
  const int b = blockIdx.x - L.b0;
  double rz = 0.0;
  for (int n = b * kT + threadIdx.x; n < L.nn; n += L.nb * kT) {
    const size_t o = 3 * (size_t)n;
    double v[3], z[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] = (double)(((unsigned long long)(o + i) * 2654435761ull >> 7) % 2001) / 1000.0 - 1.0;
    dinv3(L.dinv + 9 * (size_t)n, v, z);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      L.r[o + i] = v[i];
      L.z[o + i] = z[i];
      L.p[o + i] = z[i];
      rz += v[i] * z[i];
    }
  }
  const double t = block_reduce_all<kT>(rz, sh);
  if (threadIdx.x == 0) L.P[kLzBlocks + b] = t;
}

__global__ __launch_bounds__(kT) void k_lz_spmv(LzArgs A) {
  __shared__ double sh[kT / 64];
  const LzLevel& L = A.L[lz_level(A)];
  const int b = blockIdx.x - L.b0;
  double dot = 0.0;
  if (L.vals) {
    constexpr int kRows = kT / kLanesPerRow;
    const int lane = threadIdx.x % kLanesPerRow;
    const double* __restrict__ p = L.p;
    auto X = [&](int c, int j) { return p[3 * (size_t)c + j]; };
    for (int row = b * kRows + threadIdx.x / kLanesPerRow; row < L.nn; row += L.nb * kRows) {
      double acc[3];
      spmv_row(L.vals, L.rowmap, L.col, row, lane, X, acc);
      if (lane < 3) {
        const double a = lane == 0 ? acc[0] : (lane == 1 ? acc[1] : acc[2]);
        const size_t d = 3 * (size_t)row + lane;
        L.q[d] = a;
        dot += p[d] * a;
      }
    }
  } else {
    for (size_t i = b * (size_t)kT + threadIdx.x; i < 3 * (size_t)L.nn; i += (size_t)L.nb * kT) dot += L.p[i] * L.q[i];
  }
  const double t = block_reduce_all<kT>(dot, sh);
  if (threadIdx.x == 0) L.P[b] = t;
}

__global__ __launch_bounds__(kT) void k_lz_update(LzArgs A, int step) {
  __shared__ double sh[kT / 64];
  const LzLevel& L = A.L[lz_level(A)];
  const int b = blockIdx.x - L.b0;
  const double pq = sum_partials_all<kT>(L.P, L.nb, sh);
  const double rz = sum_partials_all<kT>(L.P + (1 + (step & 1)) * kLzBlocks, L.nb, sh);
  if (b == 0 && threadIdx.x == 0) {
    L.coef[2 * step] = rz;
    L.coef[2 * step + 1] = pq;
  }
  const double alpha = rz / pq;
  double rzn = 0.0;
  for (int n = b * kT + threadIdx.x; n < L.nn; n += L.nb * kT) {
    const size_t o = 3 * (size_t)n;
    double v[3], z[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) v[i] = L.r[o + i] - alpha * L.q[o + i];
    dinv3(L.dinv + 9 * (size_t)n, v, z);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      L.r[o + i] = v[i];
      L.z[o + i] = z[i];
      rzn += v[i] * z[i];
    }
  }
  const double t = block_reduce_all<kT>(rzn, sh);
  if (threadIdx.x == 0) L.P[(1 + ((step + 1) & 1)) * kLzBlocks + b] = t;
}

__global__ __launch_bounds__(kT) void k_lz_dir(LzArgs A, int step) {
  __shared__ double sh[kT / 64];
  const LzLevel& L = A.L[lz_level(A)];
  const int b = blockIdx.x - L.b0;
  const double rz = sum_partials_all<kT>(L.P + (1 + (step & 1)) * kLzBlocks, L.nb, sh);
  const double rzn = sum_partials_all<kT>(L.P + (1 + ((step + 1) & 1)) * kLzBlocks, L.nb, sh);
  const double beta = rzn / rz;
  for (size_t i = b * (size_t)kT + threadIdx.x; i < 3 * (size_t)L.nn; i += (size_t)L.nb * kT)
    L.p[i] = fma(beta, L.p[i], L.z[i]);
}

// Dense copy of a block-CRS matrix, one work-group per block row.
__global__ __launch_bounds__(64) void k_crs_to_dense(const double* __restrict__ vals, const int* __restrict__ rowmap,
                                                     const int* __restrict__ col, int nn, double* __restrict__ A,
                                                     double* flag) {
  const int r = blockIdx.x, n = 3 * nn;
  if (r == 0 && threadIdx.x == 0) *flag = 0.0;
  double* a = A + (size_t)3 * r * n;
  for (int k = threadIdx.x; k < 3 * n; k += 64) a[k] = 0.0;
  __syncthreads();
  const int s0 = rowmap[r], len = 9 * (rowmap[r + 1] - s0);
  for (int k = threadIdx.x; k < len; k += 64) {
    const int s = s0 + k / 9, i = (k % 9) / 3, j = k % 3;
    a[(size_t)i * n + 3 * col[s] + j] = vals[9 * (size_t)s + 3 * i + j];
  }
}

// In-place Gauss-Jordan inverse of an n x n matrix, n <= 32 kGjTile, by one work-group of
// 32 x 32 threads that holds it in registers (thread (ty, tx) the elements (ty + 32 a,
// tx + 32 b)); a step exchanges its pivot row and column through LDS, one barrier a step.
// 135 dofs (4x2x2 hexes): ~60 us, where the host's Cholesky with its two copies and waits
// took ~0.6 ms.
constexpr int kGjTile = 5;
__global__ __launch_bounds__(1024) void k_gj_small(double* A, int n, double* flag) {
  __shared__ double prow[2][32 * kGjTile], pcol[2][32 * kGjTile];
  const int tx = threadIdx.x % 32, ty = threadIdx.x / 32;
  double m[kGjTile][kGjTile];
#pragma unroll
  for (int a = 0; a < kGjTile; ++a)
#pragma unroll
    for (int b = 0; b < kGjTile; ++b) {
      const int i = ty + 32 * a, j = tx + 32 * b;
      m[a][b] = i < n && j < n ? A[(size_t)i * n + j] : (i == j ? 1.0 : 0.0);
    }
#pragma unroll
  for (int ka = 0; ka < kGjTile; ++ka)
    for (int kr = 0; kr < 32; ++kr) {
      const int k = 32 * ka + kr;
      if (k >= n) break;
      const int h = k & 1;
      if (ty == kr)
#pragma unroll
        for (int b = 0; b < kGjTile; ++b) prow[h][tx + 32 * b] = m[ka][b];
      if (tx == kr)
#pragma unroll
        for (int a = 0; a < kGjTile; ++a) pcol[h][ty + 32 * a] = m[a][ka];
      __syncthreads();  // the other half's readers are one barrier behind
      const double piv = prow[h][k], inv = 1.0 / piv;
      if (!(piv > 0.0) && threadIdx.x == 0) *flag = 1.0;
#pragma unroll
      for (int a = 0; a < kGjTile; ++a) {
        const bool ik = ty + 32 * a == k;
        const double c = pcol[h][ty + 32 * a];
#pragma unroll
        for (int b = 0; b < kGjTile; ++b) {
          const bool jk = tx + 32 * b == k;
          const double r = (jk ? 1.0 : prow[h][tx + 32 * b]) * inv;
          m[a][b] = ik ? r : (jk ? 0.0 : m[a][b]) - c * r;
        }
      }
    }
#pragma unroll
  for (int a = 0; a < kGjTile; ++a)
#pragma unroll
    for (int b = 0; b < kGjTile; ++b) {
      const int i = ty + 32 * a, j = tx + 32 * b;
      if (i < n && j < n) A[(size_t)i * n + j] = m[a][b];
    }
}

// One Gauss-Jordan step of a larger matrix, S -> D (two buffers: every element reads the
// pivot row and column of S).
__global__ __launch_bounds__(kT) void k_gj_step(const double* __restrict__ S, double* __restrict__ D, int n, int k,
                                                double* flag) {
  const double piv = S[(size_t)k * n + k], inv = 1.0 / piv;
  if (!(piv > 0.0) && blockIdx.x == 0 && threadIdx.x == 0) *flag = 1.0;
  for (int i = blockIdx.x; i < n; i += gridDim.x) {
    const double c = S[(size_t)i * n + k];
    for (int j = threadIdx.x; j < n; j += kT) {
      const double r = (j == k ? 1.0 : S[(size_t)k * n + j]) * inv;
      D[(size_t)i * n + j] = i == k ? r : (j == k ? 0.0 : S[(size_t)i * n + j]) - c * r;
    }
  }
}

}  // namespace

hipError_t launch_mg_restrict(const double* rf, double* rc, const int32_t* cgrid, const int32_t* fnode_of_grid,
                              BoxDims fd, const uint8_t* cbcmask, int ncn, hipStream_t s, const double* cdinv,
                              double inv_theta, double* cx, double* cd) {
  k_mg_restrict<<<blocks_of(8 * (size_t)ncn), kT, 0, s>>>(rf, rc, cgrid, fnode_of_grid, fd, cbcmask, ncn, cdinv, inv_theta, cx,
                                              cd);
  return hipGetLastError();
}
hipError_t launch_mg_rows(int mode, const MgRowArgs& a, hipStream_t s) {
  const int grid = red_grid((size_t)a.nrows, kT / kLanesPerRow);
  if (a.vals32) {
    switch (mode) {
      case kMgRes: k_mg_rows<kMgRes, float><<<grid, kT, 0, s>>>(a); break;
      case kMgResCheb0: k_mg_rows<kMgResCheb0, float><<<grid, kT, 0, s>>>(a); break;
      case kMgCheb: k_mg_rows<kMgCheb, float><<<grid, kT, 0, s>>>(a); break;
      case kMgChebAdd: k_mg_rows<kMgChebAdd, float><<<grid, kT, 0, s>>>(a); break;
      default: return hipErrorInvalidValue;
    }
  } else {
    switch (mode) {
      case kMgRes: k_mg_rows<kMgRes, double><<<grid, kT, 0, s>>>(a); break;
      case kMgResCheb0: k_mg_rows<kMgResCheb0, double><<<grid, kT, 0, s>>>(a); break;
      case kMgCheb: k_mg_rows<kMgCheb, double><<<grid, kT, 0, s>>>(a); break;
      case kMgChebAdd: k_mg_rows<kMgChebAdd, double><<<grid, kT, 0, s>>>(a); break;
      default: return hipErrorInvalidValue;
    }
  }
  return hipGetLastError();
}
hipError_t launch_to_f32(const double* a, float* b, size_t n, hipStream_t s) {
  k_to_f32<<<blocks_of(n), kT, 0, s>>>(a, b, n);
  return hipGetLastError();
}
hipError_t launch_mg_prolong_add(const double* ec, double* xf, const int32_t* fgrid, const int32_t* cnode_of_grid,
                                 BoxDims cd, const uint8_t* fbcmask, int nfn, hipStream_t s,
                                 const MgLattice& lat) {
  k_mg_prolong_add<<<blocks_of(nfn), kT, 0, s>>>(ec, xf, fgrid, cnode_of_grid, cd, fbcmask, nfn, lat);
  return hipGetLastError();
}
hipError_t launch_mg_wrestrict(const double* wf, double* wc, const int32_t* cgrid, const int32_t* fnode_of_grid,
                               BoxDims fd, int ncn, hipStream_t s) {
  k_mg_wrestrict<<<blocks_of(ncn), kT, 0, s>>>(wf, wc, cgrid, fnode_of_grid, fd, ncn);
  return hipGetLastError();
}
hipError_t launch_simp_w(const double* z, double* w, int n, const Material& m, hipStream_t s) {
  k_simp_w<<<blocks_of(n), kT, 0, s>>>(z, w, n, m);
  return hipGetLastError();
}
hipError_t launch_cheb_first(double* x, double* d, const double* r, const double* dinv, double inv_theta, int nn,
                             hipStream_t s, const double* t, const MgLattice& lat) {
  k_cheb_first<<<blocks_of(nn), kT, 0, s>>>(x, d, r, dinv, inv_theta, nn, t, lat);
  return hipGetLastError();
}
hipError_t launch_cheb_next(double* x, double* d, const double* r, const double* Kx, const double* dinv, double c1,
                            double c2, int nn, hipStream_t s) {
  k_cheb_next<<<blocks_of(nn), kT, 0, s>>>(x, d, r, Kx, dinv, c1, c2, nn);
  return hipGetLastError();
}
hipError_t launch_sub(double* out, const double* a, const double* b, size_t n, hipStream_t s) {
  k_sub<<<blocks_of(n), kT, 0, s>>>(out, a, b, n);
  return hipGetLastError();
}
hipError_t launch_add(double* y, const double* x, size_t n, hipStream_t s) {
  k_add<<<blocks_of(n), kT, 0, s>>>(y, x, n);
  return hipGetLastError();
}
hipError_t launch_add2(double* out, const double* a, const double* b, size_t n, hipStream_t s) {
  k_add2<<<blocks_of(n), kT, 0, s>>>(out, a, b, n);
  return hipGetLastError();
}
hipError_t launch_dense_gemv(const double* A, const double* x, double* y, int n, hipStream_t s) {
  k_dense_gemv<<<std::max(1, std::min(1024, (n + 3) / 4)), kT, 0, s>>>(A, x, y, n);
  return hipGetLastError();
}
hipError_t launch_mg_update(double* x, double* r, const double* p, const double* q, const double* scal, int nn,
                            double* P_rr, int grid, hipStream_t s, double* z, const double* dinv, double inv_theta,
                            const MgLattice& lat) {
  k_mg_update<<<grid, kT, 0, s>>>(x, r, p, q, scal, nn, P_rr, z, dinv, inv_theta, lat);
  return hipGetLastError();
}
hipError_t launch_mg_pupdate(double* p, const double* z, const double* scal, int nn, int first, hipStream_t s,
                             const MgLattice& lat) {
  k_mg_pupdate<<<blocks_of(nn), kT, 0, s>>>(p, z, scal, nn, first, lat);
  return hipGetLastError();
}

hipError_t launch_lz_init(const LzArgs& a, hipStream_t s) {
  k_lz_init<<<a.blocks, kT, 0, s>>>(a);
  return hipGetLastError();
}
hipError_t launch_lz_spmv(const LzArgs& a, hipStream_t s) {
  k_lz_spmv<<<a.blocks, kT, 0, s>>>(a);
  return hipGetLastError();
}
hipError_t launch_lz_update(const LzArgs& a, int step, hipStream_t s) {
  k_lz_update<<<a.blocks, kT, 0, s>>>(a, step);
  return hipGetLastError();
}
hipError_t launch_lz_dir(const LzArgs& a, int step, hipStream_t s) {
  k_lz_dir<<<a.blocks, kT, 0, s>>>(a, step);
  return hipGetLastError();
}
size_t mg_dense_scratch(int nn) {
  const size_t n = 3 * (size_t)nn;
  return n <= 32 * kGjTile ? 0 : n * n;
}
hipError_t launch_mg_dense_inverse(const double* vals, const int32_t* rowmap, const int32_t* col, int nn, double* A,
                                   double* T, double* flag, hipStream_t s) {
  const int n = 3 * nn;
  if (n <= 32 * kGjTile) {
    k_crs_to_dense<<<nn, 64, 0, s>>>(vals, rowmap, col, nn, A, flag);
    k_gj_small<<<1, 1024, 0, s>>>(A, n, flag);
    return hipGetLastError();
  }
  // n steps between the two buffers, ending in A
  double* src = n % 2 ? T : A;
  k_crs_to_dense<<<nn, 64, 0, s>>>(vals, rowmap, col, nn, src, flag);
  for (int k = 0; k < n; ++k) {
    double* dst = src == A ? T : A;
    k_gj_step<<<std::min(n, 2048), kT, 0, s>>>(src, dst, n, k, flag);
    src = dst;
  }
  return hipGetLastError();
}

}  // namespace pa
