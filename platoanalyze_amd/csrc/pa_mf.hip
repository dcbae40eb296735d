// Mixed-precision solve: FP32 matrix-free operator inside an FP64 Jacobi-PCG (FP64
// vectors and reductions, residual replaced by the true FP64 residual f - K u).
#include "pa_mf.hpp"
#include "pa_dpp.hpp"
#include "pa_fixed.hpp"
#include "pa_reduce.hpp"
#include "pa_solver.hpp"

namespace pa {

namespace {

constexpr int kT = 256;

__device__ __forceinline__ int xcd_map(int b, int n) {
  const int q = n / kNumXcd, r = n % kNumXcd;
  const int x = b % kNumXcd, k = b / kNumXcd;
  return x * q + (x < r ? x : r) + k;
}

__device__ __forceinline__ float powi_n(float x, int n) {  // n >= 1
  float r = x;
  for (int k = 1; k < n; ++k) r *= x;
  return r;
}

__device__ __forceinline__ float powi_f(float x, float p, int pint) {
  if (pint > 0) {
    float r = x;
    for (int k = 1; k < pint; ++k) r *= x;
    return r;
  }
  return powf(x, p);
}

template <typename T>
__device__ __forceinline__ void gradients_t(const T x[4][3], T g[4][3], T& vol) {
  const T j11 = x[0][0] - x[3][0], j12 = x[1][0] - x[3][0], j13 = x[2][0] - x[3][0];
  const T j21 = x[0][1] - x[3][1], j22 = x[1][1] - x[3][1], j23 = x[2][1] - x[3][1];
  const T j31 = x[0][2] - x[3][2], j32 = x[1][2] - x[3][2], j33 = x[2][2] - x[3][2];
  const T det = j11 * j22 * j33 + j12 * j23 * j31 + j13 * j21 * j32 - j11 * j23 * j32 - j12 * j21 * j33 -
                j13 * j22 * j31;
  const T inv = T(1) / det;
  g[0][0] = (j22 * j33 - j23 * j32) * inv;
  g[0][1] = (j13 * j32 - j12 * j33) * inv;
  g[0][2] = (j12 * j23 - j13 * j22) * inv;
  g[1][0] = (j23 * j31 - j21 * j33) * inv;
  g[1][1] = (j11 * j33 - j13 * j31) * inv;
  g[1][2] = (j13 * j21 - j11 * j23) * inv;
  g[2][0] = (j21 * j32 - j22 * j31) * inv;
  g[2][1] = (j12 * j31 - j11 * j32) * inv;
  g[2][2] = (j11 * j22 - j12 * j21) * inv;
#pragma unroll
  for (int d = 0; d < 3; ++d) g[3][d] = -(g[0][d] + g[1][d] + g[2][d]);
  vol = fabs(det) * (T(1) / T(6));
}

// FP32 nodal forces K_e p_e of the element with local nodes ln (SIMP_INT: SIMP with an integer
// exponent; the other models' FP64 powers double the registers)
template <bool SIMP_INT>
__device__ __forceinline__ void mf_element(const Material& m, float c00, float c01, float c33, float rmin, float pp,
                                           const float4* nd4, const float* xl, const int ln[4], float F[4][3]) {
  float x[4][3], g[4][3], u[4][3], vol, rho = 0.0f;
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    const float4 p = nd4[ln[a]];
    x[a][0] = p.x;
    x[a][1] = p.y;
    x[a][2] = p.z;
    rho += p.w;
#pragma unroll
    for (int i = 0; i < 3; ++i) u[a][i] = xl[3 * ln[a] + i];
  }
  gradients_t(x, g, vol);
  rho *= 0.25f;
  const float vw = vol * (SIMP_INT || m.model == kPenaltySimp ? rmin + (1.0f - rmin) * (SIMP_INT ? powi_n(rho, m.pint) : powi_f(rho, pp, m.pint))
                                                    : (float)penalty_w(m, (double)rho));
  float e[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    e[0] += u[a][0] * g[a][0];
    e[1] += u[a][1] * g[a][1];
    e[2] += u[a][2] * g[a][2];
    e[3] += u[a][2] * g[a][1] + u[a][1] * g[a][2];
    e[4] += u[a][2] * g[a][0] + u[a][0] * g[a][2];
    e[5] += u[a][1] * g[a][0] + u[a][0] * g[a][1];
  }
  const float s0 = vw * (c00 * e[0] + c01 * e[1] + c01 * e[2]);
  const float s1 = vw * (c01 * e[0] + c00 * e[1] + c01 * e[2]);
  const float s2 = vw * (c01 * e[0] + c01 * e[1] + c00 * e[2]);
  const float s3 = vw * c33 * e[3], s4 = vw * c33 * e[4], s5 = vw * c33 * e[5];
#pragma unroll
  for (int a = 0; a < 4; ++a) {
    F[a][0] = s0 * g[a][0] + s5 * g[a][1] + s4 * g[a][2];
    F[a][1] = s5 * g[a][0] + s1 * g[a][1] + s3 * g[a][2];
    F[a][2] = s4 * g[a][0] + s3 * g[a][1] + s2 * g[a][2];
  }
}

// q = K p with the PCG direction update fused in; one work-group per chunk.  The
// vectors are FP64; the element operator is FP32: the node table (FP32 coordinates +
// density) and p = z + beta p_prev at the table's nodes (rounded to FP32, constrained
// dofs 0) are staged in LDS, the element loop computes K_e p_e in FP32 and adds it into
// 64-bit fixed-point row accumulators (scale from the chunk's largest |p|: the sums do
// not depend on the order of the adds), and the rows are written back with the
// chunk's p.q partial.
// The chunk's own rows of p_cur are written in FP64 (unrounded).
template <int NT>
__global__ __launch_bounds__(NT) void k_mf_apply(MfArgs A) {
  // LDS: own-row p and row accumulators (FP64, 3 x even(max_rows) each: multiples of
  // 16 bytes), node table, p at the table's nodes (FP32).  FP64 LDS atomics run at
  // several times the rate of FP32 ones on this part, and add no rounding of their own.
  extern __shared__ double smem_d[];
  const int mr2 = (A.max_rows + 1) & ~1;
  double* pown = smem_d;
  double* acc = pown + 3 * mr2;
  float4* nd4 = reinterpret_cast<float4*>(acc + 3 * mr2);
  float* xl = reinterpret_cast<float*>(nd4 + A.max_nodes);
  __shared__ double sh[2 * NT / 64];
  __shared__ double red[NT / 64];

  double beta = 0.0;
  if (!A.first) {
    double a = A.P_rz_new[0], b = A.P_rz_old[0];
    if (A.np_rz > 1) sum_partials_two<NT>(A.P_rz_new, A.np_rz, A.P_rz_old, A.np_rz, sh, a, b);
    beta = a / b;
  }
  const int c = xcd_map(blockIdx.x, A.nchunks);
  const int r0 = A.chunk_rows[c], r1 = A.chunk_rows[c + 1], nr = r1 - r0;
  const int n0 = A.node_offs[c], nnode = A.node_offs[c + 1] - n0;
  double pmax = 0.0;
  for (int k = threadIdx.x; k < nnode; k += NT) {
    const int gid = A.nodes[n0 + k];
    nd4[k] = A.Xz[gid];
    const uint32_t bm = A.bcmask[gid];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const size_t d = 3 * (size_t)gid + i;
      double v = A.first ? A.z[d] : fma(beta, A.p_prev[d], A.z[d]);
      v = (bm >> i) & 1u ? 0.0 : v;
      xl[3 * k + i] = (float)v;
      pmax = max_nan(pmax, fabs((double)(float)v));
      if (k < nr) {  // rows come first in the table
        A.p_cur[d] = v;
        pown[3 * k + i] = v;
      }
    }
  }
  for (int k = threadIdx.x; k < 3 * nr; k += NT) acc[k] = 0.0;
  block_max_write<NT>(pmax, red);
  __syncthreads();
  // |contribution| <= vol |grad N|^2 * 3 * (|c00| + 2|c01| + |c33|) * 8 max|p| for weights
  // <= 1, plus FP32 rounding (the factor 2)
  const double S = fixed_scale_54(48.0 * (fabs(A.m.c00) + 2.0 * fabs(A.m.c01) + fabs(A.m.c33)) *
                                  (double)A.gbound[c] * block_max_read<NT>(red));

  const float c00 = (float)A.m.c00, c01 = (float)A.m.c01, c33 = (float)A.m.c33;
  const float rmin = (float)A.m.rmin, pp = (float)A.m.p;
  const int l0 = A.list_offs[c], l1 = A.list_offs[c + 1];
  for (int k = l0 + threadIdx.x; k < l1; k += NT) {
    const uint2 lw = reinterpret_cast<const uint2*>(A.ent_ln)[k];
    const int ln[4] = {(int)(lw.x & 0xFFFFu), (int)(lw.x >> 16), (int)(lw.y & 0xFFFFu), (int)(lw.y >> 16)};
    float F[4][3];
    mf_element<false>(A.m, c00, c01, c33, rmin, pp, nd4, xl, ln, F);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if (ln[a] < nr) {
        double* dst = &acc[3 * ln[a]];
#pragma unroll
        for (int i = 0; i < 3; ++i) lds_add_fixed64(dst + i, (double)F[a][i], S);
      }
    }
  }
  __syncthreads();
  double dot = 0.0;
  const double inv = 1.0 / S;  // a power of two: exact (NaN for a non-finite p)
  for (int k = threadIdx.x; k < 3 * nr; k += NT) {
    const size_t gd = 3 * (size_t)r0 + k;
    const double pv = pown[k];
    const double av = S == S ? fixed_value(acc[k], inv) : NAN;
    const double yv = (A.bcmask[r0 + k / 3] >> (k % 3)) & 1u ? pv : av;
    A.y[gd] = yv;
    dot += pv * yv;
  }
  const double t = block_reduce_all<NT>(dot, sh);
  if (threadIdx.x == 0) A.partials[c] = t;
}

// k_mf_apply without atomics: the elements leave their FP32 forces in LDS and four lanes a
// row add its own in FP64, in list order.  No accumulators to clear, no scale (a maximum
// over the work-group and a barrier), no conversions to and from fixed point.  The element
// and row lists and the nodes are on their way from memory while beta is summed.  What is
// left on small meshes is a chain of memory and LDS latencies, one pass of 512 threads over
// a chunk's 500 to 800 elements.  Graded hexes, against k_mf_apply: 35x19x17 (67830 tets)
// 9.0 -> 7.0 us an apply, 97x51x45 (1.34 million) 66 -> 55 us an iteration; 256 threads
// 7.6 us and 58 us.
template <int NT>
__global__ __launch_bounds__(NT, 4) void k_mf_gather(MfArgs A) {
  extern __shared__ double smem_d[];
  double* pown = smem_d;  // own-row p (FP64), node table, p at its nodes, forces [entry][4][3]
  float4* nd4 = reinterpret_cast<float4*>(pown + 3 * ((A.max_rows + 1) & ~1));
  float4* fl = nd4 + A.max_nodes;
  float* xl = reinterpret_cast<float*>(fl + 3 * A.max_list);
  __shared__ double sh[2 * NT / 64];
  constexpr int kInc = 8;  // prefetched incidences of a lane (four lanes a row)

  const int c = xcd_map(blockIdx.x, A.nchunks);
  const int r0 = A.chunk_rows[c], nr = A.chunk_rows[c + 1] - r0;
  const int n0 = A.node_offs[c], nnode = A.node_offs[c + 1] - n0;
  const int l0 = A.list_offs[c], l1 = A.list_offs[c + 1];
  const int lane = threadIdx.x & 3, lr0 = threadIdx.x >> 2;
  const uint2* ents = reinterpret_cast<const uint2*>(A.ent_ln);
  uint2 ent = l0 + (int)threadIdx.x < l1 ? ents[l0 + threadIdx.x] : uint2{0, 0};
  const int row0 = r0 + min(lr0, nr - 1);
  const int i0 = A.inc_offs[row0] + lane, i1 = A.inc_offs[row0 + 1];
  int inc[kInc];
#pragma unroll
  for (int k = 0; k < kInc; ++k) inc[k] = A.inc[max(0, min(i0 + 4 * k, i1 - 1))];
  // a thread's first node is on its way while beta is summed
  struct Node {
    int gid;
    float4 x;
    uint32_t bm;
    double z[3], p[3];
  };
  auto load = [&](int k) {
    Node n;
    n.gid = A.nodes[n0 + k];
    n.x = A.Xz[n.gid];
    n.bm = A.bcmask[n.gid];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      n.z[i] = A.z[3 * (size_t)n.gid + i];
      n.p[i] = A.first ? 0.0 : A.p_prev[3 * (size_t)n.gid + i];
    }
    return n;
  };
  const Node mine = load(min((int)threadIdx.x, nnode - 1));
  double beta = 0.0;
  if (!A.first) {
    double a, b;
    sum_partials_two<NT>(A.P_rz_new, A.np_rz, A.P_rz_old, A.np_rz, sh, a, b);
    beta = a / b;
  }
  auto store = [&](int k, const Node& n) {
    nd4[k] = n.x;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      double v = A.first ? n.z[i] : fma(beta, n.p[i], n.z[i]);
      v = (n.bm >> i) & 1u ? 0.0 : v;
      xl[3 * k + i] = (float)v;
      if (k < nr) {  // rows come first in the table
        A.p_cur[3 * (size_t)n.gid + i] = v;
        pown[3 * k + i] = v;
      }
    }
  };
  if ((int)threadIdx.x < nnode) store(threadIdx.x, mine);
  for (int k = threadIdx.x + NT; k < nnode; k += NT) store(k, load(k));
  __syncthreads();
  const float c00 = (float)A.m.c00, c01 = (float)A.m.c01, c33 = (float)A.m.c33;
  const float rmin = (float)A.m.rmin, pp = (float)A.m.p;
  for (int k = l0 + threadIdx.x; k < l1; k += NT) {
    const int ln[4] = {(int)(ent.x & 0xFFFFu), (int)(ent.x >> 16), (int)(ent.y & 0xFFFFu), (int)(ent.y >> 16)};
    if (k + NT < l1) ent = ents[k + NT];
    float F[4][3];
    mf_element<true>(A.m, c00, c01, c33, rmin, pp, nd4, xl, ln, F);
    float4* f = fl + 3 * (k - l0);
    f[0] = make_float4(F[0][0], F[0][1], F[0][2], F[1][0]);
    f[1] = make_float4(F[1][1], F[1][2], F[2][0], F[2][1]);
    f[2] = make_float4(F[2][2], F[3][0], F[3][1], F[3][2]);
  }
  __syncthreads();
  const float* ff = reinterpret_cast<const float*>(fl);
  double dot = 0.0;
  for (int lr = lr0; lr < nr; lr += NT / 4) {
    double s[3] = {0.0, 0.0, 0.0};
    auto add = [&](int e) {
#pragma unroll
      for (int i = 0; i < 3; ++i) s[i] += (double)ff[3 * e + i];
    };
    int i = A.inc_offs[r0 + lr] + lane;
    const int end = A.inc_offs[r0 + lr + 1];
    if (lr == lr0) {
#pragma unroll
      for (int k = 0; k < kInc; ++k)
        if (i + 4 * k < end) add(inc[k]);
      i += 4 * kInc;
    }
    for (; i < end; i += 4) add(A.inc[i]);
#pragma unroll
    for (int q = 0; q < 3; ++q) {  // the four lanes receive the same bits
      s[q] += dpp_f64<kDppXor1>(s[q]);
      s[q] += dpp_f64<kDppXor2>(s[q]);
    }
    if (lane < 3) {
      const double pv = pown[3 * lr + lane];
      const double av = lane == 0 ? s[0] : lane == 1 ? s[1] : s[2];
      const double yv = (A.bcmask[r0 + lr] >> lane) & 1u ? pv : av;
      A.y[3 * (size_t)(r0 + lr) + lane] = yv;
      dot += pv * yv;
    }
  }
  const double t = block_reduce_all<NT>(dot, sh);
  if (threadIdx.x == 0) A.partials[c] = t;
}

// Diagonal blocks K_rr (FP64) accumulated per owned vertex, then inverted per row.
template <int NT>
__global__ __launch_bounds__(NT) void k_mf_diag(DiagArgs A) {
  extern __shared__ double dsm[];
  double* D = dsm;  // 9 per row
  const int c = xcd_map(blockIdx.x, A.nchunks);
  const int r0 = A.chunk_rows[c], r1 = A.chunk_rows[c + 1], nr = r1 - r0;
  const int n0 = A.node_offs[c];
  for (int k = threadIdx.x; k < 9 * nr; k += NT) D[k] = 0.0;
  __syncthreads();
  // fixed-point sums (order-independent): |contribution| <= vol |grad N|^2 (|c01| + 2|c33|)
  const double S = fixed_scale_54((double)A.gbound[c] * (fabs(A.m.c01) + 2.0 * fabs(A.m.c33)));
  const int l0 = A.list_offs[c], l1 = A.list_offs[c + 1];
  for (int k = l0 + threadIdx.x; k < l1; k += NT) {
    const uint2 lw = reinterpret_cast<const uint2*>(A.ent_ln)[k];
    const int ln[4] = {(int)(lw.x & 0xFFFFu), (int)(lw.x >> 16), (int)(lw.y & 0xFFFFu), (int)(lw.y >> 16)};
    double x[4][3], g[4][3], vol, rho = 0.0;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      const size_t gid = (size_t)A.nodes[n0 + ln[a]];
#pragma unroll
      for (int d = 0; d < 3; ++d) x[a][d] = A.X[3 * gid + d];
      rho += A.z[gid];
    }
    gradients_t(x, g, vol);
    rho = rho / 4.0;
    const double vw = vol * penalty_w(A.m, rho);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if (ln[a] >= nr) continue;
      const double gg = g[a][0] * g[a][0] + g[a][1] * g[a][1] + g[a][2] * g[a][2];
      double* dst = &D[9 * ln[a]];
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) {
          double v = (A.m.c01 + A.m.c33) * g[a][i] * g[a][j];
          if (i == j) v += A.m.c33 * gg;
          lds_add_fixed64(dst + 3 * i + j, vw * v, S);
        }
    }
  }
  __syncthreads();
  const double inv = 1.0 / S;
  for (int lr = threadIdx.x; lr < nr; lr += NT) {
    double a[9];
#pragma unroll
    for (int q = 0; q < 9; ++q) a[q] = fixed_value(D[9 * lr + q], inv);
    block_inv3_masked(a, A.bcmask[r0 + lr], A.dinv + 9 * (size_t)(r0 + lr));
  }
}

__device__ __forceinline__ void dinv3(const double* __restrict__ D, const double r[3], double z[3]) {
  z[0] = D[0] * r[0] + D[1] * r[1] + D[2] * r[2];
  z[1] = D[3] * r[0] + D[4] * r[1] + D[5] * r[2];
  z[2] = D[6] * r[0] + D[7] * r[1] + D[8] * r[2];
}

// z = Dinv r; partials of r.z
__global__ __launch_bounds__(kT) void k_pcgm_init(const double* __restrict__ r, double* __restrict__ z,
                                                  const double* __restrict__ dinv, int nn,
                                                  double* __restrict__ P_rz) {
  __shared__ double sh[kT / 64];
  double rz = 0.0;
  const XcdSpan sp = xcd_span(nn);
  for (int n = sp.lo + sp.j * kT + threadIdx.x; n < sp.hi; n += sp.bx * kT) {
    const size_t d = 3 * (size_t)n;
    const double rv[3] = {r[d], r[d + 1], r[d + 2]};
    double zv[3];
    dinv3(dinv + 9 * (size_t)n, rv, zv);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      z[d + i] = zv[i];
      rz += rv[i] * zv[i];
    }
  }
  const double t = block_reduce_all<kT>(rz, sh);
  if (threadIdx.x == 0) P_rz[blockIdx.x] = t;
}

constexpr int kFin = 1024;  // threads of the one-work-group finishers

__global__ __launch_bounds__(kFin) void k_pcgm_alpha(const double* partials, int n, double* scal) {
  __shared__ double sh[kFin / 64];
  const double pq = sum_partials_wide<kFin>(partials, n, sh);
  if (threadIdx.x == 0) {
    scal[kPQ] = pq;
    scal[kAlpha] = scal[kRZ] / pq;
  }
}

__global__ __launch_bounds__(kFin) void k_pcgm_beta(const double* P_rz, int n, double* scal, int mode) {
  __shared__ double sh[kFin / 64];
  const double rz = sum_partials_wide<kFin>(P_rz, n, sh);
  if (threadIdx.x == 0) {
    if (mode == kBetaStep) scal[kBeta] = rz / scal[kRZ];
    scal[kRZ] = rz;
  }
}

// r = mask(b - R) (b optional); partials of r.r
__global__ __launch_bounds__(kT) void k_neg_mask(const double* __restrict__ R, const double* __restrict__ b,
                                                 const uint8_t* __restrict__ bcmask, double* __restrict__ r, int nn,
                                                 double* __restrict__ P) {
  __shared__ double sh[kT / 64];
  double rr = 0.0;
  const XcdSpan sp = xcd_span(nn);
  for (int n = sp.lo + sp.j * kT + threadIdx.x; n < sp.hi; n += sp.bx * kT) {
    const uint32_t bm = bcmask[n];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const size_t d = 3 * (size_t)n + i;
      const double v = (bm >> i) & 1u ? 0.0 : (b ? b[d] : 0.0) - R[d];
      r[d] = v;
      rr += v * v;
    }
  }
  const double t = block_reduce_all<kT>(rr, sh);
  if (threadIdx.x == 0) P[blockIdx.x] = t;
}

__global__ __launch_bounds__(kT) void k_jacobi_step(double* __restrict__ u, const double* __restrict__ Ku,
                                                    const double* __restrict__ dinv, const uint8_t* __restrict__ bcmask,
                                                    int nn, double omega) {
  for (int n = blockIdx.x * kT + threadIdx.x; n < nn; n += gridDim.x * kT) {
    const size_t d = 3 * (size_t)n;
    const double r[3] = {Ku[d], Ku[d + 1], Ku[d + 2]};
    double c[3];
    dinv3(dinv + 9 * (size_t)n, r, c);
    const uint32_t bm = bcmask[n];
#pragma unroll
    for (int i = 0; i < 3; ++i)
      if (!((bm >> i) & 1u)) u[d + i] -= omega * c[i];
  }
}

__global__ __launch_bounds__(kT) void k_make_xz(const double* X, const double* z, float4* Xz, int nn) {
  for (int n = blockIdx.x * kT + threadIdx.x; n < nn; n += gridDim.x * kT)
    Xz[n] = make_float4((float)X[3 * (size_t)n], (float)X[3 * (size_t)n + 1], (float)X[3 * (size_t)n + 2],
                        (float)z[n]);
}

int grid_of(size_t n, int cap = 1024) {
  size_t g = (n + kT - 1) / kT;
  return (int)(g < 1 ? 1 : (g > (size_t)cap ? cap : g));
}

}  // namespace

static size_t mf_gather_lds(const MfArgs& a) {
  return sizeof(double) * 3 * ((a.max_rows + 1) & ~1) + sizeof(float4) * (a.max_nodes + 3 * (size_t)a.max_list) +
         sizeof(float) * 3 * a.max_nodes;
}
// Forces in LDS where two work-groups still share a CU (Kuhn meshes: 750 entries, 44 KB);
// denser chunks add with atomics.  So do all penalty models but SIMP with an integer exponent:
// with every model's code k_mf_gather spills at its register limit, and from 51x27x25 hexes on
// it is the slower one (us an iteration, RAMP, 97x51x45: graded hexes 81 against 64 with
// k_mf_apply, five tets 119 and 82; below, within 7 % either way).
bool mf_gathers(const MfArgs& a) {
  return a.inc && mf_gather_lds(a) <= 64 * 1024 && a.m.model == kPenaltySimp && a.m.pint > 0;
}

hipError_t launch_mf_apply(const MfArgs& a, hipStream_t s) {
  if (mf_gathers(a)) {
    k_mf_gather<512><<<a.nchunks, 512, mf_gather_lds(a), s>>>(a);
    return hipGetLastError();
  }
  const size_t lds = sizeof(double) * 6 * ((a.max_rows + 1) & ~1) + sizeof(float4) * a.max_nodes +
                     sizeof(float) * 3 * a.max_nodes;
  k_mf_apply<256><<<a.nchunks, 256, lds, s>>>(a);
  return hipGetLastError();
}
hipError_t launch_mf_diag_inv(const DiagArgs& a, hipStream_t s) {
  k_mf_diag<256><<<a.nchunks, 256, sizeof(double) * 9 * a.max_rows, s>>>(a);
  return hipGetLastError();
}
hipError_t launch_pcgm_init(const double* r, double* z, const double* dinv, int nn, double* P_rz, int grid,
                            hipStream_t s) {
  k_pcgm_init<<<grid, kT, 0, s>>>(r, z, dinv, nn, P_rz);
  return hipGetLastError();
}
hipError_t launch_pcgm_alpha(const double* partials, int n, double* scal, hipStream_t s) {
  k_pcgm_alpha<<<1, kFin, 0, s>>>(partials, n, scal);
  return hipGetLastError();
}
hipError_t launch_pcgm_beta(const double* P_rz, int n, double* scal, int mode, hipStream_t s) {
  k_pcgm_beta<<<1, kFin, 0, s>>>(P_rz, n, scal, mode);
  return hipGetLastError();
}
hipError_t launch_neg_mask(const double* R, const double* b, const uint8_t* bcmask, double* r, int nn, double* P,
                           int grid, hipStream_t s) {
  k_neg_mask<<<grid, kT, 0, s>>>(R, b, bcmask, r, nn, P);
  return hipGetLastError();
}
hipError_t launch_jacobi_step(double* u, const double* Ku, const double* dinv, const uint8_t* bcmask, int nn,
                              double omega, hipStream_t s) {
  k_jacobi_step<<<grid_of(nn, 4096), kT, 0, s>>>(u, Ku, dinv, bcmask, nn, omega);
  return hipGetLastError();
}
hipError_t launch_make_xz(const double* X, const double* z, float4* Xz, int nn, hipStream_t s) {
  k_make_xz<<<grid_of(nn, 4096), kT, 0, s>>>(X, z, Xz, nn);
  return hipGetLastError();
}

}  // namespace pa
