// Jacobian assembly of Kuhn-split box lattices (pa_boxjac.hpp).
//
// In the tet of axis path (a, b, c) the vertex gradients are -e_a/h_a, e_a/h_a - e_b/h_b,
// e_b/h_b - e_c/h_c and e_c/h_c, so a block K_{p, p+d} has few nonzero terms, each a sum of
// at most six element weights times lambda or mu over two spacings.  A work-group takes up to
// 32 consecutive rows (one contiguous piece of the CRS values), gathers z and u of the
// points around them once, computes the weights of the hexes around them in LDS, and each
// wave forms the blocks of two of the seven edge directions: one half of its lanes the block
// of p = r towards r + d, the other half that of p = r - d, transposed.  The blocks are
// staged in LDS and streamed out in whole lines.
//
// The general lattice kernels need a scatter of z and u and a pass over the weights before
// they start, gather up to six weights a block from global memory (105 loads of 64 scattered
// lanes for 32 rows) and multiply each with a 3x3 block from LDS.  K and R, general -> this:
// 20x10x10 17.7 -> 10.6 us, 64x32x32 33 -> 20, 128x64x64 174 -> 126, 200x100x100 640 -> 435,
// 256x128x128 1640 -> 1305 us (3.5 TB/s of values; streaming alone takes 757 us, and the
// kernel without its stores 943 us: four work-groups a CU, all the staging LDS holds, do not
// overlap the two further).  Tried and slower: two to three tiles in flight through persistent
// work-groups (registers spill), storing waves of their own, 24-row tiles, plain stores
// (128x64x64 185 us: they push the gathered z and u out of the caches).
#include "pa_boxjac.hpp"

#include <algorithm>
#include <type_traits>

#include "pa_box.hpp"
#include "pa_reduce.hpp"
#include "pa_solver.hpp"

// K alone and K with R are two instances; products and sums are fused only where written, so
// that both give the same bits.
#pragma clang fp contract(off)

namespace pa {

namespace {

constexpr int kT = 256;

// index of the path that starts (a, b) in kKuhnPath's order
__host__ __device__ constexpr int path_of(int a, int b) { return 2 * a + (b == (a + 2) % 3 ? (a == 1 ? 0 : 1) : (a == 1 ? 1 : 0)); }
static_assert(path_of(0, 1) == 0 && path_of(0, 2) == 1 && path_of(1, 0) == 2 && path_of(1, 2) == 3 &&
                  path_of(2, 0) == 4 && path_of(2, 1) == 5,
              "paths in lexicographic order");

struct Hexes {  // weights of the tile's hexes and the strides of its hex lattice
  const double (*w)[kJacHexes];
  int s[3];
};

// Sum of the weights of the six tets at the axis edge from the lower corner of hex p.
template <int a>
__device__ __forceinline__ double axis_sum(const Hexes& H, int p) {
  constexpr int b = (a + 1) % 3, c = (a + 2) % 3;
  const int pb = p - H.s[b], pc = p - H.s[c], pbc = pb - H.s[c];
  return H.w[path_of(a, b)][p] + H.w[path_of(a, c)][p] + H.w[path_of(b, a)][pb] + H.w[path_of(c, a)][pc] +
         H.w[path_of(b, c)][pbc] + H.w[path_of(c, b)][pbc];
}

// Blocks K_{p, p + d}, p the lower corner of hex p: d = e_a, e_a + e_b, e_x + e_y + e_z.
template <int a>
__device__ __forceinline__ void axis_block(const BoxJacArgs& A, const Hexes& H, int p, double M[3][3]) {
  constexpr int b = (a + 1) % 3, c = (a + 2) % 3;
  const int pb = p - H.s[b], pc = p - H.s[c], pbc = pb - H.s[c];
  const double w1 = H.w[path_of(a, b)][p], w2 = H.w[path_of(a, c)][p], w3 = H.w[path_of(b, a)][pb],
               w4 = H.w[path_of(c, a)][pc], w5 = H.w[path_of(b, c)][pbc], w6 = H.w[path_of(c, b)][pbc];
  const double E = A.h[a][a] * (((w1 + w2) + (w3 + w4)) + (w5 + w6));
  const double ab = w1 + w4, ba = w3 + w6, ac = w2 + w3, ca = w4 + w5;
  M[a][a] = -(A.lam + 2.0 * A.mu) * E;
  M[b][b] = M[c][c] = -A.mu * E;
  M[a][b] = A.h[a][b] * fma(A.lam, ab, A.mu * ba);
  M[b][a] = A.h[a][b] * fma(A.lam, ba, A.mu * ab);
  M[a][c] = A.h[a][c] * fma(A.lam, ac, A.mu * ca);
  M[c][a] = A.h[a][c] * fma(A.lam, ca, A.mu * ac);
  M[b][c] = -A.h[b][c] * fma(A.lam, w3, A.mu * w4);
  M[c][b] = -A.h[b][c] * fma(A.lam, w4, A.mu * w3);
}

template <int a>
__device__ __forceinline__ void face_block(const BoxJacArgs& A, const Hexes& H, int p, double M[3][3]) {
  constexpr int b = (a + 1) % 3, c = (a + 2) % 3;
  const int pc = p - H.s[c];
  const double w1 = H.w[path_of(a, b)][p], w2 = H.w[path_of(b, a)][p], w3 = H.w[path_of(c, a)][pc],
               w4 = H.w[path_of(c, b)][pc];
  const double ab = w1 + w3, ba = w2 + w4;
  M[a][a] = M[b][b] = M[c][c] = 0.0;
  M[a][b] = -A.h[a][b] * fma(A.lam, ab, A.mu * ba);
  M[b][a] = -A.h[a][b] * fma(A.lam, ba, A.mu * ab);
  M[a][c] = A.h[a][c] * fma(A.lam, w1, A.mu * w4);
  M[c][a] = A.h[a][c] * fma(A.lam, w4, A.mu * w1);
  M[b][c] = A.h[b][c] * fma(A.lam, w2, A.mu * w3);
  M[c][b] = A.h[b][c] * fma(A.lam, w3, A.mu * w2);
}

__device__ __forceinline__ void main_block(const BoxJacArgs& A, const Hexes& H, int p, double M[3][3]) {
#pragma unroll
  for (int a = 0; a < 3; ++a) {
    M[a][a] = 0.0;
#pragma unroll
    for (int c = 0; c < 3; ++c)
      if (c != a)  // first step a, last step c; and the reverse
        M[a][c] = -A.h[a][c] * fma(A.lam, H.w[path_of(a, 3 - a - c)][p], A.mu * H.w[path_of(c, 3 - a - c)][p]);
  }
}

// Weights of the tets that have the lower corner of hex p between an a and a b step.
template <int a>
__device__ __forceinline__ double between_sum(const Hexes& H, int p) {
  constexpr int b = (a + 1) % 3, c = (a + 2) % 3;
  return (H.w[path_of(a, b)][p - H.s[a]] + H.w[path_of(b, a)][p - H.s[b]]) +
         (H.w[path_of(c, a)][p - H.s[c] - H.s[a]] + H.w[path_of(c, b)][p - H.s[c] - H.s[b]]);
}

// Values of out before its first 128-byte line boundary (out: any 8-byte alignment).
__device__ __forceinline__ int to_line(const double* out) {
  return (int)((16u - (unsigned)(reinterpret_cast<size_t>(out) >> 3)) & 15u);
}

// Streams n staged values to out: single values to the first line boundary, then 16 bytes a
// thread, so that a wave's stores cover whole lines.  s + to_line(out) is 16-byte aligned.
__device__ __forceinline__ void stream_lines(const double* s, double* out, int n, int tid) {
  typedef double v2d __attribute__((ext_vector_type(2)));
  constexpr int kU = 4;  // pairs per thread read from LDS back to back, then stored
  const int head = min(n, to_line(out));
  if (tid < head) __builtin_nontemporal_store(s[tid], out + tid);
  for (int q0 = head + 2 * tid; q0 + 1 < n; q0 += 2 * kT * kU) {
    v2d v[kU];
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int q = q0 + 2 * kT * u;
      if (q + 1 < n) v[u] = *reinterpret_cast<const v2d*>(s + q);
    }
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      const int q = q0 + 2 * kT * u;
      if (q + 1 < n) __builtin_nontemporal_store(v[u], reinterpret_cast<v2d*>(out + q));
    }
  }
  if (((n - head) & 1) && tid == 0) __builtin_nontemporal_store(s[n - 1], out + n - 1);
}

// x + the value of the same lane of the wave's other half
__device__ __forceinline__ double sum_halves(double x) {
  const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(x), __double2loint(x), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(x), __double2hiint(x), false, false);
  return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

template <bool WITH_R, bool SIMP_INT>
__global__ __launch_bounds__(kT, 4) void k_box_jac_kuhn(BoxJacArgs A) {
  // the points' z and u and the hexes' weights, then (read into registers) the tile's values
  constexpr int kSeg = kJacRows * kJacMaxRow * 9;
  static_assert((WITH_R ? 4 : 1) * kJacPoints + 6 * kJacHexes <= kSeg, "one region");
  __shared__ __align__(16) double seg[kSeg + 1];
  double* zs = seg;
  double (*us)[kJacPoints] = reinterpret_cast<double (*)[kJacPoints]>(seg + kJacPoints);
  double (*w6)[kJacHexes] = reinterpret_cast<double (*)[kJacHexes]>(seg + (WITH_R ? 4 : 1) * kJacPoints);
  __shared__ double part[WITH_R ? 4 : 1][3][kJacRows];  // residual sums per wave
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // contiguous runs of tiles per XCD (work-group b runs on XCD b % 8)
  const int qd = A.ntiles / kNumXcd, rd = A.ntiles % kNumXcd, xc = blockIdx.x % kNumXcd;
  const int tile = xc * qd + min(xc, rd) + (int)blockIdx.x / kNumXcd;
  const JacTile T = A.tiles[tile];
  const int rows = T.dims & 255;
  struct {
    int x, y, z;
  } const B = {(int)(T.origin & 1023) - 1, (int)((T.origin >> 10) & 1023) - 1, (int)(T.origin >> 20) - 1};
  const int PX = (int)((T.dims >> 8) & 255) + 2, PY = (int)((T.dims >> 16) & 255) + 2, PZ = (int)(T.dims >> 24) + 2;
  const int HX = PX - 1, HY = PY - 1, npts = PX * PY * PZ, nhex = HX * HY * (PZ - 1);
  // t / d for t < 256, d < 256: the quotient is at least 1 / (2 d) from a whole number
  auto div = [](int a, int d) { return (int)(((float)a + 0.5f) * __builtin_amdgcn_rcpf((float)d)); };

  // the row of this lane (both halves of a wave hold the same 32 rows)
  const int r = lane & 31, half = lane >> 5, sg = half ? -1 : 1;
  const bool live = r < rows;
  const int row = T.row0 + min(r, rows - 1);
  const int g = A.gpack[row];
  const int sl = A.rowmap[row] - T.slot0;
  const unsigned long long pm = A.perm[row];
  const int kl = WITH_R ? A.lidx[row] : -1;
  if (t < npts) {
    const int line = div(t, PX), k = div(line, PY), i = B.x + t - line * PX, j = B.y + line - k * PY;
    const bool in = (unsigned)i < (unsigned)A.nx && (unsigned)j < (unsigned)A.ny && (unsigned)(B.z + k) < (unsigned)A.nz;
    double z = 0.0, u[3] = {0.0, 0.0, 0.0};
    if (in) {
      const int id = A.node_of[i + (size_t)A.nx * (j + (size_t)A.ny * (B.z + k))];
      z = A.z[id];
      if constexpr (WITH_R) {
#pragma unroll
        for (int c = 0; c < 3; ++c) u[c] = A.u[3 * (size_t)id + c];
      }
    }
    zs[t] = z;
    if constexpr (WITH_R) {
#pragma unroll
      for (int c = 0; c < 3; ++c) us[c][t] = u[c];
    }
  }
  lds_barrier();
  if (t < nhex) {
    const int line = div(t, HX), hk = div(line, HY), hi = t - line * HX, hj = line - hk * HY;
    const int i = B.x + hi, j = B.y + hj, kk = B.z + hk;
    double w[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (i >= 0 && j >= 0 && kk >= 0 && i < A.nx - 1 && j < A.ny - 1 && kk < A.nz - 1) {
      const int p = hi + PX * (hj + PY * hk);
      double zc[8];
#pragma unroll
      for (int c = 0; c < 8; ++c) zc[c] = zs[p + (c & 1) + PX * ((c >> 1) & 1) + PX * PY * (c >> 2)];
#pragma unroll
      for (int a = 0; a < 3; ++a)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          if (a == b) continue;
          const double rho = (zc[0] + zc[1 << a] + zc[(1 << a) | (1 << b)] + zc[7]) / 4.0;
          w[path_of(a, b)] = A.vol * (SIMP_INT ? fma(1.0 - A.m.rmin, simp_pow(rho, A.m.p, A.m.pint), A.m.rmin)
                                               : penalty_w(A.m, rho));
        }
    }
#pragma unroll
    for (int q = 0; q < 6; ++q) w6[q][t] = w[q];
  }
  lds_barrier();

  const int ri = g & 1023, rj = (g >> 10) & 1023, rk = g >> 20;
  const int li = ri - B.x, lj = rj - B.y, lk = rk - B.z;  // the row's point and hex in the tile
  const Hexes H{w6, {1, HX, HX * HY}};
  const int h0 = li + HX * (lj + HY * lk), p0 = li + PX * (lj + PY * lk);
  double Rr[3] = {0.0, 0.0, 0.0}, ur[3], f = 0.0;
  if constexpr (WITH_R) {
#pragma unroll
    for (int i = 0; i < 3; ++i) ur[i] = us[i][p0];
    if (kl >= 0 && wave < 3) f = A.load_f[3 * (size_t)kl + wave];
  }
  // Block towards row + d (first half) or row - d (second half).
  auto edge = [&](int dx, int dy, int dz, double M[3][3], auto block) {
    const int dh = dx + HX * (dy + HY * dz), dp = dx + PX * (dy + PY * dz);
    block(h0 - (half ? dh : 0), M);
#pragma unroll
    for (int i = 0; i < 3; ++i)
#pragma unroll
      for (int j = i + 1; j < 3; ++j) {
        const double x = M[i][j], y = M[j][i];
        M[i][j] = half ? y : x;
        M[j][i] = half ? x : y;
      }
    if constexpr (WITH_R) {
      double du[3];
#pragma unroll
      for (int i = 0; i < 3; ++i) du[i] = us[i][p0 + sg * dp] - ur[i];
#pragma unroll
      for (int i = 0; i < 3; ++i) Rr[i] = fma(M[i][0], du[0], fma(M[i][1], du[1], fma(M[i][2], du[2], Rr[i])));
    }
  };
  // Its place in the row: stencil lane l of +d, lane 13 - l of -d, where the offsets ascend in
  // dx + 3 dy + 9 dz and 7 to 13 are the positive ones.
  double* vals = A.vals + 9 * (size_t)T.slot0;
  double* stage = seg + (to_line(vals) & 1);
  auto place = [&](int l) { return stage + 9 * (sl + (int)((pm >> (4 * l)) & 15)); };
  auto put = [&](int l, int dx, int dy, int dz, const double M[3][3]) {
    if (live && (unsigned)(ri + sg * dx) < (unsigned)A.nx && (unsigned)(rj + sg * dy) < (unsigned)A.ny &&
        (unsigned)(rk + sg * dz) < (unsigned)A.nz) {
      double* d = place(half ? 13 - l : l);
#pragma unroll
      for (int i = 0; i < 3; ++i)
#pragma unroll
        for (int j = 0; j < 3; ++j) d[3 * i + j] = M[i][j];
    }
  };
  auto residual = [&]() {
    if constexpr (WITH_R) {
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        Rr[i] = sum_halves(Rr[i]);
        if (half == 0) part[wave][i][r] = Rr[i];
      }
    }
  };
  // axis edge, face diagonal and one off-diagonal pair of the diagonal block
  auto axis_work = [&](auto axis, int l, int lf) {
    constexpr int a = decltype(axis)::value, b = (a + 1) % 3;
    double M[3][3], F[3][3];
    edge(a == 0, a == 1, a == 2, M, [&](int p, double D[3][3]) { axis_block<a>(A, H, p, D); });
    edge(a == 0 || b == 0, a == 1 || b == 1, a == 2 || b == 2, F,
         [&](int p, double D[3][3]) { face_block<a>(A, H, p, D); });
    const double o = -(A.lam + A.mu) * A.h[a][b] * between_sum<a>(H, h0);
    residual();
    lds_barrier();  // all have read points and weights
    put(l, a == 0, a == 1, a == 2, M);
    put(lf, a == 0 || b == 0, a == 1 || b == 1, a == 2 || b == 2, F);
    if (live && half == 0) {
      double* d = place(kBoxDiagLane);
      d[3 * a + b] = d[3 * b + a] = o;
    }
  };
  if (wave == 0) {
    axis_work(std::integral_constant<int, 0>{}, 7, 9);
  } else if (wave == 1) {
    axis_work(std::integral_constant<int, 1>{}, 8, 12);
  } else if (wave == 2) {
    axis_work(std::integral_constant<int, 2>{}, 10, 11);
  } else {
    double M[3][3];
    edge(1, 1, 1, M, [&](int p, double D[3][3]) { main_block(A, H, p, D); });
    // the diagonal of the diagonal block from the sums of the six axis edges (three in each
    // half of the wave)
    const double e0 = axis_sum<0>(H, h0 - (half ? H.s[0] : 0)), e1 = axis_sum<1>(H, h0 - (half ? H.s[1] : 0)),
                 e2 = axis_sum<2>(H, h0 - (half ? H.s[2] : 0));
    const double s0 = A.h[0][0] * sum_halves(e0), s1 = A.h[1][1] * sum_halves(e1),
                 s2 = A.h[2][2] * sum_halves(e2);
    residual();
    lds_barrier();
    put(13, 1, 1, 1, M);
    if (live && half == 0) {
      double* d = place(kBoxDiagLane);
      const double tr = A.mu * (s0 + s1 + s2), lm = A.lam + A.mu;
      d[0] = fma(lm, s0, tr);
      d[4] = fma(lm, s1, tr);
      d[8] = fma(lm, s2, tr);
    }
  }
  const int end = A.rowmap[T.row0 + rows];
  lds_barrier();
  stream_lines(stage, vals, 9 * (end - T.slot0), t);
  if constexpr (WITH_R) {
    if (wave < 3 && half == 0 && live)
      A.R[3 * (size_t)(T.row0 + r) + wave] =
          ((part[0][wave][r] + part[1][wave][r]) + (part[2][wave][r] + part[3][wave][r])) - f;
  }
}

}  // namespace

std::vector<JacTile> box_jac_tiles(const std::vector<int32_t>& gpack, const int32_t* rowmap) {
  std::vector<JacTile> tiles;
  const int n = (int)gpack.size();
  for (int r = 0; r < n;) {
    int lo[3] = {1 << 20, 1 << 20, 1 << 20}, hi[3] = {-1, -1, -1}, rows = 0;
    for (; r + rows < n && rows < kJacRows; ++rows) {
      const int g = gpack[r + rows], p[3] = {g & 1023, (g >> 10) & 1023, g >> 20};
      int l[3], h[3], hexes = 1, points = 1;
      for (int k = 0; k < 3; ++k) {
        l[k] = std::min(lo[k], p[k]);
        h[k] = std::max(hi[k], p[k]);
        hexes *= h[k] - l[k] + 2;
        points *= h[k] - l[k] + 3;
        if (hexes > kJacHexes || points > kJacPoints) break;  // (and no overflow)
      }
      if (hexes > kJacHexes || points > kJacPoints) break;
      std::copy(l, l + 3, lo);
      std::copy(h, h + 3, hi);
    }
    JacTile t;
    t.row0 = r;
    t.dims = (uint32_t)rows | (uint32_t)(hi[0] - lo[0] + 1) << 8 | (uint32_t)(hi[1] - lo[1] + 1) << 16 |
             (uint32_t)(hi[2] - lo[2] + 1) << 24;
    t.origin = (uint32_t)lo[0] | (uint32_t)lo[1] << 10 | (uint32_t)lo[2] << 20;
    t.slot0 = rowmap[r];
    tiles.push_back(t);
    r += rows;
  }
  return tiles;
}

hipError_t launch_box_jac_kuhn(const BoxJacArgs& a, hipStream_t s) {
  const bool ip = a.m.model == kPenaltySimp && a.m.pint > 0;
  if (a.R) {
    if (ip) k_box_jac_kuhn<true, true><<<a.ntiles, kT, 0, s>>>(a);
    else k_box_jac_kuhn<true, false><<<a.ntiles, kT, 0, s>>>(a);
  } else {
    if (ip) k_box_jac_kuhn<false, true><<<a.ntiles, kT, 0, s>>>(a);
    else k_box_jac_kuhn<false, false><<<a.ntiles, kT, 0, s>>>(a);
  }
  return hipGetLastError();
}

}  // namespace pa
