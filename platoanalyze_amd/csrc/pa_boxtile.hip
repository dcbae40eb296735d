// Brick kernels of Kuhn-split box lattices (pa_boxtile.hpp).
//
// A work-group owns a 4x4x4 brick of lattice points.  It gathers u and z of the 6x6x6
// points around it once (through the lattice-to-node map: no lattice copies of u and z and
// no array of element weights), a thread computes all six tets of one of the 5x5x5 hexes
// that touch the brick from its eight corners in registers, leaves the hex's eight corner
// contributions in LDS, and the brick's points sum theirs from eight hexes in a fixed order.
// A tet is evaluated 125 / 64 = 1.95 times on average; one row per lane from its 24 tets
// evaluates it four times, reads 15 points and 24 weights a row, and needs a scatter pass
// and a weight pass before it.  In the tet of axis path (a, b, c) the displacement
// gradient's columns are the three edge differences over the spacings.
//
// What bounds it: FP64 arithmetic and the latency of the two dependent gathers (map, then
// u and z) at twelve waves a CU: registers, as LDS holds the corner contributions of half the
// corners at a time.  128x64x64 hexes, one thread per row with lattice copies and a weight
// array -> bricks with all corners and every penalty model's code -> this: residual 62 -> 48.5
// -> 36 us a call, energy and gradient (chunk kernel) 149 -> 60 -> 49; p-norm adjoint
// gradient, 64x32x32, 182 -> 124 -> 104 (89 to 92 since its factor is summed on the device).
// Four waves a SIMD spill (residual 51 us, gradient 109).
// kTileResidualW reads the tets' weights instead, where a power or a sine each would be
// evaluated 1.95 times (128x64x64, Heaviside: 93 us with the pass that makes them, 119 without).
#include "pa_boxtile.hpp"

#include <cmath>
#include <type_traits>

#include "pa_box.hpp"
#include "pa_reduce.hpp"

namespace pa {

namespace {

constexpr int kT = 128;                            // threads; 125 of them have a hex
constexpr int kOwn = kTileNodes, kHex = kOwn + 1, kPts = kOwn + 2;
constexpr int kHexes = kHex * kHex * kHex, kPoints = kPts * kPts * kPts;
static_assert(kHexes <= kT, "a thread per hex");

// Value i (of three) of a staged vector at corner c of a hex, at compile-time offsets from
// its lower corner's address.  The points stay in LDS, so that the compiler may read a value
// again instead of holding all corners' 24 a vector through the six tets.
struct Corners {
  const double* p;
  __device__ __forceinline__ double operator()(int c, int i) const {
    return p[i * kPoints + (c & 1) + kPts * ((c >> 1) & 1) + kPts * kPts * (c >> 2)];
  }
};

// Voigt strain (engineering shear) of tet Q of the hex with corner displacements U
template <int Q>
__device__ __forceinline__ void tet_strain_of(const Corners& U, const double ih[3], double e[6]) {
  constexpr int a = kKuhnPath[Q][0], b = kKuhnPath[Q][1], c = kKuhnPath[Q][2];
  constexpr int v1 = 1 << a, v2 = (1 << a) | (1 << b);
  double G[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const double u1 = U(v1, i), u2 = U(v2, i);
    G[i][a] = (u1 - U(0, i)) * ih[a];
    G[i][b] = (u2 - u1) * ih[b];
    G[i][c] = (U(7, i) - u2) * ih[c];
  }
  e[0] = G[0][0];
  e[1] = G[1][1];
  e[2] = G[2][2];
  e[3] = G[1][2] + G[2][1];
  e[4] = G[0][2] + G[2][0];
  e[5] = G[0][1] + G[1][0];
}

__device__ __forceinline__ void stress_of(const Material& m, const double e[6], double s[6]) {
  const double l = m.c01 * (e[0] + e[1] + e[2]), d = m.c00 - m.c01;
#pragma unroll
  for (int k = 0; k < 3; ++k) s[k] = fma(d, e[k], l);
#pragma unroll
  for (int k = 3; k < 6; ++k) s[k] = m.c33 * e[k];
}

template <int Q>
__device__ __forceinline__ double tet_rho(const double Z[8]) {
  constexpr int v1 = 1 << kKuhnPath[Q][0], v2 = v1 | (1 << kKuhnPath[Q][1]);
  return (Z[0] + Z[v1] + Z[v2] + Z[7]) / 4.0;
}

// F[corner] += force of the stress k * s on the tet's vertices: edge l along axis c adds
// k s[:, c] / h_c to its upper vertex and subtracts it from its lower one
template <int Q>
__device__ __forceinline__ void tet_force(const double s[6], double k, const double ih[3], double F[8][3]) {
  constexpr int V[3][3] = {{0, 5, 4}, {5, 1, 3}, {4, 3, 2}};  // Voigt index of (i, j)
  constexpr int a = kKuhnPath[Q][0], b = kKuhnPath[Q][1];
  constexpr int v[4] = {0, 1 << a, (1 << a) | (1 << b), 7};
#pragma unroll
  for (int l = 0; l < 3; ++l) {
    const int c = kKuhnPath[Q][l];
    const double kh = k * ih[c];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const double t = kh * s[V[i][c]];
      F[v[l + 1]][i] += t;
      F[v[l]][i] -= t;
    }
  }
}

template <int Q>
__device__ __forceinline__ void tet_scalar(double k, double F[8]) {
  constexpr int v1 = 1 << kKuhnPath[Q][0], v2 = v1 | (1 << kKuhnPath[Q][1]);
  F[0] += k;
  F[v1] += k;
  F[v2] += k;
  F[7] += k;
}

template <int N, typename F>
__device__ __forceinline__ void each_tet(const F& f) {
  if constexpr (N < 6) {
    f(std::integral_constant<int, N>{});
    each_tet<N + 1>(f);
  }
}

// von Mises direction t = dJ/dsigma and J = vm^2
__device__ __forceinline__ double von_mises2(const double s[6]) {
  const double d01 = s[0] - s[1], d12 = s[1] - s[2], d20 = s[2] - s[0];
  return 0.5 * (d01 * d01 + d12 * d12 + d20 * d20) + 3.0 * (s[3] * s[3] + s[4] * s[4] + s[5] * s[5]);
}

template <int MODE, bool SIMP>  // SIMP: powers by multiplication only (see launch_box_tile)
__global__ __launch_bounds__(kT, 3) void k_box_tile(BoxTileArgs A) {
  constexpr bool kWgt = MODE == kTileResidualW;  // the tets' weights are given
  constexpr bool kRes = MODE == kTileResidual || kWgt, kGradZ = MODE == kTileEnergyGradZ, kPnG = MODE == kTilePNormGrad;
  constexpr bool kAdj = MODE == kTileAdjZ, kPn = MODE == kTilePNorm || kPnG;
  constexpr bool kVec = kRes || kPnG, kScal = kGradZ || kPnG || kAdj;  // corner vectors, corner scalars
  constexpr bool kSum = MODE == kTileEnergy || kGradZ || MODE == kTilePNorm;
  constexpr int kOut = (kVec ? 3 : 0) + (kScal ? 1 : 0);
  // the points' u and z (and u2), and the contributions of four of a hex's corners at a time
  __shared__ double sm[kPoints * (kAdj ? 7 : 4)], sc[kOut > 0 ? 4 * kOut * kT : 1];
  // per hex and tet, where the penalty model's code shall exist once (a rolled loop): density
  // and strain measure, then coefficients
  __shared__ double cl[SIMP ? 1 : 6][SIMP ? 1 : kT], rl[SIMP ? 1 : 6][SIMP ? 1 : kT];
  __shared__ int ids[kPoints];
  __shared__ double sh[kT / 64];

  const int t = threadIdx.x;
  // contiguous runs of bricks per XCD (work-group b runs on XCD b % 8)
  const int nb = A.bx * A.by * A.bz, qd = nb / kNumXcd, rd = nb % kNumXcd, xc = blockIdx.x % kNumXcd;
  const int brick = xc * qd + min(xc, rd) + (int)blockIdx.x / kNumXcd;
  const int i0 = brick % A.bx * kOwn, j0 = brick / A.bx % A.by * kOwn, k0 = brick / (A.bx * A.by) * kOwn;
  for (int p = t; p < kPoints; p += kT) {
    const int i = i0 - 1 + p % kPts, j = j0 - 1 + p / kPts % kPts, k = k0 - 1 + p / (kPts * kPts);
    const bool in = (unsigned)i < (unsigned)A.nx && (unsigned)j < (unsigned)A.ny && (unsigned)k < (unsigned)A.nz;
    const int id = in ? A.node_of[i + (size_t)A.nx * (j + (size_t)A.ny * k)] : -1;
    ids[p] = id;
    if (id >= 0) {
#pragma unroll
      for (int c = 0; c < 3; ++c) sm[c * kPoints + p] = A.u[3 * (size_t)id + c];
      sm[3 * kPoints + p] = A.z[id];
      if constexpr (kAdj) {
#pragma unroll
        for (int c = 0; c < 3; ++c) sm[(4 + c) * kPoints + p] = A.u2[3 * (size_t)id + c];
      }
    }
  }
  __syncthreads();
  // hex t: lower corner at lattice point (i0 - 1 + hx, ...)
  const int hx = t % kHex, hy = t / kHex % kHex, hz = t / (kHex * kHex);
  const int gi = i0 - 1 + hx, gj = j0 - 1 + hy, gk = k0 - 1 + hz;
  const bool hex = t < kHexes && gi >= 0 && gj >= 0 && gk >= 0 && gi < A.nx - 1 && gj < A.ny - 1 && gk < A.nz - 1;
  const int at = hx + kPts * (hy + kPts * hz);
  const Corners U{sm + at}, L{sm + 4 * kPoints + at};
  double Z[8];
  if (hex) {
#pragma unroll
    for (int c = 0; c < 8; ++c) Z[c] = U(c, 3);
  }
  double sum = 0.0, F[8][3], S[8];
#pragma unroll
  for (int c = 0; c < 8; ++c) {
#pragma unroll
    for (int i = 0; i < 3; ++i) F[c][i] = 0.0;
    S[c] = 0.0;
  }
  if (hex) {
    const double ih[3] = {A.ih[0], A.ih[1], A.ih[2]};
    const int pni = SIMP ? (int)A.pn : (A.pn <= 16.0 && A.pn == floor(A.pn)) ? (int)A.pn : 0;
    // strain measure of a tet that its coefficients need
    auto measure = [&](auto q) {
      constexpr int Q = decltype(q)::value;
      double e[6], s[6], v = 0.0;
      if constexpr (!kRes) {
        tet_strain_of<Q>(U, ih, e);
        stress_of(A.m, e, s);
        if constexpr (kPn) {
          if (A.measure == 0) {
#pragma unroll
            for (int k = 0; k < 6; ++k) v += s[k] * s[k];
          } else {
            v = von_mises2(s);
          }
        } else if constexpr (kAdj) {
          double l[6];
          tet_strain_of<Q>(L, ih, l);
#pragma unroll
          for (int k = 0; k < 6; ++k) v += s[k] * l[k];
        } else {
#pragma unroll
          for (int k = 0; k < 6; ++k) v += s[k] * e[k];
        }
      }
      return v;
    };
    // its coefficients: cf of the corner vectors, cs of the corner scalars (kWgt: rho is the weight)
    auto coefficients = [&](double rho, double v, double& cf, double& cs) {
      cf = cs = 0.0;
      if constexpr (kWgt) {
        cf = A.vol * rho;
      } else if constexpr (kRes) {
        cf = A.vol * penalty_w_as<SIMP>(A.m, rho);
      } else if constexpr (kAdj) {
        cs = v * (0.25 * penalty_dw_as<SIMP>(A.m, rho) * A.vol);
      } else if constexpr (!kPn) {
        sum += 0.5 * A.vol * penalty_w_as<SIMP>(A.m, rho) * v;
        if constexpr (kGradZ) cs = A.scale * (0.125 * A.vol * v * penalty_dw_as<SIMP>(A.m, rho));
      } else {
        // m, with dm/du = c_u B^T C0 t and dm/drho = c_z m (t: see the forces below)
        double mval, cu, cz;
        if (A.measure == 0) {
          const double w = penalty_w_as<SIMP>(A.m, rho);
          mval = fabs(w) * sqrt(v);
          cu = mval > 0.0 ? w * w / mval : 0.0;
          cz = kPnG ? penalty_dw_as<SIMP>(A.m, rho) / w : 0.0;
        } else {
          const double vm0 = sqrt(v), rq = SIMP ? sqrt(rho) : pow_of(rho, A.q, 0);
          mval = rq * vm0;
          cu = vm0 > 0.0 ? rq / (2.0 * vm0) : 0.0;
          cz = kPnG ? A.q / rho : 0.0;
        }
        const double mp = SIMP ? powi(mval, pni) : pow_of(mval, A.pn, pni);
        sum += mp * A.vol;
        if constexpr (kPnG) {
          const double k = *A.pscale * A.vol * A.pn;
          cf = k * (mval > 0.0 ? mp / mval : 0.0) * cu;
          cs = 0.25 * k * mp * cz;
        }
      }
    };
    auto forces = [&](auto q, double cf, double cs) {
      constexpr int Q = decltype(q)::value;
      if constexpr (kVec) {
        double e[6], s[6];
        tet_strain_of<Q>(U, ih, e);
        stress_of(A.m, e, s);
        if constexpr (kPnG) {
          if (A.measure != 0) {  // t = dJ/dsigma; measure 0: t = sigma
            const double tr = s[0] + s[1] + s[2];
#pragma unroll
            for (int k = 0; k < 3; ++k) s[k] = 3.0 * s[k] - tr;
#pragma unroll
            for (int k = 3; k < 6; ++k) s[k] *= 6.0;
          }
          double tau[6];
          stress_of(A.m, s, tau);
          tet_force<Q>(tau, cf, ih, F);
        } else {
          tet_force<Q>(s, cf, ih, F);
        }
      }
      if constexpr (kScal) tet_scalar<Q>(cs, S);
    };
    if constexpr (SIMP) {
      const double* W = kWgt ? A.W + 6 * (gi + 1 + (A.nx + 1) * (gj + 1 + (size_t)(A.ny + 1) * (gk + 1))) : nullptr;
      each_tet<0>([&](auto q) {
        constexpr int Q = decltype(q)::value;
        double cf, cs, rho;
        if constexpr (kWgt) rho = W[A.tperm[Q]];
        else rho = tet_rho<Q>(Z);
        coefficients(rho, measure(q), cf, cs);
        forces(q, cf, cs);
      });
    } else {
      each_tet<0>([&](auto q) {
        constexpr int Q = decltype(q)::value;
        rl[Q][t] = tet_rho<Q>(Z);
        cl[Q][t] = measure(q);
      });
#pragma unroll 1
      for (int q = 0; q < 6; ++q) {
        double cf, cs;
        coefficients(rl[q][t], cl[q][t], cf, cs);
        cl[q][t] = cf;
        rl[q][t] = cs;
      }
      if constexpr (kOut > 0)
        each_tet<0>([&](auto q) {
          constexpr int Q = decltype(q)::value;
          forces(q, cl[Q][t], rl[Q][t]);
        });
    }
  }
  if constexpr (kOut > 0) {
    constexpr int kNodes = kOwn * kOwn * kOwn, kItems = (kOut * kNodes + kT - 1) / kT;
    double v[kItems];
#pragma unroll
    for (int i = 0; i < kItems; ++i) v[i] = 0.0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // the hexes' lower, then upper corners
      if (h) __syncthreads();      // the lower ones have been read
      if (t < kHexes) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          if constexpr (kVec) {
#pragma unroll
            for (int i = 0; i < 3; ++i) sc[(kOut * c + i) * kT + t] = F[4 * h + c][i];
          }
          if constexpr (kScal) sc[(kOut * c + kOut - 1) * kT + t] = S[4 * h + c];
        }
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < kItems; ++i) {
        const int w = t + i * kT;
        if (w >= kOut * kNodes) break;
        const int n = w / kOut, o = w - kOut * n;
        const int a = n % kOwn, b = n / kOwn % kOwn, c = n / (kOwn * kOwn);
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {  // the node is corner cc + 4 h of hex (a + 1 - bits)
          const int hh = (a + 1 - (cc & 1)) + kHex * ((b + 1 - (cc >> 1)) + kHex * (c + 1 - h));
          v[i] += sc[(kOut * cc + o) * kT + hh];
        }
      }
    }
#pragma unroll
    for (int i = 0; i < kItems; ++i) {
      const int w = t + i * kT;
      if (w >= kOut * kNodes) break;
      const int n = w / kOut, o = w - kOut * n;
      const int a = n % kOwn, b = n / kOwn % kOwn, c = n / (kOwn * kOwn);
      const int id = ids[(a + 1) + kPts * ((b + 1) + kPts * (c + 1))];
      if (id < 0) continue;
      if constexpr (kRes) {
        const int k = A.lidx ? A.lidx[id] : -1;
        A.out[3 * (size_t)id + o] = v[i] - (k >= 0 ? A.load_f[3 * (size_t)k + o] : 0.0);
      } else if constexpr (kPnG) {
        if (o < 3) A.out[3 * (size_t)id + o] = v[i];
        else A.out2[id] = v[i];
      } else {
        A.out[id] = v[i];
      }
    }
  }
  if constexpr (kSum) {  // every hex is summed by the brick that owns its lower corner
    const double own = hex && hx > 0 && hy > 0 && hz > 0 ? sum : 0.0;
    const double r = block_reduce_all<kT>(own, sh);
    if (t == 0 && A.partials) A.partials[brick] = r;
  }
}

}  // namespace

template <int MODE>
static void launch(bool simp, const BoxTileArgs& a, hipStream_t s) {
  const int grid = a.bx * a.by * a.bz;
  if (simp) k_box_tile<MODE, true><<<grid, kT, 0, s>>>(a);
  else k_box_tile<MODE, false><<<grid, kT, 0, s>>>(a);
}

hipError_t launch_box_tile(int mode, const BoxTileArgs& a, hipStream_t s) {
  // integer SIMP exponents; in the p-norms also an integer p and, for the relaxed von Mises
  // measure, q = 1/2
  bool simp = a.m.model == kPenaltySimp && a.m.pint > 0;
  if (mode == kTilePNorm || mode == kTilePNormGrad)
    simp = simp && a.pn >= 1.0 && a.pn <= 16.0 && a.pn == std::floor(a.pn) && (a.measure == 0 || a.q == 0.5);
  switch (mode) {
    case kTileResidual: launch<kTileResidual>(simp, a, s); break;
    case kTileResidualW: k_box_tile<kTileResidualW, true><<<a.bx * a.by * a.bz, kT, 0, s>>>(a); break;
    case kTileEnergy: launch<kTileEnergy>(simp, a, s); break;
    case kTileEnergyGradZ: launch<kTileEnergyGradZ>(simp, a, s); break;
    case kTilePNorm: launch<kTilePNorm>(simp, a, s); break;
    case kTilePNormGrad: launch<kTilePNormGrad>(simp, a, s); break;
    case kTileAdjZ: launch<kTileAdjZ>(simp, a, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace pa
