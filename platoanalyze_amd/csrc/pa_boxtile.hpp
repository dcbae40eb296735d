// Element kernels of uniform Kuhn-split box lattices by bricks of nodes: residual, energy
// and its density gradient, stress p-norm and its partials, (dR/dz)^T lambda.
#pragma once
#include <hip/hip_runtime.h>

#include "pa_kernels.hpp"

namespace pa {

struct BoxTileArgs {
  const int* node_of;   // node at lattice point (i, j, k): i + nx (j + ny k)
  int nx, ny, nz;       // nodes per axis
  int bx, by, bz;       // bricks per axis
  double ih[3], vol;    // 1 / spacing per axis, tet volume
  const double* u;      // node order
  const double* u2;     // second state (lambda) of kTileAdjZ
  const double* z;
  double* out;          // 3 per node (residual, p-norm dF/du) or 1 (energy gradient, adjoint)
  double* out2;         // 1 per node (p-norm dF/dz)
  double* partials;     // one per brick: energy or p-norm sum (null: none)
  const int* lidx;      // per node: its entry in load_f, or -1 (kTileResidual; null: no load)
  const double* load_f;
  const double* W;      // kTileResidualW: weights of the padded hexes, six a hex, path q's at tperm[q]
  int tperm[6];
  double scale;         // factor of the energy gradient (1, or -1 for the total derivative)
  int measure;          // p-norm: 0 Voigt norm of the weighted stress, 1 relaxed von Mises
  double pn, q;
  const double* pscale;  // factor of the p-norm gradients, on the device
  Material m;
};

enum TileMode { kTileResidual = 0, kTileEnergy = 1, kTileEnergyGradZ = 2, kTilePNorm = 3, kTilePNormGrad = 4,
                kTileAdjZ = 5, kTileResidualW = 6 };

constexpr int kTileNodes = 4;  // a brick owns kTileNodes^3 lattice points
inline int tile_bricks(int nodes) { return (nodes + kTileNodes - 1) / kTileNodes; }

hipError_t launch_box_tile(int mode, const BoxTileArgs& a, hipStream_t s);

}  // namespace pa
