// Jacobian (and residual) assembly of uniform Kuhn-split box lattices by tiles of
// consecutive rows, without lattice copies of z and u or an array of element weights.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "pa_kernels.hpp"

namespace pa {

constexpr int kJacRows = 32;      // rows of a tile
constexpr int kJacMaxRow = 15;    // blocks of a row: 14 neighbours and the diagonal
constexpr int kJacHexes = 160;    // hexes around a tile (of its bounding box)
constexpr int kJacPoints = 256;   // lattice points of those hexes
// Rows a tile must hold on average, unless one round of work-groups takes them all: with
// 128x64x64 hexes numbered in shuffled runs of 24 / 16 / 12 / 8 nodes this kernel takes 145 /
// 190 / 232 / 307 us and the general lattice kernels 192 / 195 / 200 / 200; with 20x10x10 it
// is the faster one for every numbering (12.6 to 16.3 against 18.5 to 21.3 us).
constexpr int kJacMinRows = 16, kJacRound = 1024;

// A run of consecutive rows whose lattice points fill a small box: row0, then the count and
// the box's points per axis (8 bits each), its lowest point (10 bits per axis), and the
// first CRS slot.
struct JacTile {
  int row0;
  uint32_t dims;    // rows | bx << 8 | by << 16 | bz << 24
  uint32_t origin;  // ox | oy << 10 | oz << 20
  int slot0;
};

struct BoxJacArgs {
  const JacTile* tiles;
  int ntiles;
  const int* node_of;              // node at lattice point (i, j, k): i + nx (j + ny k)
  const int* rowmap;
  const int* gpack;                // per node: i | j << 10 | k << 20
  const unsigned long long* perm;  // per row: CRS slot of stencil lane l in bits 4l..4l+3
  const double* z;
  const double* u;                 // null without a residual
  const int* lidx;                 // per node: its entry in load_f, or -1
  const double* load_f;
  double* vals;
  double* R;
  int nx, ny, nz;                  // points per axis
  double vol;                      // of a tet
  double lam, mu;
  double h[3][3];                  // 1 / (spacing_i spacing_j)
  Material m;
};

// Tiles of the rows in node order (gpack: lattice point per node): as many consecutive rows
// as keep the box within the limits above.
std::vector<JacTile> box_jac_tiles(const std::vector<int32_t>& gpack, const int32_t* rowmap);

// K values of every row, and R = K u - f when a.R.
hipError_t launch_box_jac_kuhn(const BoxJacArgs& a, hipStream_t s);

}  // namespace pa
