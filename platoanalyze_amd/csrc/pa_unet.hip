// U-Net kernels: implicit-GEMM 3x3x3 convolutions on v_mfma_f32_16x16x32_bf16, weight
// gradients, packing, Adam and the loss.
//
// MFMA 16x16x32 (bf16 in, fp32 accumulate) operand layout, lane l of 64:
//   A (16 x 32): row l % 16, k = 8 (l / 16) .. 8 (l / 16) + 7
//   B (32 x 16): column l % 16, same k range
//   C (16 x 16): column l % 16, rows 4 (l / 16) .. 4 (l / 16) + 3
#include "pa_unet.hpp"

#include <atomic>
#include <type_traits>

#include "pa_reduce.hpp"

namespace pa {
namespace unet {

namespace {

typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kT = 256;
constexpr int kConvFillWaves = 2048;  // eight waves per CU of a 256-CU part
constexpr int kConvMaxSlices = 32;

__device__ __forceinline__ bf16_t f2bf(float f) {  // round to nearest even
  const uint32_t u = __float_as_uint(f);
  if ((u & 0x7F800000u) == 0x7F800000u) return (bf16_t)(u >> 16);  // inf / nan
  return (bf16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
__device__ __forceinline__ float bf2f(bf16_t b) { return __uint_as_float((uint32_t)b << 16); }
__device__ __forceinline__ bool bf_pos(bf16_t b) { return !(b & 0x8000u) && (b & 0x7FFFu); }

// Input voxel linked to output voxel (ox, oy, oz) by tap (dx, dy, dz); false when the
// link falls outside the input grid (zero padding) or off the stride lattice.
__device__ __forceinline__ bool link(const Grid& gi, int s, int transposed, int ox, int oy, int oz, int dx, int dy,
                                     int dz, int& vi) {
  int ix, iy, iz;
  if (!transposed) {
    ix = s * ox + dx - 1;
    iy = s * oy + dy - 1;
    iz = s * oz + dz - 1;
  } else {
    ix = ox + 1 - dx;
    iy = oy + 1 - dy;
    iz = oz + 1 - dz;
    if (ix < 0 || iy < 0 || iz < 0) return false;
    if (s == 2) {
      if ((ix | iy | iz) & 1) return false;
      ix >>= 1;
      iy >>= 1;
      iz >>= 1;
    }
  }
  if (ix < 0 || iy < 0 || iz < 0 || ix >= gi.nx || iy >= gi.ny || iz >= gi.nz) return false;
  vi = (ix * gi.ny + iy) * gi.nz + iz;
  return true;
}

__device__ __forceinline__ void decode(const Grid& g, int o, int& x, int& y, int& z) {
  z = o % g.nz;
  const int r = o / g.nz;
  y = r % g.ny;
  x = r / g.ny;
}

// Bias, ReLU, gate and the stores of output element (m, n) with the reduction sum v.
__device__ __forceinline__ void conv_epilogue(const ConvArgs& A, int m, int n, float v) {
  if (A.bias) v += A.bias[n];
  if (A.relu) v = fmaxf(v, 0.0f);
  if (A.gate && !bf_pos(A.gate[(size_t)m * A.ldg + A.gcol + n])) v = 0.0f;
  if (A.Y) A.Y[(size_t)m * A.ldy + A.ycol + n] = f2bf(v);
  if (A.Yf) {
    float* d = A.Yf + (size_t)m * A.ldyf + A.yfcol + n;
    *d = A.accumulate ? *d + v : v;
  }
}

// One work-group = 4 wavefronts; a wavefront computes 16 output voxels x 64 channels over
// K steps [blockIdx.z * kper, (blockIdx.z + 1) * kper) of 32 (SPLIT: raw sums into the
// slice's part array; else the whole reduction and the epilogue).
template <bool XF32, bool SPLIT>
__global__ __launch_bounds__(kT) void k_conv(ConvArgs A, int kper) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int Vo = A.go.count(), Vi = A.gi.count();
  const int Mtot = A.batch * Vo;
  const int m0 = (blockIdx.x * 4 + wave) * 16;
  const int n0 = blockIdx.y * 64;
  const int Ktot = 27 * A.cin;
  const int kbeg = SPLIT ? (int)blockIdx.z * kper * 32 : 0;
  const int kend = SPLIT ? min(Ktot, kbeg + kper * 32) : Ktot;
  const int mrow = m0 + (lane & 15);
  const bool mvalid = mrow < Mtot;
  int b = 0, ox = 0, oy = 0, oz = 0;
  if (mvalid) {
    b = mrow / Vo;
    decode(A.go, mrow - b * Vo, ox, oy, oz);
  }
  const size_t xbase = (size_t)b * Vi;
  f32x4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // this lane's k offset inside a 32-wide K step, tracked as (tap, channel)
  const int kq = 8 * (lane >> 4);
  int t = (kbeg + kq) / A.cin, ch = (kbeg + kq) - ((kbeg + kq) / A.cin) * A.cin;
  for (int kc = kbeg; kc < kend; kc += 32) {
    const int k0 = kc + kq;
    bf16x8 a = {0, 0, 0, 0, 0, 0, 0, 0};
    if (mvalid && k0 < Ktot) {
      int vi;
      if (link(A.gi, A.stride, A.transposed, ox, oy, oz, t / 9, (t / 3) % 3, t % 3, vi)) {
        const size_t off = (xbase + vi) * (size_t)A.ldx + A.xcol + ch;
        if constexpr (XF32) {
          const float4 p = *reinterpret_cast<const float4*>(A.Xf + off);
          const float4 q = *reinterpret_cast<const float4*>(A.Xf + off + 4);
          a = bf16x8{(short)f2bf(p.x), (short)f2bf(p.y), (short)f2bf(p.z), (short)f2bf(p.w),
                     (short)f2bf(q.x), (short)f2bf(q.y), (short)f2bf(q.z), (short)f2bf(q.w)};
        } else {
          a = *reinterpret_cast<const bf16x8*>(A.X + off);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + 16 * j + (lane & 15);
      bf16x8 bv = {0, 0, 0, 0, 0, 0, 0, 0};
      if (n < A.cout && k0 < Ktot) bv = *reinterpret_cast<const bf16x8*>(A.Bt + (size_t)n * A.ldb + k0);
      acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bv, acc[j], 0, 0, 0);
    }
    ch += 32;
    while (ch >= A.cin) {
      ch -= A.cin;
      ++t;
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + 16 * j + (lane & 15);
    if (n >= A.cout) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + 4 * (lane >> 4) + i;
      if (m >= Mtot) continue;
      if constexpr (SPLIT) A.part[((size_t)blockIdx.z * Mtot + m) * A.cout + n] = acc[j][i];
      else conv_epilogue(A, m, n, acc[j][i]);
    }
  }
}

// Sum of the slices of a split reduction, in slice order, and the epilogue.
__global__ __launch_bounds__(kT) void k_conv_reduce(ConvArgs A, int nslices) {
  const size_t Mtot = (size_t)A.batch * A.go.count(), total = Mtot * A.cout;
  for (size_t e = blockIdx.x * (size_t)kT + threadIdx.x; e < total; e += (size_t)gridDim.x * kT) {
    float v = A.part[e];
    for (int z = 1; z < nslices; ++z) v += A.part[(size_t)z * total + e];
    conv_epilogue(A, (int)(e / A.cout), (int)(e % A.cout), v);
  }
}

// Convolution with the input staged in LDS (every layer whose tile fits; k_conv above
// serves the others).
//
// A work-group takes the output voxels of a run of y lines and z at one x, stages the input
// lines their taps reach once as rows of channels in BF16 (FP32 gradients converted here and
// not at each of 27 uses), and computes tiles of 16 voxels x 16 channels, up to kConvM a
// wave, with the weights of the next kConvAhead steps on their way from L2.
// A staged row is an odd number of 16-byte banks long, so the 16 rows of an operand read
// spread over them and its address is one addition.  The weights are the MFMA's row operand:
// a lane then holds four consecutive channels of one voxel and the epilogue moves 8 or 16
// bytes a lane.
// Transposed stride-2 links reach 1, 2, 4 or 8 of the 27 taps by the voxel's parities:
// voxels are grouped by parity and the steps without a linked tap skipped.
// The sums are those of k_conv to the bit: the same K steps in the same order (a skipped
// step would have added zeros), the same slices of a split reduction, added in slice order;
// eight waves share the slices and exchange them through LDS instead of a workspace and a
// second kernel.
//
// 65x33x33, base 16, against k_conv for all layers: the forward call at batch 1 271 ->
// 174 us, the 29 convolutions of a gradient at batch 4 1280 -> 644 us.  What is left is
// latency: a launch has about one round of work-groups, each with its staging loads, a
// barrier and a serial chain of at most 27 cin / 32 K steps.
constexpr int kConvM = 4, kConvAhead = 4;
constexpr size_t kConvLdsGoal = 80 * 1024, kConvLdsMax = 120 * 1024;
constexpr int kConvGroups = 512;  // work-groups a launch should keep: two per CU

struct ConvTile {
  int kind;                      // 0 direct, 1 transposed stride 1, 2 transposed stride 2
  int ty, tz, nty, ntz;          // output lines and z per tile, tiles per axis
  int mt;                        // split: 16-voxel tiles of a work-group
  int planes, lq, qz;            // staged planes, lines, z
  int nch, row;                  // 8-channel chunks, bytes of a staged row
  int ksteps, kper, nsl;         // K steps of 32, per slice, slices
  int nty_n;                     // runs of NT channel tiles per work-group
  int tzc;                       // z of a parity class (kind 2; else of the tile)
  // staging strides of a thread's next chunk: rows, and those as planes, lines and z
  int nthr, srow, sd, sl, sz;
  unsigned div_nch, div_lq, div_qz, div_tzc;  // small_div factors
};

// a / d for a, d < 2^16 by the host's factor floor(2^32 / d) + 1 (0 for d = 1)
__device__ __forceinline__ int small_div(int a, unsigned f) { return f ? (int)__umulhi((unsigned)a, f) : a; }
inline unsigned small_div_factor(int d) { return d == 1 ? 0u : (unsigned)((1ull << 32) / d) + 1u; }

// Eight floats to BF16, nearest even (v_cvt_pk_bf16_f32; f2bf costs seven operations each).
__device__ __forceinline__ bf16x8 cvt_bf16x8(const float4& p, const float4& q) {
  typedef __bf16 b8 __attribute__((ext_vector_type(8)));
  typedef float f8 __attribute__((ext_vector_type(8)));
  const b8 r = __builtin_convertvector(f8{p.x, p.y, p.z, p.w, q.x, q.y, q.z, q.w}, b8);
  return __builtin_bit_cast(bf16x8, r);
}

// Epilogue of channels n .. n + 3 of output voxel m.
__device__ __forceinline__ void conv_epilogue4(const ConvArgs& A, size_t m, int n, f32x4 v) {
  if (A.bias) {
    const float4 b = *reinterpret_cast<const float4*>(A.bias + n);
    v[0] += b.x;
    v[1] += b.y;
    v[2] += b.z;
    v[3] += b.w;
  }
  if (A.relu) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = fmaxf(v[i], 0.0f);
  }
  if (A.gate) {
    const ushort4 g = *reinterpret_cast<const ushort4*>(A.gate + m * A.ldg + A.gcol + n);
    if (!bf_pos(g.x)) v[0] = 0.0f;
    if (!bf_pos(g.y)) v[1] = 0.0f;
    if (!bf_pos(g.z)) v[2] = 0.0f;
    if (!bf_pos(g.w)) v[3] = 0.0f;
  }
  if (A.Y) {
    typedef __bf16 b4 __attribute__((ext_vector_type(4)));
    *reinterpret_cast<b4*>(A.Y + m * A.ldy + A.ycol + n) = __builtin_convertvector(v, b4);
  }
  if (A.Yf) {
    float4* d = reinterpret_cast<float4*>(A.Yf + m * A.ldyf + A.yfcol + n);
    if (A.accumulate) {
      const float4 o = *d;
      *d = make_float4(o.x + v[0], o.y + v[1], o.z + v[2], o.w + v[3]);
    } else {
      *d = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
}

template <int NT, bool XF32, int SPLIT>  // SPLIT: waves sharing the slices, 0: one pass
__global__ __launch_bounds__(SPLIT ? 64 * SPLIT : kT) void k_conv_tile(ConvArgs A, ConvTile T) {
  extern __shared__ char cv_lds[];
  constexpr int NTHR = SPLIT ? 64 * SPLIT : kT, kWaves = NTHR / 64;
  const int nline = T.planes * T.lq;
  // split sums [kWaves][mt][NT][64]; a zero operand; the staged rows; per K step and lane
  // group: byte offset of its chunk from a voxel's row, and its tap; steps with a linked tap
  // and how many precede a step (kind 2)
  f32x4* red = reinterpret_cast<f32x4*>(cv_lds);
  char* Al = cv_lds + (SPLIT ? (size_t)kWaves * T.mt * NT * 1024 : 0);
  unsigned* kt = reinterpret_cast<unsigned*>(Al + 16 + (size_t)nline * T.qz * T.row);
  unsigned short* ks = reinterpret_cast<unsigned short*>(kt + 4 * T.ksteps);
  unsigned short* kn = ks + T.ksteps;
  const int lane = threadIdx.x & 63, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int Ktot = 27 * A.cin;
  int r = blockIdx.x;
  const int z0 = r % T.ntz * T.tz;
  r /= T.ntz;
  const int y0 = r % T.nty * T.ty;
  r /= T.nty;
  const int ox = r % A.go.nx, b = r / A.go.nx;
  const int s = T.kind == 0 ? A.stride : 1;
  // the work-group's parity class and its linked taps: a parity bit links the outer taps of
  // its axis, none the middle one
  const int py = (int)blockIdx.z >> 1, pz = (int)blockIdx.z & 1;
  unsigned allow = (1u << 27) - 1;
  int nsteps = T.ksteps;
  if (T.kind == 2) {
    auto axis = [](int p) { return p ? 5u : 2u; };
    const unsigned az = axis(pz), ay = axis(py), ax = axis(ox & 1);
    const unsigned line = (ay & 1 ? az : 0) | (ay & 2 ? az << 3 : 0) | (ay & 4 ? az << 6 : 0);
    allow = (ax & 1 ? line : 0) | (ax & 2 ? line << 9 : 0) | (ax & 4 ? line << 18 : 0);
    // every wave counts, the first writes: the count is then known without a barrier
    int n = 0;
    for (int e0 = 0; e0 < T.ksteps; e0 += 64) {
      const int e = e0 + lane;
      const int t0 = 32 * e / A.cin, t1 = min(26, (32 * e + 31) / A.cin);
      const bool on = e < T.ksteps && ((2u << t1) - (1u << t0)) & allow;
      const unsigned long long m = __ballot(on);
      const int before = n + __popcll(m & ((1ull << lane) - 1));
      if (wave == 0 && e < T.ksteps) kn[e] = (unsigned short)before;
      if (wave == 0 && on) ks[before] = (unsigned short)e;
      n += __popcll(m);
    }
    if (threadIdx.x == 0) kn[T.ksteps] = (unsigned short)n;
    nsteps = __builtin_amdgcn_readfirstlane(n);
  }
  for (int e = threadIdx.x; e < 4 * T.ksteps; e += NTHR) {
    const int t = min(27, small_div(e, T.div_nch));  // entry e: chunk e of the 27 nch, step e / 4
    const int dx = t / 9, dy = t / 3 % 3, dz = t % 3;
    const int ax = T.kind == 0 ? dx : T.kind == 1 ? 2 - dx : dx == 0, ay = T.kind == 0 ? dy : T.kind == 1 ? 2 - dy : dy == 0,
              az = T.kind == 0 ? dz : T.kind == 1 ? 2 - dz : dz == 0;
    const int off = ((ax * T.lq + ay) * T.qz + az) * T.row + (e - t * T.nch) * 16;
    kt[e] = t < 27 ? (unsigned)t << 27 | (unsigned)off : 27u << 27;  // past the end: no tap
  }
  if (threadIdx.x < 4) reinterpret_cast<int*>(Al)[threadIdx.x] = 0;
  // Input rows, a chunk a thread, kB chunks in flight; outside the grid: zeros.  A thread's
  // chunks are nthr apart (a multiple of nch), so its position advances by constants.
  {
    const int xq = T.kind == 2 ? ox >> 1 : s * ox - 1, yq = T.kind == 2 ? y0 >> 1 : s * y0 - 1,
              zq = T.kind == 2 ? z0 >> 1 : s * z0 - 1;
    constexpr int kB = XF32 ? 4 : 8;
    const int rows = nline * T.qz;
    int row = small_div(threadIdx.x, T.div_nch);
    const int c = (int)threadIdx.x - row * T.nch;
    int line = small_div(row, T.div_qz), z = row - line * T.qz, d = small_div(line, T.div_lq), l = line - d * T.lq;
    if ((int)threadIdx.x >= T.nthr) row = rows;  // no chunk of its own
    const size_t xb = (size_t)b * A.gi.count() * A.ldx + A.xcol + 8 * c;
    while (row < rows) {
      bf16x8 w[kB];
      float4 f[kB][2];
      const int row0 = row;
#pragma unroll
      for (int u = 0; u < kB; ++u) {
        const int x = xq + d, y = yq + l, zz = zq + z;
        w[u] = bf16x8{0, 0, 0, 0, 0, 0, 0, 0};
        f[u][0] = f[u][1] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row < rows && (unsigned)x < (unsigned)A.gi.nx && (unsigned)y < (unsigned)A.gi.ny && (unsigned)zz < (unsigned)A.gi.nz) {
          const size_t off = xb + (size_t)((x * A.gi.ny + y) * A.gi.nz + zz) * A.ldx;
          if constexpr (XF32) {
            f[u][0] = *reinterpret_cast<const float4*>(A.Xf + off);
            f[u][1] = *reinterpret_cast<const float4*>(A.Xf + off + 4);
          } else {
            w[u] = *reinterpret_cast<const bf16x8*>(A.X + off);
          }
        }
        row += T.srow;
        z += T.sz;
        l += T.sl;
        d += T.sd;
        if (z >= T.qz) {
          z -= T.qz;
          ++l;
        }
        if (l >= T.lq) {
          l -= T.lq;
          ++d;
        }
      }
      char* to = Al + 16 + row0 * T.row + 16 * c;
#pragma unroll
      for (int u = 0; u < kB; ++u)
        if (row0 + u * T.srow < rows)
          *reinterpret_cast<bf16x8*>(to + u * T.srow * T.row) = XF32 ? cvt_bf16x8(f[u][0], f[u][1]) : w[u];
    }
  }
  __syncthreads();

  const int tye = min(T.ty, A.go.ny - y0), tze = min(T.tz, A.go.nz - z0);
  const int nyc = T.kind == 2 ? (tye - py + 1) / 2 : tye, nzc = T.kind == 2 ? (tze - pz + 1) / 2 : tze;
  // voxel positions of the class, at most 16 kConvM a wave (split: in all)
  const int cnt = nyc * T.tzc;
  const int v0 = SPLIT ? 0 : 16 * kConvM * wave;
  const int tiles = max(0, min(kConvM, (cnt - v0 + 15) / 16));
  const char* row[kConvM];
#pragma unroll
  for (int j = 0; j < kConvM; ++j) {
    const int idx = v0 + 16 * j + (lane & 15);
    const int yy = small_div(idx, T.div_tzc), zz = idx - yy * T.tzc;
    row[j] = Al + 16 + (idx < cnt ? (yy * s * T.qz + zz * s) * T.row : 0);
  }
  const bool partial = T.kind == 2 || A.cin % 32;  // a step may hold chunks without a linked tap
  auto step = [&](int k) { return T.kind == 2 ? __builtin_amdgcn_readfirstlane((int)ks[k]) : k; };
  for (int nt = 0; nt < T.nty_n; ++nt) {
    const int n0 = ((int)blockIdx.y * T.nty_n + nt) * 16 * NT;
    if (n0 >= A.cout) break;
    unsigned wo[NT];  // channels past the last read the last one's weights; never stored
#pragma unroll
    for (int q = 0; q < NT; ++q) wo[q] = (unsigned)(min(n0 + 16 * q + (lane & 15), A.cout - 1) * A.ldb + 8 * g) * 2u;
    f32x4 acc[kConvM][NT], tot[SPLIT ? 1 : kConvM][NT];
    // steps [i, iend) of the step list into acc; the next kConvAhead steps' weights load
    // from L2 while this run is multiplied.  The number of tiles N is a template argument and
    // not a branch around the products: where a block between an MFMA and a read of its result
    // rewrites only some of the accumulators, this compiler misses the shortest way round it
    // and leaves fewer than the 8 wait states that the read needs (built so: down to 1).  The
    // tail's branches below are sound: each block rewrites all N NT accumulators, so every
    // way to a read starts in the last block passed.  tests/test_mfma_waits.py checks the
    // built code's shortest ways (now 10).
    auto run = [&](int i, int iend, auto N) {
#pragma unroll
      for (int j = 0; j < kConvM; ++j)
#pragma unroll
        for (int q = 0; q < NT; ++q) acc[j][q] = f32x4{0.f, 0.f, 0.f, 0.f};
      bf16x8 w[kConvAhead][NT];
      int st[kConvAhead];
      auto load = [&](int k, int u) {
        st[u] = step(min(k, iend - 1));
        const char* base = reinterpret_cast<const char*>(A.Bt) + (size_t)64 * st[u];  // wave-uniform
#pragma unroll
        for (int q = 0; q < NT; ++q) w[u][q] = *reinterpret_cast<const bf16x8*>(base + wo[q]);
      };
      auto multiply = [&](int u) {
        const unsigned e = kt[4 * st[u] + g];
        const int off = (int)(e & 0x7FFFFFFu);
        const bool linked = (allow >> (e >> 27)) & 1u;
#pragma unroll
        for (int j = 0; j < decltype(N)::value; ++j) {
          const char* p = row[j] + off;
          if (partial) p = linked ? p : Al;
          const bf16x8 x = *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
          for (int q = 0; q < NT; ++q) acc[j][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u][q], x, acc[j][q], 0, 0, 0);
        }
      };
      if (i >= iend) return;
#pragma unroll
      for (int u = 0; u < kConvAhead; ++u) load(i + u, u);
      for (; i + kConvAhead <= iend; i += kConvAhead) {
#pragma unroll
        for (int u = 0; u < kConvAhead; ++u) {
          multiply(u);
          load(i + kConvAhead + u, u);
        }
      }
#pragma unroll
      for (int u = 0; u < kConvAhead - 1; ++u)
        if (i + u < iend) multiply(u);
    };
    auto run_tiles = [&](int i, int iend) {
      if (tiles == 4) run(i, iend, std::integral_constant<int, 4>{});
      else if (tiles == 3) run(i, iend, std::integral_constant<int, 3>{});
      else if (tiles == 2) run(i, iend, std::integral_constant<int, 2>{});
      else run(i, iend, std::integral_constant<int, 1>{});
    };
    if constexpr (SPLIT > 0) {
      for (int rd = 0; rd * kWaves < T.nsl; ++rd) {  // the waves take the slices in turn
        const int slice = rd * kWaves + wave;
        int i = min(T.ksteps, slice * T.kper), iend = min(T.ksteps, (slice + 1) * T.kper);
        if (T.kind == 2) {
          i = __builtin_amdgcn_readfirstlane((int)kn[i]);
          iend = __builtin_amdgcn_readfirstlane((int)kn[iend]);
        }
        run_tiles(i, iend);
        __syncthreads();  // the last round's sums have been read
#pragma unroll
        for (int j = 0; j < kConvM; ++j)
          if (j < T.mt)
#pragma unroll
            for (int q = 0; q < NT; ++q) red[((wave * T.mt + j) * NT + q) * 64 + lane] = acc[j][q];
        __syncthreads();
        // wave w adds the slices of tile w in order
        if (wave < T.mt) {
          const int have = min(kWaves, T.nsl - kWaves * rd);
#pragma unroll
          for (int q = 0; q < NT; ++q)
            for (int k = 0; k < have; ++k) {
              const f32x4 v = red[((k * T.mt + wave) * NT + q) * 64 + lane];
              if (rd == 0 && k == 0) tot[0][q] = v;
              else
#pragma unroll
                for (int c = 0; c < 4; ++c) tot[0][q][c] += v[c];
            }
        }
      }
    } else {
      run_tiles(0, nsteps);
#pragma unroll
      for (int j = 0; j < kConvM; ++j)
#pragma unroll
        for (int q = 0; q < NT; ++q) tot[j][q] = acc[j][q];
    }
#pragma unroll
    for (int j = 0; j < (SPLIT ? 1 : kConvM); ++j) {
      const int tile = SPLIT ? wave : j;
      const int idx = v0 + 16 * tile + (lane & 15);
      const int yy = small_div(idx, T.div_tzc), zz = idx - yy * T.tzc;
      if (tile >= tiles || idx >= cnt || zz >= nzc) continue;
      const int oy = y0 + (T.kind == 2 ? 2 * yy + py : yy), oz = z0 + (T.kind == 2 ? 2 * zz + pz : zz);
      const size_t m = (((size_t)b * A.go.nx + ox) * A.go.ny + oy) * A.go.nz + oz;
#pragma unroll
      for (int q = 0; q < NT; ++q) {
        const int n = n0 + 16 * q + 4 * g;
        if (n < A.cout) conv_epilogue4(A, m, n, tot[j][q]);
      }
    }
  }
}

// Weight and bias gradients of one layer.
//
// Every form of the convolution pairs a voxel b of a base grid with the voxels s b + d - 1
// of a halo grid (d the tap): a direct layer's base is its output and its halo its input, a
// transposed layer's the other way round.  So dW[tap] = sum_b Q[s b + d - 1] (x) P[b] with Q
// the halo tensor and P the base tensor: a GEMM over voxels whose 27 taps read the same two
// tiles.  A work-group takes 16 halo x PB base channels and a share of the tiles (a run of y
// lines and z at one x), stages P and the three planes of Q in LDS as BF16 rows of channels
// (dY rounded from FP32 once, its bias sums taken on the way), and each wave accumulates
// seven taps in registers.  The MFMA operands need eight consecutive voxels per lane where
// memory has consecutive channels: ds_read_b64_tr_b16 turns four voxel rows into columns, at
// row addresses of any stride, so a tap is only an address offset.
// Each work-group writes its sums to a slab; k_slab_sum adds the slabs in order, so the
// gradient repeats to the bit.
//
// Before, each (tap, 16 input channels) had work-groups of its own that gathered X and dY
// from global memory 2 and 4 bytes a lane and added with atomics: 65x33x33, batch 4, base
// 16: 3300 us for the 15 layers and 515 us for the bias sums; now 378 us and 85 us for the slab sums.
// LDS reads (one operand per two MFMAs) and the staging loads bound it.
constexpr int kWgradBlocks = 512;   // work-groups of one layer: two per CU
constexpr int kWgradLds = 64 * 1024;  // staged tiles, so that two work-groups share a CU
constexpr int kQB = 16;             // halo channels of a work-group

struct WgradTile {
  int ty, tz, nty, ntz, ntiles;  // base lines and z per tile, tiles per axis
  int lq, qz, kp;                // halo lines and z per plane; base voxels padded to 32
  int pt, slabs;                 // base channel blocks; voxel shares
  size_t slab;                   // floats of a slab: the layer's weights and biases
};

__device__ __forceinline__ bf16x8 tr_pair(const bf16_t* lo, const bf16_t* hi) {
  typedef short s4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4* lds_s4;
  const s4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(lo));
  const s4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(hi));
  return bf16x8{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
}

template <int PB, bool TR>
__global__ __launch_bounds__(kT, 2) void k_wgrad(WgradArgs A, WgradTile T) {
  extern __shared__ char wg_lds[];
  const int rq = 3 * T.lq * T.qz;
  bf16_t* Pl = reinterpret_cast<bf16_t*>(wg_lds);              // [kp][PB]
  bf16_t* Ql = Pl + T.kp * PB;                                 // [rq][kQB]
  unsigned short* koff = reinterpret_cast<unsigned short*>(Ql + rq * kQB);  // [kp] halo row of a base voxel
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q0 = (int)blockIdx.y / T.pt * kQB, p0 = (int)blockIdx.y % T.pt * PB;
  const Grid gb = TR ? A.gi : A.go, gq = TR ? A.go : A.gi;
  const int cq = TR ? A.cout : A.cin, cp = TR ? A.cin : A.cout;
  const int s = A.stride;
  for (int k = threadIdx.x; k < T.kp; k += kT) {
    const int y = k / T.tz, z = k - y * T.tz;
    koff[k] = (unsigned short)(k < T.ty * T.tz ? y * s * T.qz + z * s : 0);
  }
  f32x4 acc[7][PB / 16];
#pragma unroll
  for (int u = 0; u < 7; ++u)
#pragma unroll
    for (int j = 0; j < PB / 16; ++j) acc[u][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float bias[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) bias[i] = 0.0f;
  const bool sum_bias = TR ? p0 == 0 : q0 == 0;
  int tap[7];  // halo rows from a voxel's first tap
#pragma unroll
  for (int u = 0; u < 7; ++u) {
    const int t = min(wave + 4 * u, 26);
    tap[u] = (t / 9 * T.lq + t / 3 % 3) * T.qz + t % 3;
  }
  const int g = lane >> 4, i4 = (lane & 15) >> 2, ch = (lane & 3) * 4;

  for (int tile = blockIdx.x; tile < T.ntiles; tile += gridDim.x) {
    int r = tile;
    const int z0 = r % T.ntz * T.tz;
    r /= T.ntz;
    const int y0 = r % T.nty * T.ty;
    r /= T.nty;
    const int bx = r % gb.nx, b = r / gb.nx;
    __syncthreads();  // the last tile has been read
    // base rows: 8 channels a thread
    constexpr int kPc = PB / 8;
    for (int e = threadIdx.x; e < T.kp * kPc; e += kT) {
      const int k = e / kPc, c = p0 + e % kPc * 8;
      const int y = k / T.tz, z = z0 + k - y * T.tz;
      const bool in = k < T.ty * T.tz && y0 + y < gb.ny && z < gb.nz && c < cp;
      const size_t v = in ? (((size_t)b * gb.nx + bx) * gb.ny + y0 + y) * gb.nz + z : 0;
      bf16x8 w = {0, 0, 0, 0, 0, 0, 0, 0};
      if constexpr (TR) {
        if (in) w = *reinterpret_cast<const bf16x8*>(A.X + v * A.ldx + A.xcol + c);
      } else if (in) {
        float f[8];
        *reinterpret_cast<float4*>(f) = *reinterpret_cast<const float4*>(A.dY + v * A.lddy + A.dycol + c);
        *reinterpret_cast<float4*>(f + 4) = *reinterpret_cast<const float4*>(A.dY + v * A.lddy + A.dycol + c + 4);
        w = cvt_bf16x8(*reinterpret_cast<float4*>(f), *reinterpret_cast<float4*>(f + 4));
#pragma unroll
        for (int i = 0; i < 8; ++i) bias[i] += f[i];
      }
      *reinterpret_cast<bf16x8*>(Pl + k * PB + e % kPc * 8) = w;
    }
    // halo rows: three planes of lines
    for (int e = threadIdx.x; e < rq * 2; e += kT) {
      const int row = e >> 1, c = q0 + (e & 1) * 8;
      const int d = row / (T.lq * T.qz), rest = row - d * T.lq * T.qz, ly = rest / T.qz, lz = rest - ly * T.qz;
      const int x = s * bx + d - 1, y = s * y0 + ly - 1, z = s * z0 + lz - 1;
      const bool in = (unsigned)x < (unsigned)gq.nx && (unsigned)y < (unsigned)gq.ny && (unsigned)z < (unsigned)gq.nz &&
                      c < cq;
      const size_t v = in ? (((size_t)b * gq.nx + x) * gq.ny + y) * gq.nz + z : 0;
      bf16x8 w = {0, 0, 0, 0, 0, 0, 0, 0};
      if constexpr (!TR) {
        if (in) w = *reinterpret_cast<const bf16x8*>(A.X + v * A.ldx + A.xcol + c);
      } else if (in) {
        float f[8];
        *reinterpret_cast<float4*>(f) = *reinterpret_cast<const float4*>(A.dY + v * A.lddy + A.dycol + c);
        *reinterpret_cast<float4*>(f + 4) = *reinterpret_cast<const float4*>(A.dY + v * A.lddy + A.dycol + c + 4);
        w = cvt_bf16x8(*reinterpret_cast<float4*>(f), *reinterpret_cast<float4*>(f + 4));
        // each voxel of the halo grid belongs to one tile: the positions s b .. s b + s - 1
        if (d >= 1 && d <= s && ly >= 1 && ly <= s * T.ty && lz >= 1 && lz <= s * T.tz) {
#pragma unroll
          for (int i = 0; i < 8; ++i) bias[i] += f[i];
        }
      }
      *reinterpret_cast<bf16x8*>(Ql + row * kQB + (e & 1) * 8) = w;
    }
    __syncthreads();
    for (int k0 = 0; k0 < T.kp; k0 += 32) {
      // lane (g, i4): rows k0 + 8 g + i4 and + 4 of both operands
      const int k = k0 + 8 * g + i4;
      const bf16_t* pr = Pl + k * PB + ch;
      const bf16_t* ql = Ql + (int)koff[k] * kQB + ch;
      const bf16_t* qh = Ql + (int)koff[k + 4] * kQB + ch;
      bf16x8 pb[PB / 16];
#pragma unroll
      for (int j = 0; j < PB / 16; ++j) pb[j] = tr_pair(pr + 16 * j, pr + 4 * PB + 16 * j);
#pragma unroll
      for (int u = 0; u < 7; ++u) {
        const bf16x8 qa = tr_pair(ql + tap[u] * kQB, qh + tap[u] * kQB);
#pragma unroll
        for (int j = 0; j < PB / 16; ++j) acc[u][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qa, pb[j], acc[u][j], 0, 0, 0);
      }
    }
  }
  // C rows: halo channel 4 (l / 16) + i, columns: base channel l % 16
  float* out = A.part + (size_t)blockIdx.x * T.slab;
#pragma unroll
  for (int u = 0; u < 7; ++u) {
    const int t = wave + 4 * u;
    if (t >= 27) continue;
#pragma unroll
    for (int j = 0; j < PB / 16; ++j) {
      const int p = p0 + 16 * j + (lane & 15);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int q = q0 + 4 * g + i;
        if (q < cq && p < cp) out[((size_t)t * A.cin + (TR ? p : q)) * A.cout + (TR ? q : p)] = acc[u][j][i];
      }
    }
  }
  if (sum_bias) {  // a thread's chunk of 8 channels is fixed: sum the threads of each chunk
    __syncthreads();
    float* bs = reinterpret_cast<float*>(wg_lds);
#pragma unroll
    for (int i = 0; i < 8; ++i) bs[threadIdx.x * 8 + i] = bias[i];
    __syncthreads();
    constexpr int kC = TR ? 2 : PB / 8;  // chunks
    const int c0 = TR ? q0 : p0;
    if (threadIdx.x < kC * 8 && c0 + (int)threadIdx.x < A.cout) {
      float v = 0.0f;
      for (int k = threadIdx.x / 8; k < kT; k += kC) v += bs[k * 8 + threadIdx.x % 8];
      out[(size_t)27 * A.cin * A.cout + c0 + threadIdx.x] = v;
    }
  }
}

// dst[e] = sum of the slabs' e-th values: 16 lanes of four values, 16 runs of slabs added in
// parallel, then in order.  A run's loads are issued eight at a time: one by one, 512 slabs of
// a small layer were a chain of 32 memory latencies (65x33x33, batch 4, base 16, the 15
// layers: 113 us, now 85).
__global__ __launch_bounds__(kT) void k_slab_sum(const float* __restrict__ part, int slabs, size_t n,
                                                 float* __restrict__ dst) {
  __shared__ float4 sh[16][16];
  const int l = threadIdx.x % 16, r = threadIdx.x / 16;
  const int per = (slabs + 15) / 16, b0 = min(slabs, r * per), b1 = min(slabs, b0 + per);
  for (size_t e0 = blockIdx.x * (size_t)64; e0 < n; e0 += (size_t)gridDim.x * 64) {
    const size_t e = e0 + 4 * l;  // n is a multiple of 8 (channels), and so are the offsets
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (e < n)
      for (int b = b0; b < b1; b += 8) {
        float4 p[8];
#pragma unroll
        for (int k = 0; k < 8; ++k)
          p[k] = b + k < b1 ? *reinterpret_cast<const float4*>(part + (size_t)(b + k) * n + e) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
          v.x += p[k].x;
          v.y += p[k].y;
          v.z += p[k].z;
          v.w += p[k].w;
        }
      }
    sh[r][l] = v;
    __syncthreads();
    if (r == 0 && e < n) {
      for (int k = 1; k < 16; ++k) {
        const float4 p = sh[k][l];
        v.x += p.x;
        v.y += p.y;
        v.z += p.z;
        v.w += p.w;
      }
      *reinterpret_cast<float4*>(dst + e) = v;
    }
    __syncthreads();
  }
}

__global__ __launch_bounds__(kT) void k_pack(const float* W, int cin, int cout, bf16_t* Bf, int ldf, bf16_t* Bd, int ldd) {
  const size_t n = (size_t)27 * cin * cout;
  for (size_t e = blockIdx.x * (size_t)kT + threadIdx.x; e < n; e += (size_t)gridDim.x * kT) {
    const int co = (int)(e % cout);
    const size_t r = e / cout;
    const int ci = (int)(r % cin);
    const int t = (int)(r / cin);
    const bf16_t v = f2bf(W[e]);
    Bf[(size_t)co * ldf + (size_t)t * cin + ci] = v;
    Bd[(size_t)ci * ldd + (size_t)t * cout + co] = v;
  }
}

__global__ __launch_bounds__(kT) void k_adam(float* w, const float* g, float* m, float* v, size_t n, float lr,
                                             float b1, float b2, float eps, float c1, float c2) {
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) {
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  }
}

__global__ __launch_bounds__(kT) void k_mse(const float* p, const float* y, size_t n, float* dp, double* P) {
  __shared__ double sh[kT / 64];
  double s = 0.0;
  const float sc = 2.0f / (float)n;
  for (size_t i = blockIdx.x * (size_t)kT + threadIdx.x; i < n; i += (size_t)gridDim.x * kT) {
    const float d = p[i] - y[i];
    s += (double)d * d;
    dp[i] = sc * d;
  }
  const double t = block_reduce_all<kT>(s, sh);
  if (threadIdx.x == 0) P[blockIdx.x] = t / (double)n;
}

int blocks_for(size_t n, int cap = 4096) {
  size_t g = (n + kT - 1) / kT;
  return (int)(g < 1 ? 1 : (g > (size_t)cap ? cap : g));
}

}  // namespace

// n split evenly into runs of at most `most`, each a multiple of `unit`
static int even_runs(int n, int most, int unit = 1) {
  const int runs = (n + most - 1) / most;
  return ((n + runs - 1) / runs + unit - 1) / unit * unit;
}

// Tile of a staged convolution (`waves` sharing the slices, 0: one pass); false when no tile
// fits the LDS budget.
static bool conv_tile(const ConvArgs& a, int ksteps, int kper, int nsl, int nt, int waves, ConvTile& t, size_t& lds) {
  t.kind = a.transposed ? (a.stride == 2 ? 2 : 1) : 0;
  const int unit = t.kind == 2 ? 2 : 1, s = t.kind == 0 ? a.stride : 1, ncls = t.kind == 2 ? 4 : 1;
  t.nch = a.cin / 8;
  t.row = 16 * (t.nch | 1);  // an odd number of 16-byte banks: 16 consecutive rows hit all of them
  t.ksteps = ksteps;
  t.kper = kper;
  t.nsl = nsl;
  t.planes = t.kind == 2 ? 2 : 3;
  // 16-voxel tiles of a work-group (kind 2: of one parity class)
  auto tiles = [&](int ty, int tz) { return t.kind == 2 ? (ty / 2 * (tz / 2) + 15) / 16 : (ty * tz + 15) / 16; };
  auto bytes = [&]() {
    t.lq = t.kind == 2 ? t.ty / 2 + 1 : (t.ty - 1) * s + 3;
    t.qz = t.kind == 2 ? t.tz / 2 + 1 : (t.tz - 1) * s + 3;
    t.mt = std::min(kConvM, tiles(t.ty, t.tz));
    return (size_t)waves * t.mt * nt * 1024 + 16 + (size_t)t.planes * t.lq * t.qz * t.row + (size_t)16 * ksteps +
           4 * (size_t)ksteps + 2;
  };
  // z runs of at most 64; shorter ones where a single line of wide channels does not fit
  for (int most = 64; most >= 8; most /= 2) {
    t.tz = even_runs(a.go.nz, most, unit);
    t.ty = unit;
    if (bytes() <= kConvLdsMax) break;
  }
  if (bytes() > kConvLdsMax) return false;
  // lines: enough tiles for four waves of kConvM (or kConvM, the waves sharing the slices),
  // while two work-groups fit a CU and the grid still covers the CUs twice
  const int most = nsl > 1 ? kConvM : 4 * kConvM;
  const int nb = ((a.cout + 15) / 16 + nt - 1) / nt;
  int best = t.ty;
  for (int y = t.ty + unit; y <= a.go.ny + unit - 1 && y <= 32; y += unit) {
    t.ty = y;
    const long wgs = (long)a.batch * a.go.nx * ((a.go.ny + y - 1) / y) * ((a.go.nz + t.tz - 1) / t.tz) * nb * ncls;
    if (bytes() > kConvLdsGoal || tiles(y, t.tz) > most || wgs < kConvGroups) break;
    best = y;
  }
  t.ty = even_runs(a.go.ny, best, unit);
  lds = bytes();
  t.nty = (a.go.ny + t.ty - 1) / t.ty;
  t.ntz = (a.go.nz + t.tz - 1) / t.tz;
  // channel tiles: in one work-group while the voxel tiles alone fill the chip
  const long wgs = (long)a.batch * a.go.nx * t.nty * t.ntz * ncls;
  t.nty_n = (int)std::max<long>(1, std::min<long>(nb, wgs * nb / 1024));
  t.tzc = t.kind == 2 ? t.tz / 2 : t.tz;
  t.div_nch = small_div_factor(t.nch);
  t.div_lq = small_div_factor(t.lq);
  t.div_qz = small_div_factor(t.qz);
  t.div_tzc = small_div_factor(t.tzc);
  const int threads = waves ? 64 * waves : kT;
  t.srow = std::max(1, threads / t.nch);
  t.nthr = t.srow * t.nch;
  t.sz = t.srow % t.qz;
  t.sl = t.srow / t.qz % t.lq;
  t.sd = t.srow / t.qz / t.lq;
  return t.nthr <= threads;
}

template <int NT, bool XF32, int SPLIT>
static void launch_conv_tile(const ConvArgs& a, const ConvTile& t, dim3 grid, size_t lds, hipStream_t s) {
  if (lds > 64 * 1024) {  // once per device
    static std::atomic<unsigned long long> done{0};
    int dev = 0;
    (void)hipGetDevice(&dev);
    const unsigned long long bit = 1ull << (dev & 63);
    if (!(done.load() & bit)) {
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(&k_conv_tile<NT, XF32, SPLIT>),
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)kConvLdsMax);
      done.fetch_or(bit);
    }
  }
  k_conv_tile<NT, XF32, SPLIT><<<grid, SPLIT ? 64 * SPLIT : kT, lds, s>>>(a, t);
}

hipError_t launch_conv(const ConvArgs& a, hipStream_t s) {
  const int M = a.batch * a.go.count();
  const int waves = ((M + 15) / 16) * ((a.cout + 63) / 64);
  const int ksteps = (27 * a.cin + 31) / 32;
  // slices of at least two K steps until 64-channel work-groups of 64 voxels would hold
  // about kConvFillWaves waves
  int nsl = 1;
  if (a.part && waves < kConvFillWaves) {
    nsl = std::min({(kConvFillWaves + waves - 1) / waves, ksteps / 2, kConvMaxSlices});
    while (nsl > 1 && (size_t)nsl * M * a.cout > a.part_cap) --nsl;
  }
  int kper = ksteps;
  if (nsl > 1) {
    kper = (ksteps + nsl - 1) / nsl;
    nsl = (ksteps + kper - 1) / kper;  // every slice non-empty
  }
  ConvTile t{};
  size_t lds = 0;
  // two channel tiles share an input operand where there are two; eight waves where there
  // are slices for them
  const int nt = a.cout > 16 && nsl == 1 ? 2 : 1, sw = nsl > 4 ? 8 : nsl > 1 ? 4 : 0;
  if (conv_tile(a, ksteps, kper, nsl, nt, sw, t, lds)) {
    const dim3 grid(a.batch * a.go.nx * t.nty * t.ntz, ((a.cout + 16 * nt - 1) / (16 * nt) + t.nty_n - 1) / t.nty_n,
                    t.kind == 2 ? 4 : 1);
    if (sw == 8) {
      if (a.X) launch_conv_tile<1, false, 8>(a, t, grid, lds, s);
      else launch_conv_tile<1, true, 8>(a, t, grid, lds, s);
    } else if (sw == 4) {
      if (a.X) launch_conv_tile<1, false, 4>(a, t, grid, lds, s);
      else launch_conv_tile<1, true, 4>(a, t, grid, lds, s);
    } else if (nt == 2) {
      if (a.X) launch_conv_tile<2, false, 0>(a, t, grid, lds, s);
      else launch_conv_tile<2, true, 0>(a, t, grid, lds, s);
    } else {
      if (a.X) launch_conv_tile<1, false, 0>(a, t, grid, lds, s);
      else launch_conv_tile<1, true, 0>(a, t, grid, lds, s);
    }
    return hipGetLastError();
  }
  dim3 grid((M + 63) / 64, (a.cout + 63) / 64);
  if (nsl <= 1) {
    if (a.X) k_conv<false, false><<<grid, kT, 0, s>>>(a, ksteps);
    else k_conv<true, false><<<grid, kT, 0, s>>>(a, ksteps);
    return hipGetLastError();
  }
  grid.z = nsl;
  if (a.X) k_conv<false, true><<<grid, kT, 0, s>>>(a, kper);
  else k_conv<true, true><<<grid, kT, 0, s>>>(a, kper);
  k_conv_reduce<<<blocks_for((size_t)M * a.cout), kT, 0, s>>>(a, nsl);
  return hipGetLastError();
}

hipError_t launch_wgrad(const WgradArgs& a, hipStream_t s) {
  const bool tr = a.transposed != 0;
  const Grid gb = tr ? a.gi : a.go;
  const int cq = tr ? a.cout : a.cin, cp = tr ? a.cin : a.cout;
  const int pb = cp > 16 ? 32 : 16;
  WgradTile t{};
  auto bytes = [&]() {
    t.lq = (t.ty - 1) * a.stride + 3;
    t.qz = (t.tz - 1) * a.stride + 3;
    t.kp = (t.ty * t.tz + 31) / 32 * 32;
    return (size_t)t.kp * pb * 2 + (size_t)3 * t.lq * t.qz * kQB * 2 + (size_t)t.kp * 2;
  };
  // z runs of at most 64, then as many lines as fit (at least one: 3 x 3 x 131 halo rows)
  t.tz = even_runs(gb.nz, 64);
  t.ty = 1;
  for (int y = 2; y <= std::min(gb.ny, 16); ++y) {
    const int keep = t.ty;
    t.ty = y;
    if (bytes() > kWgradLds) {
      t.ty = keep;
      break;
    }
  }
  t.ty = even_runs(gb.ny, t.ty);
  const size_t lds = std::max(bytes(), (size_t)kT * 8 * sizeof(float));
  t.nty = (gb.ny + t.ty - 1) / t.ty;
  t.ntz = (gb.nz + t.tz - 1) / t.tz;
  t.ntiles = a.batch * gb.nx * t.nty * t.ntz;
  t.pt = (cp + pb - 1) / pb;
  t.slab = (size_t)27 * a.cin * a.cout + a.cout;
  const int by = (cq + kQB - 1) / kQB * t.pt;
  t.slabs = (int)std::min<size_t>({(size_t)std::max(1, kWgradBlocks / by), (size_t)t.ntiles,
                                   std::max<size_t>(1, a.part_cap / t.slab)});
  WgradArgs w = a;
  if (t.slabs == 1) w.part = a.dW;  // biases follow the weights in the parameter vector
  const dim3 grid(t.slabs, by);
  if (pb == 32) {
    if (tr) k_wgrad<32, true><<<grid, kT, lds, s>>>(w, t);
    else k_wgrad<32, false><<<grid, kT, lds, s>>>(w, t);
  } else {
    if (tr) k_wgrad<16, true><<<grid, kT, lds, s>>>(w, t);
    else k_wgrad<16, false><<<grid, kT, lds, s>>>(w, t);
  }
  if (t.slabs > 1)
    k_slab_sum<<<(int)std::min<size_t>(2048, (t.slab + 63) / 64), kT, 0, s>>>(w.part, t.slabs, t.slab, a.dW);
  return hipGetLastError();
}

hipError_t launch_pack(const float* W, int cin, int cout, bf16_t* Bfwd, bf16_t* Bdgrad, hipStream_t s) {
  k_pack<<<blocks_for((size_t)27 * cin * cout), kT, 0, s>>>(W, cin, cout, Bfwd, packed_row(cin), Bdgrad, packed_row(cout));
  return hipGetLastError();
}

hipError_t launch_adam(float* w, const float* g, float* m, float* v, size_t n, float lr, float b1, float b2,
                       float eps, int t, hipStream_t s) {
  const float c1 = 1.0f - powf(b1, (float)t), c2 = 1.0f - powf(b2, (float)t);
  k_adam<<<blocks_for(n), kT, 0, s>>>(w, g, m, v, n, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t launch_mse(const float* pred, const float* target, size_t n, float* dp, double* partials, int grid,
                      hipStream_t s) {
  k_mse<<<grid, kT, 0, s>>>(pred, target, n, dp, partials);
  return hipGetLastError();
}

}  // namespace unet
}  // namespace pa

// ------------------------------------------------------------------ network (host)
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/plato_mi355x.h"
#include "pa_host.hpp"

namespace {

using pa::unet::bf16_t;
using pa::unet::Grid;

constexpr int kInCh = 8;   // density, load (3), coordinates (3), ones
constexpr int kOutCh = 16;  // displacement channels (3, or 9 for three load cases) + padding

// f32 -> bf16 conversion of the network input
__global__ void k_to_bf16(const float* x, bf16_t* y, size_t n) {
  for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) {
    const uint32_t u = __float_as_uint(x[i]);
    y[i] = ((u & 0x7F800000u) == 0x7F800000u) ? (bf16_t)(u >> 16) : (bf16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
  }
}

template <typename T>
struct Dev {
  T* p = nullptr;
  size_t n = 0;
  Dev() = default;
  Dev(const Dev&) = delete;
  Dev& operator=(const Dev&) = delete;
  Dev(Dev&& o) noexcept : p(o.p), n(o.n) {
    o.p = nullptr;
    o.n = 0;
  }
  hipError_t alloc(size_t k) {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = k;
    return k ? hipMalloc(&p, k * sizeof(T)) : hipSuccess;
  }
  ~Dev() {
    if (p) (void)hipFree(p);
  }
};

// A tensor view: buffer, row stride, first channel, channels.
struct View {
  void* p;
  int ld, col, c;
};

struct Layer {
  int cin, cout, stride, transposed, relu;
  int lin, lout;        // grid levels of input and output
  View in, out;         // activations (bf16; out of the last layer is fp32)
  View gin, gout;       // gradients (fp32); gin.p null for the first layer
  size_t w_off, b_off;  // offsets into the parameter vector
  bf16_t *Bf, *Bd;
};

}  // namespace

struct pa_unet_s {
  Grid g[4];
  int base = 16, batch = 0;
  std::vector<Layer> L;
  size_t nparams = 0;
  Dev<float> P, G, M, V;  // parameters, gradients, Adam moments
  Dev<bf16_t> B;          // packed bf16 operands of all layers
  std::vector<Dev<bf16_t>> act;
  std::vector<Dev<float>> grad;
  Dev<float> out, dout;
  Dev<bf16_t> in;
  Dev<double> partials;
  Dev<float> split;  // split-reduction slices of the small convolutions
  double* host_partials = nullptr;
  hipEvent_t loss_event = nullptr;  // the loss has arrived
  int step = 0;
  hipStream_t stream = nullptr;
  std::string err;
  ~pa_unet_s() {
    if (loss_event) (void)hipEventDestroy(loss_event);
    if (host_partials) (void)hipHostFree(host_partials);
  }
};

namespace {

thread_local std::string g_unet_err;

int ufail(pa_unet h, int code, const std::string& msg) {
  if (h) h->err = msg;
  g_unet_err = msg;
  return code;
}

#define PA_UHIP(h, x)                                                                       \
  do {                                                                                      \
    hipError_t e_ = (x);                                                                    \
    if (e_ != hipSuccess) return ufail(h, PA_ERR_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
  } while (0)

// Buffers per batch size: activations and gradients of every level.
//   act: 0 in(8) [l0], 1 e0(C) [l0], 2 cat0(2C) [l0], 3 e1(2C) [l1], 4 cat1(4C) [l1],
//        5 e2(4C) [l2], 6 cat2(8C) [l2], 7 e3(8C) [l3], 8 b3(8C) [l3], 9 d2(4C) [l2],
//        10 d1(2C) [l1], 11 d0(C) [l0]
struct Buf {
  int level, ch;
};
constexpr int kNumBuf = 12;
constexpr size_t kSplitFloats = (size_t)8 << 20;  // 32 MB of split-reduction slices

void build_layers(pa_unet h) {
  const int C = h->base;
  const Buf bufs[kNumBuf] = {{0, kInCh}, {0, C}, {0, 2 * C}, {1, 2 * C}, {1, 4 * C}, {2, 4 * C},
                             {2, 8 * C}, {3, 8 * C}, {3, 8 * C}, {2, 4 * C}, {1, 2 * C}, {0, C}};
  (void)bufs;
  // (input buffer, col, cin) -> (output buffer, col, cout), stride, transposed, relu
  struct Def {
    int bi, ci, cin, bo, co, cout, s, tr, relu;
  };
  const Def defs[] = {
      {0, 0, kInCh, 1, 0, C, 1, 0, 1},          // enc0
      {1, 0, C, 2, 0, C, 1, 0, 1},              // enc0b -> skip 0
      {2, 0, C, 3, 0, 2 * C, 2, 0, 1},          // down0
      {3, 0, 2 * C, 4, 0, 2 * C, 1, 0, 1},      // enc1 -> skip 1
      {4, 0, 2 * C, 5, 0, 4 * C, 2, 0, 1},      // down1
      {5, 0, 4 * C, 6, 0, 4 * C, 1, 0, 1},      // enc2 -> skip 2
      {6, 0, 4 * C, 7, 0, 8 * C, 2, 0, 1},      // down2
      {7, 0, 8 * C, 8, 0, 8 * C, 1, 0, 1},      // bottleneck
      {8, 0, 8 * C, 6, 4 * C, 4 * C, 2, 1, 1},  // up2 -> cat2
      {6, 0, 8 * C, 9, 0, 4 * C, 1, 0, 1},      // dec2
      {9, 0, 4 * C, 4, 2 * C, 2 * C, 2, 1, 1},  // up1 -> cat1
      {4, 0, 4 * C, 10, 0, 2 * C, 1, 0, 1},     // dec1
      {10, 0, 2 * C, 2, C, C, 2, 1, 1},         // up0 -> cat0
      {2, 0, 2 * C, 11, 0, C, 1, 0, 1},         // dec0
      {11, 0, C, -1, 0, kOutCh, 1, 0, 0},       // output (fp32)
  };
  const int lev[kNumBuf] = {0, 0, 0, 1, 1, 2, 2, 3, 3, 2, 1, 0};
  const int ldb[kNumBuf] = {kInCh, C, 2 * C, 2 * C, 4 * C, 4 * C, 8 * C, 8 * C, 8 * C, 4 * C, 2 * C, C};
  h->L.clear();
  size_t off = 0;
  for (const Def& d : defs) {
    Layer l{};
    l.cin = d.cin;
    l.cout = d.cout;
    l.stride = d.s;
    l.transposed = d.tr;
    l.relu = d.relu;
    l.lin = lev[d.bi];
    l.lout = d.bo >= 0 ? lev[d.bo] : 0;
    l.in = View{(void*)(intptr_t)d.bi, ldb[d.bi], d.ci, d.cin};
    l.out = d.bo >= 0 ? View{(void*)(intptr_t)d.bo, ldb[d.bo], d.co, d.cout} : View{nullptr, kOutCh, 0, kOutCh};
    l.w_off = off;
    off += (size_t)27 * d.cin * d.cout;
    l.b_off = off;
    off += d.cout;
    h->L.push_back(l);
  }
  h->nparams = off;
}

int ensure_batch(pa_unet h, int batch) {
  if (batch == h->batch) return PA_OK;
  const int C = h->base;
  const int lev[kNumBuf] = {0, 0, 0, 1, 1, 2, 2, 3, 3, 2, 1, 0};
  const int ldb[kNumBuf] = {kInCh, C, 2 * C, 2 * C, 4 * C, 4 * C, 8 * C, 8 * C, 8 * C, 4 * C, 2 * C, C};
  h->act.clear();
  h->grad.clear();
  h->act.resize(kNumBuf);
  h->grad.resize(kNumBuf);
  for (int b = 0; b < kNumBuf; ++b) {
    const size_t n = (size_t)batch * h->g[lev[b]].count() * ldb[b];
    PA_UHIP(h, h->act[b].alloc(n));
    PA_UHIP(h, h->grad[b].alloc(n));
  }
  const size_t no = (size_t)batch * h->g[0].count() * kOutCh;
  PA_UHIP(h, h->out.alloc(no));
  PA_UHIP(h, h->dout.alloc(no));
  if (!h->split.p) PA_UHIP(h, h->split.alloc(kSplitFloats));
  h->batch = batch;
  return PA_OK;
}

pa::unet::ConvArgs fwd_args(pa_unet h, const Layer& l) {
  pa::unet::ConvArgs a{};
  const int bi = (int)(intptr_t)l.in.p;
  a.X = h->act[bi].p;
  a.ldx = l.in.ld;
  a.xcol = l.in.col;
  a.cin = l.cin;
  a.gi = h->g[l.lin];
  a.go = h->g[l.lout];
  a.batch = h->batch;
  a.stride = l.stride;
  a.transposed = l.transposed;
  a.Bt = l.Bf;
  a.ldb = pa::unet::packed_row(l.cin);
  a.cout = l.cout;
  a.bias = h->P.p + l.b_off;
  a.relu = l.relu;
  if (l.out.p) {
    a.Y = h->act[(int)(intptr_t)l.out.p].p;
    a.ldy = l.out.ld;
    a.ycol = l.out.col;
  } else {
    a.Yf = h->out.p;
    a.ldyf = kOutCh;
  }
  a.part = h->split.p;
  a.part_cap = h->split.n;
  return a;
}

// y: where the output goes, if not to h->out
int forward(pa_unet h, float* y = nullptr) {
  for (const Layer& l : h->L) {
    pa::unet::ConvArgs a = fwd_args(h, l);
    if (y && a.Yf) a.Yf = y;
    PA_UHIP(h, pa::unet::launch_conv(a, h->stream));
  }
  return PA_OK;
}

int backward(pa_unet h) {
  for (int k = (int)h->L.size() - 1; k >= 0; --k) {
    const Layer& l = h->L[k];
    const int bi = (int)(intptr_t)l.in.p;
    // gradient of this layer's output (already multiplied by the ReLU derivative)
    const float* dY = l.out.p ? h->grad[(int)(intptr_t)l.out.p].p : h->dout.p;
    const int lddy = l.out.ld, dycol = l.out.col;
    pa::unet::WgradArgs w{};
    w.X = h->act[bi].p;
    w.ldx = l.in.ld;
    w.xcol = l.in.col;
    w.cin = l.cin;
    w.gi = h->g[l.lin];
    w.go = h->g[l.lout];
    w.batch = h->batch;
    w.stride = l.stride;
    w.transposed = l.transposed;
    w.dY = dY;
    w.lddy = lddy;
    w.dycol = dycol;
    w.cout = l.cout;
    w.dW = h->G.p + l.w_off;
    w.part = h->split.p;
    w.part_cap = h->split.n;
    PA_UHIP(h, pa::unet::launch_wgrad(w, h->stream));
    if (k == 0) continue;  // no gradient for the network input
    pa::unet::ConvArgs a{};
    a.Xf = dY;
    a.ldx = lddy;
    a.xcol = dycol;
    a.cin = l.cout;
    a.gi = h->g[l.lout];
    a.go = h->g[l.lin];
    a.batch = h->batch;
    a.stride = l.stride;
    a.transposed = !l.transposed;
    a.Bt = l.Bd;
    a.ldb = pa::unet::packed_row(l.cout);
    a.cout = l.cin;
    a.Yf = h->grad[bi].p;
    a.ldyf = l.in.ld;
    a.yfcol = l.in.col;
    // skip tensors receive a second gradient from the down-sampling layer (their first
    // consumer in the backward order is the decoder conv that reads the concatenation)
    a.accumulate = (l.stride == 2 && !l.transposed) ? 1 : 0;
    a.gate = h->act[bi].p;  // every layer input except the network input is a ReLU output
    a.ldg = l.in.ld;
    a.gcol = l.in.col;
    a.part = h->split.p;
    a.part_cap = h->split.n;
    PA_UHIP(h, pa::unet::launch_conv(a, h->stream));
  }
  return PA_OK;
}

int repack(pa_unet h) {
  for (const Layer& l : h->L)
    PA_UHIP(h, pa::unet::launch_pack(h->P.p + l.w_off, l.cin, l.cout, l.Bf, l.Bd, h->stream));
  return PA_OK;
}

int load_input(pa_unet h, const float* x, int batch) {
  if (int rc = ensure_batch(h, batch)) return rc;
  const size_t n = (size_t)batch * h->g[0].count() * kInCh;
  k_to_bf16<<<(int)std::min<size_t>(4096, (n + 255) / 256), 256, 0, h->stream>>>(x, h->act[0].p, n);
  PA_UHIP(h, hipGetLastError());
  return PA_OK;
}

int loss_and_grad(pa_unet h, const float* target, double* loss) {
  const size_t n = (size_t)h->batch * h->g[0].count() * kOutCh;
  const int grid = (int)std::min<size_t>(1024, (n + 255) / 256);
  PA_UHIP(h, pa::unet::launch_mse(h->out.p, target, n, h->dout.p, h->partials.p, grid, h->stream));
  PA_UHIP(h, hipMemcpyAsync(h->host_partials, h->partials.p, grid * sizeof(double), hipMemcpyDeviceToHost,
                            h->stream));
  if (!h->loss_event) PA_UHIP(h, hipEventCreateWithFlags(&h->loss_event, hipEventDisableTiming));
  PA_UHIP(h, hipEventRecord(h->loss_event, h->stream));
  // the backward pass is queued before the host waits for the loss, so the GPU does not wait
  // for the host
  const int rc = backward(h);
  PA_UHIP(h, hipEventSynchronize(h->loss_event));
  double s = 0.0;
  for (int i = 0; i < grid; ++i) s += h->host_partials[i];
  if (loss) *loss = s;
  return rc;
}

}  // namespace

extern "C" {

const char* pa_unet_last_error(void) { return g_unet_err.c_str(); }

int pa_unet_create(pa_unet* out, int nx, int ny, int nz, int base_channels, unsigned long long seed) {
  if (!out) return ufail(nullptr, PA_ERR_ARG, "pa_unet_create: null output");
  *out = nullptr;
  if (base_channels < 8 || base_channels % 8) return ufail(nullptr, PA_ERR_ARG, "base_channels must be a multiple of 8");
  if (nx < 5 || ny < 5 || nz < 5 || (nx - 1) % 4 || (ny - 1) % 4 || (nz - 1) % 4)
    return ufail(nullptr, PA_ERR_ARG, "node grid dimensions must be 1 mod 4 and >= 5 (odd on three levels)");
  auto h = new pa_unet_s();
  h->base = base_channels;
  h->g[0] = Grid{nx, ny, nz};
  for (int l = 1; l < 4; ++l)
    h->g[l] = Grid{(h->g[l - 1].nx + 1) / 2, (h->g[l - 1].ny + 1) / 2, (h->g[l - 1].nz + 1) / 2};
  build_layers(h);
  auto cleanup = [&](int rc) {
    delete h;
    return rc;
  };
  if (h->P.alloc(h->nparams) || h->G.alloc(h->nparams) || h->M.alloc(h->nparams) || h->V.alloc(h->nparams) ||
      h->partials.alloc(1024) || hipHostMalloc(&h->host_partials, 1024 * sizeof(double)))
    return cleanup(ufail(nullptr, PA_ERR_HIP, "pa_unet_create: device allocation failed"));
  size_t nb = 0;
  auto fsize = [](const Layer& l) { return (size_t)l.cout * pa::unet::packed_row(l.cin); };
  auto dsize = [](const Layer& l) { return (size_t)l.cin * pa::unet::packed_row(l.cout); };
  for (const Layer& l : h->L) nb += fsize(l) + dsize(l);
  // the rows' padding stays zero: the pack kernel writes the weights only
  if (h->B.alloc(nb) || hipMemset(h->B.p, 0, nb * sizeof(bf16_t))) return cleanup(ufail(nullptr, PA_ERR_HIP, "pa_unet_create: device allocation failed"));
  size_t o = 0;
  for (Layer& l : h->L) {
    l.Bf = h->B.p + o;
    o += fsize(l);
    l.Bd = h->B.p + o;
    o += dsize(l);
  }
  // He-normal weights (fan-in 27 cin), zero biases
  std::vector<float> p(h->nparams, 0.0f);
  std::vector<pa::NormalRun> runs;
  for (const Layer& l : h->L) runs.push_back({l.w_off, (size_t)27 * l.cin * l.cout, std::sqrt(2.0f / (27.0f * l.cin))});
  pa::normal_runs(seed, runs, p.data());
  if (hipMemcpy(h->P.p, p.data(), p.size() * sizeof(float), hipMemcpyHostToDevice) ||
      hipMemset(h->M.p, 0, h->nparams * sizeof(float)) || hipMemset(h->V.p, 0, h->nparams * sizeof(float)))
    return cleanup(ufail(nullptr, PA_ERR_HIP, "pa_unet_create: upload failed"));
  if (repack(h) || hipStreamSynchronize(nullptr)) return cleanup(ufail(nullptr, PA_ERR_HIP, "pa_unet_create: pack failed"));
  *out = h;
  return PA_OK;
}

int pa_unet_destroy(pa_unet h) {
  delete h;
  return PA_OK;
}

int pa_unet_set_stream(pa_unet h, void* stream) {
  if (!h) return ufail(nullptr, PA_ERR_ARG, "null handle");
  h->stream = (hipStream_t)stream;
  return PA_OK;
}

int pa_unet_num_params(pa_unet h, size_t* n) {
  if (!h || !n) return ufail(h, PA_ERR_ARG, "null argument");
  *n = h->nparams;
  return PA_OK;
}

int pa_unet_params(pa_unet h, float* dst, const float* src) {
  if (!h) return ufail(nullptr, PA_ERR_ARG, "null handle");
  if (dst) PA_UHIP(h, hipMemcpyAsync(dst, h->P.p, h->nparams * sizeof(float), hipMemcpyDeviceToDevice, h->stream));
  if (src) {
    PA_UHIP(h, hipMemcpyAsync(h->P.p, src, h->nparams * sizeof(float), hipMemcpyDeviceToDevice, h->stream));
    if (int rc = repack(h)) return rc;
  }
  return PA_OK;
}

int pa_unet_forward(pa_unet h, const float* x, int batch, float* y) {
  if (!h || !x || !y || batch < 1) return ufail(h, PA_ERR_ARG, "pa_unet_forward: bad argument");
  if (int rc = load_input(h, x, batch)) return rc;
  // the last layer stores 16 bytes a lane, so its output goes straight to a y aligned to that
  const bool direct = reinterpret_cast<size_t>(y) % 16 == 0;
  if (int rc = forward(h, direct ? y : nullptr)) return rc;
  if (!direct)
    PA_UHIP(h, hipMemcpyAsync(y, h->out.p, (size_t)batch * h->g[0].count() * kOutCh * sizeof(float),
                              hipMemcpyDeviceToDevice, h->stream));
  return PA_OK;
}

int pa_unet_gradient(pa_unet h, const float* x, const float* target, int batch, float* grad, double* loss) {
  if (!h || !x || !target || batch < 1) return ufail(h, PA_ERR_ARG, "pa_unet_gradient: bad argument");
  if (int rc = load_input(h, x, batch)) return rc;
  if (int rc = forward(h)) return rc;
  if (int rc = loss_and_grad(h, target, loss)) return rc;
  if (grad) PA_UHIP(h, hipMemcpyAsync(grad, h->G.p, h->nparams * sizeof(float), hipMemcpyDeviceToDevice, h->stream));
  return PA_OK;
}

int pa_unet_train_step(pa_unet h, const float* x, const float* target, int batch, float lr, double* loss) {
  if (int rc = pa_unet_gradient(h, x, target, batch, nullptr, loss)) return rc;
  ++h->step;
  PA_UHIP(h, pa::unet::launch_adam(h->P.p, h->G.p, h->M.p, h->V.p, h->nparams, lr, 0.9f, 0.999f, 1e-8f, h->step,
                                   h->stream));
  return repack(h);
}

}  // extern "C"
