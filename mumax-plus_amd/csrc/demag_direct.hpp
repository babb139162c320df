// Demag field of a small magnet by direct summation of the real-space kernel,
// in one launch.
//
// A magnet of a few thousand cells leaves the FFT passes at their launch
// latency (three to five dependent launches of 5 us each).  The direct sum
//   h(r) = sum_r' K(r - r') Ms m(r'),  K = -mu0 N (FP64 Newell, rounded once)
// costs N^2 products but no intermediate: one wavefront sums four consecutive
// x cells (a strip) over all sources.
//
// Layout.  M = Ms m is staged in LDS with rows padded to a multiple of four
// cells (zeros), so a lane reads four sources of a component as one 16-byte
// access and consecutive lanes read consecutive blocks: no bank conflicts.  A
// unit of work is four sources of one row against the strip's four cells: the
// 16 pairs share seven kernel entries (dx = D-3..D+3), so a lane loads 7
// entries for 80 (single layer) or 144 products.  The kernel is stored for
// |dy|, |dz| and signed dx, so the seven loads of a unit have one address and
// immediate offsets; the signs of the components odd in y or z are applied on
// the fly.  A strip's units are shared out over the lanes of one or more
// wavefronts of a block (direct_launch), so that a lane has few units and the
// unit loads of several wavefronts hide each other's latency.  The 12 partial
// sums of a lane are reduced over the wavefront by a reduce-scatter (21
// shuffles), and over the strip's wavefronts through LDS.  Every output is a
// sum of short chains followed by a tree, so its rounding stays at that of
// the FFT passes.
#pragma once

#include "common.hpp"

namespace mpa {

struct DirectDesc {
  int nx, ny, nz;
  int nb;     // blocks of four cells per row: ceil(nx / 4)
  int rows;   // ny nz
  int l2s, l2w;  // log2 of the strips per block and of the wavefronts per strip
  unsigned mag_nb, mag_ny;  // floor(2^32 / nb) + 1, floor(2^32 / ny) + 1
  const float4* K4;  // (xx, yy, zz, xy) at [|dz|][|dy|][4 nb + dx], 8 nb entries a row
  const float2* K2;  // (xz, yz), nullptr for a single layer
};

// q / d for q d < 2^32 with the magic factor floor(2^32 / d) + 1 (d > 1; the
// factor of d == 1 wraps to 1, and q is returned).
__device__ __forceinline__ int direct_div(int q, int d, unsigned magic) {
  return d == 1 ? q : (int)__umulhi((unsigned)q, magic);
}

// Launch shape.  Strips per block: as many as fill 256 compute units once
// (each block stages the whole source); wavefronts per strip: one per 64
// units, within a block of 16 wavefronts.
inline void direct_shape(DirectDesc& D) {
  const int strips = D.rows * D.nb;
  D.l2s = D.l2w = 0;
  while ((256 << D.l2s) < strips && D.l2s < 3) ++D.l2s;
  while ((64 << D.l2w) < strips && D.l2s + D.l2w < 4) ++D.l2w;
}
struct DirectLaunch {
  unsigned blocks, threads;
  size_t shm;
};
inline DirectLaunch direct_launch(const DirectDesc& D) {
  const int strips = D.rows * D.nb, per = 1 << D.l2s;
  return DirectLaunch{(unsigned)((strips + per - 1) / per), 64u << (D.l2s + D.l2w),
                      ((size_t)3 * D.rows * 4 * D.nb + 16 * 12) * sizeof(float)};
}

// LDS floats of the staged magnetisation.
__host__ __device__ __forceinline__ int direct_lds_floats(int nb, int rows) { return 3 * rows * 4 * nb; }

// Source of the sum: Ms m, plus Ms2 m2 when m2 is set.
struct DirectSource {
  const float* m;
  PS msat;
  const float* m2;
  PS msat2;
  const uint8_t* geom;
  size_t cs;  // component stride of m and m2
};

// Stages the source (zero outside the geometry and in the padding); the whole
// block calls it, and it ends with a block barrier.  The loads of four cells
// are issued together.
__device__ __forceinline__ void direct_stage(const DirectDesc& D, const DirectSource& S, float* lds) {
  const int row4 = 4 * D.nb, n = D.rows * row4;
  for (int e0 = threadIdx.x; e0 < n; e0 += 4 * blockDim.x) {
    float v[4][3];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = e0 + k * (int)blockDim.x;
      const int r = direct_div(e >> 2, D.nb, D.mag_nb), x = e - r * row4;
      const bool row = e < n && x < D.nx;
      const int i = row ? r * D.nx + x : 0;
      const bool in = row && (!S.geom || S.geom[i]);
      const float ms = S.msat.at(i), ms2 = S.m2 ? S.msat2.at(i) : 0.f;
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        float a = ms * S.m[c * S.cs + i];
        if (S.m2) a += ms2 * S.m2[c * S.cs + i];
        v[k][c] = in ? a : 0.f;
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int e = e0 + k * (int)blockDim.x;
      if (e < n)
#pragma unroll
        for (int c = 0; c < 3; ++c) lds[c * n + e] = v[k][c];
    }
  }
  __syncthreads();
}

// The field of block blk's strips, summed over the staged sources (lds) with
// `red` (192 floats of LDS after them) for the sums over wavefronts.  Every
// thread of the block calls it.  Returns true on the lanes l < 4 of the first
// wavefront of each strip, with the cell (index and field h); false on the
// others and for cells past the row or the last strip.
template <bool FLAT>
__device__ __forceinline__ bool direct_sum(const DirectDesc& D, const float* lds, float* red, int blk, int& cell,
                                           float3& h) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int row4 = 4 * D.nb, n = D.rows * row4;
  const int units = D.rows * D.nb;  // and strips
  const int strip = (blk << D.l2s) + (wave >> D.l2w), part = wave & ((1 << D.l2w) - 1);
  const int st = strip < units ? strip : 0;
  const int row = direct_div(st, D.nb, D.mag_nb), xb = st - row * D.nb;
  const int z = FLAT ? 0 : direct_div(row, D.ny, D.mag_ny), y = row - z * D.ny;
  float acc[12];
#pragma unroll
  for (int i = 0; i < 12; ++i) acc[i] = 0.f;
#pragma unroll 2
  for (int u0 = part << 6; u0 < units; u0 += 64 << D.l2w) {
    // lanes past the last unit read it again with zero sources
    const bool in = u0 + lane < units;
    const int u = in ? u0 + lane : units - 1;
    const int r = direct_div(u, D.nb, D.mag_nb), b = u - r * D.nb;
    const int zs = FLAT ? 0 : direct_div(r, D.ny, D.mag_ny), ys = r - zs * D.ny;
    const int dy = y - ys, dz = z - zs;
    const int ay = dy < 0 ? -dy : dy, az = dz < 0 ? -dz : dz;
    // entry of dx = 4 (xb - b) - 3
    const int k0 = (FLAT ? ay : az * D.ny + ay) * 2 * row4 + row4 + 4 * (xb - b) - 3;
    float4 k4[7];
    float2 k2[FLAT ? 1 : 7];
#pragma unroll
    for (int i = 0; i < 7; ++i) {
      k4[i] = D.K4[k0 + i];
      if constexpr (!FLAT) k2[i] = D.K2[k0 + i];
    }
    float4 s[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) s[c] = *reinterpret_cast<const float4*>(lds + c * n + 4 * u);
    const float sy = dy < 0 ? -1.f : 1.f, sz = dz < 0 ? -1.f : 1.f;
#pragma unroll
    for (int i = 0; i < 7; ++i) {
      k4[i].w *= sy;
      if constexpr (!FLAT) {
        k2[i].x *= sz;
        k2[i].y *= sy * sz;
      }
    }
    const float mx[4] = {in ? s[0].x : 0.f, in ? s[0].y : 0.f, in ? s[0].z : 0.f, in ? s[0].w : 0.f};
    const float my[4] = {in ? s[1].x : 0.f, in ? s[1].y : 0.f, in ? s[1].z : 0.f, in ? s[1].w : 0.f};
    const float mz[4] = {in ? s[2].x : 0.f, in ? s[2].y : 0.f, in ? s[2].z : 0.f, in ? s[2].w : 0.f};
#pragma unroll
    for (int o = 0; o < 4; ++o)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int i = o - j + 3;  // dx = 4 (xb - b) + o - j
        acc[3 * o] += k4[i].x * mx[j] + k4[i].w * my[j];
        acc[3 * o + 1] += k4[i].w * mx[j] + k4[i].y * my[j];
        acc[3 * o + 2] += k4[i].z * mz[j];
        if constexpr (!FLAT) {
          acc[3 * o] += k2[i].x * mz[j];
          acc[3 * o + 1] += k2[i].y * mz[j];
          acc[3 * o + 2] += k2[i].x * mx[j] + k2[i].y * my[j];
        }
      }
  }
  float a6[6];
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    const bool hi = lane & 1;
    const float keep = hi ? acc[6 + i] : acc[i], give = hi ? acc[i] : acc[6 + i];
    a6[i] = keep + __shfl_xor(give, 1, 64);
  }
  float a3[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const bool hi = lane & 2;
    const float keep = hi ? a6[3 + i] : a6[i], give = hi ? a6[i] : a6[3 + i];
    a3[i] = keep + __shfl_xor(give, 2, 64);
  }
#pragma unroll
  for (int off = 4; off < 64; off <<= 1)
#pragma unroll
    for (int i = 0; i < 3; ++i) a3[i] += __shfl_xor(a3[i], off, 64);
  // lane l < 4 holds the sum of strip cell 2 (l & 1) + (l >> 1)
  if (D.l2w > 0) {
    if (lane < 4)
#pragma unroll
      for (int i = 0; i < 3; ++i) red[wave * 12 + 3 * lane + i] = a3[i];
    __syncthreads();
    if (part == 0 && lane < 4)
      for (int w = 1; w < 1 << D.l2w; ++w)
#pragma unroll
        for (int i = 0; i < 3; ++i) a3[i] += red[(wave + w) * 12 + 3 * lane + i];
  }
  const int x = 4 * xb + 2 * (lane & 1) + (lane >> 1);
  cell = row * D.nx + x;
  h = f3(a3[0], a3[1], a3[2]);
  return part == 0 && lane < 4 && strip < units && x < D.nx;
}

}  // namespace mpa
