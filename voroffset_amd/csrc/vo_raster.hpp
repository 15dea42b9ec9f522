// vo_raster.hpp -- mesh -> dexels on the GPU (gfx950).
//
// Replaces the ray casting of vor3d::create_dexels (Dexelize.cpp:166-225):
// for every dexel centre (origin_x + (x + 0.5) * spacing, origin_y + (y + 0.5)
// * spacing) (CompressedVolumeBase.cpp:5-11), the z / spacing of every
// triangle whose xy-projection contains it, sorted ascending; pairs of
// consecutive values are the dexel's segments (even-odd fill).  Containment is
// the SOS test of point_in_triangle_2d (Dexelize.cpp:56-92), and a triangle
// whose projection has zero inexact orientation contributes nothing
// (Dexelize.cpp:107-121,151-158).  The arithmetic follows the reference's
// operation order with FMA contraction off, so every decision and every z
// equals the CPU's bit for bit.
//
// Steps: (1) count, per 8x8-dexel tile, the triangles whose bounding box may
// contain one of its dexel centres; (2) scan; (3) fill the tile lists;
// (4) four wavefronts per tile, one lane of each per dexel: each wavefront
// stages its share of the tile's triangles in LDS and every lane tests its
// centre against them; the hits of a dexel are counted, and up to kRasterKeep
// of them kept, sorted; (5) scan the counts into the output offsets; (6) the
// kept hits are copied to their columns, and tiles with fuller columns are
// swept again and their columns sorted there.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vo_wave.hpp"

namespace vo {

constexpr int kRasterTile = 8;  // dexels per tile side (64 = one wavefront)

struct RasterGrid {
  int nx, ny;
  double ox, oy, spacing;
  int tx, ty;  // tiles per row / column
};

// Tile range of triangle f: dexel centres that may lie in its closed xy
// bounding box, widened by one dexel (pruning only; the SOS test decides).
__device__ __forceinline__ bool tri_tiles(const double* V, const int32_t* F, int64_t f, const RasterGrid& g,
                                          int& ax, int& bx, int& ay, int& by) {
#pragma clang fp contract(off)
  double lo[2] = {INFINITY, INFINITY}, hi[2] = {-INFINITY, -INFINITY};
  for (int k = 0; k < 3; ++k) {
    const int64_t v = F[3 * f + k];
    for (int d = 0; d < 2; ++d) {
      lo[d] = fmin(lo[d], V[3 * v + d]);
      hi[d] = fmax(hi[d], V[3 * v + d]);
    }
  }
  const double o[2] = {g.ox, g.oy};
  const int n[2] = {g.nx, g.ny};
  int il[2], ih[2];
  for (int d = 0; d < 2; ++d) {
    const double a = floor((lo[d] - o[d]) / g.spacing - 0.5) - 1.0;
    const double b = ceil((hi[d] - o[d]) / g.spacing - 0.5) + 1.0;
    il[d] = int(fmin(fmax(a, 0.0), double(n[d])));         // clamped before the conversion
    ih[d] = int(fmax(fmin(b, double(n[d] - 1)), -1.0));
  }
  if (il[0] > ih[0] || il[1] > ih[1]) return false;
  ax = il[0] / kRasterTile;
  bx = ih[0] / kRasterTile;
  ay = il[1] / kRasterTile;
  by = ih[1] / kRasterTile;
  return true;
}

// phase 0: count per tile; phase 1: fill (cursor starts at the tile offsets)
__global__ void raster_bin_kernel(const double* V, const int32_t* F, int64_t nf, RasterGrid g, int phase,
                                  int64_t* tile_cnt, int64_t* tile_cur, int64_t* tile_tris) {
  const int64_t f = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (f >= nf) return;
  int ax, bx, ay, by;
  if (!tri_tiles(V, F, f, g, ax, bx, ay, by)) return;
  for (int b = ay; b <= by; ++b)
    for (int a = ax; a <= bx; ++a) {
      const int64_t t = int64_t(b) * g.tx + a;
      if (phase == 0)
        atomicAdd(reinterpret_cast<unsigned long long*>(tile_cnt + t), 1ull);
      else
        tile_tris[atomicAdd(reinterpret_cast<unsigned long long*>(tile_cur + t), 1ull)] = f;
    }
}

__device__ __forceinline__ int sos_orientation(double x1, double y1, double x2, double y2, double& area) {
#pragma clang fp contract(off)
  area = y1 * x2 - x1 * y2;
  if (area > 0) return 1;
  if (area < 0) return -1;
  if (y2 > y1) return 1;
  if (y2 < y1) return -1;
  if (x1 > x2) return 1;
  if (x1 < x2) return -1;
  return 0;
}

// The hit of the vertical ray through (qx, qy) with triangle p (9 doubles:
// x1 y1 z1 x2 y2 z2 x3 y3 z3); returns false when it misses.
__device__ __forceinline__ bool ray_hit(const double* p, double qx, double qy, double& z) {
#pragma clang fp contract(off)
  const double x1 = p[0] - qx, y1 = p[1] - qy;
  const double x2 = p[3] - qx, y2 = p[4] - qy;
  const double x3 = p[6] - qx, y3 = p[7] - qy;
  double a, b, c;
  const int sa = sos_orientation(x2, y2, x3, y3, a);
  if (sa == 0) return false;
  if (sos_orientation(x3, y3, x1, y1, b) != sa) return false;
  if (sos_orientation(x1, y1, x2, y2, c) != sa) return false;
  const double sum = a + b + c;
  a /= sum;
  b /= sum;
  c /= sum;
  z = a * p[2] + b * p[5] + c * p[8];
  const double a11 = p[3] - p[0], a12 = p[4] - p[1];
  const double a21 = p[6] - p[0], a22 = p[7] - p[1];
  const double delta = a11 * a22 - a12 * a21;
  return delta != 0;
}

constexpr int kRasterWaves = 4;   // wavefronts per tile
constexpr int kRasterPiece = 21;  // triangles a wavefront stages: a lane a vertex
constexpr int kRasterKeep = 8;    // hits kept per dexel between the phases
// Tiles up to which hits are kept (4 KB a tile: 256 MB).
constexpr int64_t kRasterKeepTiles = 65536;

// phase 0: per-dexel hit counts into len[col], and the hits of tiles with at
// most kRasterKeep a dexel, sorted, into keep (hit i of lane L of tile t at
// (t * kRasterKeep + i) * 64 + L; null: not kept); phase 1: hits into
// out[off[col] ..], each column sorted.
//
// A chain per tile bounds it: triangle after triangle, with the tiles on a
// mesh's filigree holding hundreds of them and most tiles none (one wavefront
// a tile and a second full sweep: 2 x 112 us for 2000 tubes on 544^2).  So
// four wavefronts share a tile, the next triangles' vertices are fetched
// while the current ones are tested, and the second sweep is left out where
// the hits were kept: 224 -> 119 us for both phases.
__global__ __launch_bounds__(kWave* kRasterWaves) void raster_cast_kernel(const double* V, const int32_t* F, RasterGrid g,
                                                                          const int64_t* tile_off,
                                                                          const int64_t* tile_tris, int phase,
                                                                          int64_t* len, const int64_t* off,
                                                                          double* keep, double* out) {
#pragma clang fp contract(off)
  __shared__ double tri[kRasterWaves][kRasterPiece * 9];
  __shared__ double hit[kRasterKeep * kWave];
  __shared__ unsigned int found[kWave];
  const int L = threadIdx.x % kWave, w = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int64_t t = blockIdx.x;
  const int x = int(t % g.tx) * kRasterTile + (L % kRasterTile);
  const int y = int(t / g.tx) * kRasterTile + (L / kRasterTile);
  const bool active = x < g.nx && y < g.ny;
  const double qx = (x + 0.5) * g.spacing + g.ox, qy = (y + 0.5) * g.spacing + g.oy;
  const int64_t col = int64_t(x) + int64_t(g.nx) * y;
  const int64_t t0 = tile_off[t], t1 = tile_off[t + 1];
  const int64_t base = (phase == 1 && active) ? off[col] : 0;
  if (phase == 1) {
    const int64_t n = active ? off[col + 1] - base : 0;
    if (keep && !__any(n > kRasterKeep)) {  // (the same columns in every wavefront)
      for (int i = w; i < kRasterKeep; i += kRasterWaves)
        if (i < n) out[base + i] = keep[(t * kRasterKeep + i) * kWave + L];
      return;
    }
  }
  if (w == 0) found[L] = 0;
  double v[3] = {0, 0, 0};
  auto fetch = [&](int64_t c) {  // this lane's vertex of the wavefront's piece at c
    const int64_t k = c + L / 3;
    if (L < 3 * kRasterPiece && k < t1) {
      const int64_t p = F[3 * tile_tris[k] + L % 3];
      for (int d = 0; d < 3; ++d) v[d] = V[3 * p + d];
    }
  };
  constexpr int kStep = kRasterWaves * kRasterPiece;
  fetch(t0 + w * kRasterPiece);
  for (int64_t c0 = t0; c0 < t1; c0 += kStep) {
    const int64_t c = c0 + w * kRasterPiece;
    const int cnt = int(max(int64_t(0), min(int64_t(kRasterPiece), t1 - c)));
    if (L < 3 * kRasterPiece)
      for (int d = 0; d < 3; ++d) tri[w][3 * L + d] = v[d];
    __syncthreads();
    fetch(c + kStep);
    if (active) {
      for (int i = 0; i < cnt; ++i) {
        double z;
        if (ray_hit(tri[w] + 9 * i, qx, qy, z)) {
          const unsigned int n = atomicAdd(&found[L], 1u);
          if (phase == 1)
            out[base + n] = z / g.spacing;
          else if (n < kRasterKeep)
            hit[n * kWave + L] = z / g.spacing;
        }
      }
    }
    __syncthreads();
  }
  if (t0 >= t1) __syncthreads();  // (found, set above)
  if (w != 0) return;
  const int64_t n = active ? int64_t(found[L]) : 0;
  if (phase == 0 && active) len[col] = n;
  if (phase == 0 && (!keep || __any(n > kRasterKeep))) return;
  // insertion sort of the column (columns hold few hits)
  auto sort = [n](double* c, int64_t step) {
    for (int64_t i = 1; i < n; ++i) {
      const double a = c[i * step];
      int64_t j = i - 1;
      while (j >= 0 && c[j * step] > a) {
        c[(j + 1) * step] = c[j * step];
        --j;
      }
      c[(j + 1) * step] = a;
    }
  };
  if (phase == 0) {
    sort(hit + L, kWave);
    for (int64_t i = 0; i < n; ++i) keep[(t * kRasterKeep + i) * kWave + L] = hit[i * kWave + L];
  } else if (active) {
    sort(out + base, 1);
  }
}

}  // namespace vo
