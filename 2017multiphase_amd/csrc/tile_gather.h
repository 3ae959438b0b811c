// Particles of a tile of 4 x 8 x 8 cells and the grid values they interpolate,
// staged in LDS, for particles in the order of the library's own sort (a row of
// cells along k is one range of particles).
//
// Interpolating from memory costs a wave four two-word gathers per field, each
// issued a few lanes at a time, whatever the caches hold; from LDS the same
// words come several times faster, and a tile's values are read once, row by
// row.  A particle whose eight corners are not all staged (it was moved, or
// lies off the grid) reads them from memory; the arithmetic is the same.
#pragma once
#include "interp.h"

namespace mpf {

constexpr int TG_X = 4, TG_Y = 8, TG_Z = 8, TG = TG_X * TG_Y * TG_Z;  // cells, threads
constexpr int TG_ROWS = TG_X * TG_Y;
// below this many particles a tile is not staged
constexpr uint32_t TG_LEAST = 256;
__host__ __device__ constexpr int tg_t(int d) { return d == 0 ? TG_X : (d == 1 ? TG_Y : TG_Z); }
// Staged values of a face field of axis A: faces [t0_d - (d != A), t0_d + T_d]
// along d; of a cell field (A = 3): cells [t0_d - 1, t0_d + T_d].
__host__ __device__ constexpr int tg_r(int A, int d) { return tg_t(d) + (d == A ? 1 : 2); }
__host__ __device__ constexpr int tg_n(int A) { return tg_r(A, 0) * tg_r(A, 1) * tg_r(A, 2); }

struct TileParticles {
  uint32_t start[TG_ROWS], before[TG_ROWS + 1];
};
// The tile at (x0, y0, z0); fills tp (LDS) and returns the number of particles
// in it.  All threads of the block call it.
__device__ __forceinline__ uint32_t tile_particles(const Grid& g, const uint32_t* __restrict__ cstart,
                                                   const uint32_t* __restrict__ cend, int x0, int y0, int z0,
                                                   TileParticles& tp) {
  const int b = threadIdx.x;
  const int ci = x0 + b / (TG_Y * TG_Z), cj = y0 + (b / TG_Z) % TG_Y, ck = z0 + b % TG_Z;
  uint32_t s = MPF_CELL_UNDEF, e = 0;
  if (ci < g.nx && cj < g.ny && ck < g.nz) {
    const int64_t c = cid(g, ci, cj, ck);
    s = cstart[c];
    e = s == MPF_CELL_UNDEF ? 0 : cend[c];
  }
#pragma unroll
  for (int o = 1; o < TG_Z; o <<= 1) {
    s = min(s, (uint32_t)__shfl_xor((int)s, o));
    e = max(e, (uint32_t)__shfl_xor((int)e, o));
  }
  if (b % TG_Z == 0) {
    tp.start[b / TG_Z] = s;
    tp.before[b / TG_Z + 1] = s < e ? e - s : 0u;
  }
  if (b == 0) tp.before[0] = 0;
  __syncthreads();
  if (b < 64) {
    uint32_t v = b < TG_ROWS ? tp.before[b + 1] : 0u;
#pragma unroll
    for (int o = 1; o < TG_ROWS; o <<= 1) {
      const uint32_t t = (uint32_t)__shfl_up((int)v, o);
      if (b >= o) v += t;
    }
    if (b < TG_ROWS) tp.before[b + 1] = v;
  }
  __syncthreads();
  return tp.before[TG_ROWS];
}
// Index of the tile's particle t.
__device__ __forceinline__ uint32_t tile_particle(const TileParticles& tp, uint32_t t) {
  int r = 0;
#pragma unroll
  for (int o = TG_ROWS / 2; o > 0; o >>= 1)
    if (tp.before[r + o] <= t) r += o;
  return tp.start[r] + (t - tp.before[r]);
}

// Stages the values of field u (axis A, or 3: cells) around the tile.
template <int A>
__device__ __forceinline__ void tile_stage(const Grid& g, const float* __restrict__ u, int x0, int y0, int z0, float* lds) {
  constexpr int R1 = tg_r(A, 1), R2 = tg_r(A, 2);
  const int n0 = g.nx + (A == 0), n1 = g.ny + (A == 1), n2 = g.nz + (A == 2);
  for (int q = threadIdx.x; q < tg_n(A); q += TG) {
    const int i = x0 - (A != 0) + q / (R1 * R2), j = y0 - (A != 1) + (q / R2) % R1, k = z0 - (A != 2) + q % R2;
    const bool in = i >= 0 && i < n0 && j >= 0 && j < n1 && k >= 0 && k < n2;
    lds[q] = in ? u[((int64_t)i * n1 + j) * n2 + k] : 0.0f;
  }
}
// Whether the corners of t are staged, and the first one's place.
template <int A>
__device__ __forceinline__ bool tile_at(const TriPos& t, int x0, int y0, int z0, int& at) {
  constexpr int R0 = tg_r(A, 0), R1 = tg_r(A, 1), R2 = tg_r(A, 2);
  const int i = t.i - (x0 - (A != 0)), j = t.j - (y0 - (A != 1)), k = t.k - (z0 - (A != 2));
  at = (i * R1 + j) * R2 + k;
  return (unsigned)i < (unsigned)(R0 - 1) && (unsigned)j < (unsigned)(R1 - 1) && (unsigned)k < (unsigned)(R2 - 1);
}
template <int A>
__device__ __forceinline__ float tile_sample(const float* lds, int at, const TriPos& t) {
  return tri_eval(lds + at, (int64_t)tg_r(A, 1) * tg_r(A, 2), tg_r(A, 2), t);
}

}  // namespace mpf
