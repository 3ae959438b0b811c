// Grid-side kernels: level set + redistancing + cell flags (a6-a8), P2G
// (a9), extrapolation and wall conditions (a10), two-phase divergence (a11),
// pressure gradient (a13), heat grid stages (a16), marching cubes (a18) and
// the solid distance/velocity fields used by the collision advection (a15).
#include "mpf_internal.h"
#include "interp.h"
#include "row_bits.h"

#include <algorithm>
#include <cmath>
#include <vector>

#include "mc_tables.inc"

namespace mpf {

namespace {

__device__ __forceinline__ f3 mk3(float x, float y, float z) { return f3{x, y, z}; }
__device__ __forceinline__ f3 sub3(f3 a, f3 b) { return mk3(a.x - b.x, a.y - b.y, a.z - b.z); }
__device__ __forceinline__ float dot3(f3 a, f3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }

// a / d for the sharp kernel of the tile scatters: the hardware reciprocal
// and one Newton-Raphson correction of the quotient (Markstein's step,
// residual by fma), within an ulp of the IEEE quotient for d >= 1e-4.
__device__ __forceinline__ float div_nr(float a, float d) {
  const float y = __builtin_amdgcn_rcpf(d);
  const float q = a * y;
  const float r = fmaf(-d, q, a);
  return fmaf(r, y, q);
}

#define CELL_LOOP_HEAD                                           \
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; \
  if (idx >= g.G) return;                                        \
  int i, j, k;                                                   \
  ijk_of(g, idx, i, j, k);

// ---------------- level set (a6) ----------------
// genlevelset + mindis_cell, spray_k.cu:2753-2806.  The minimum is taken over
// squared distances and square-rooted once: sqrt is correctly rounded and
// monotone, so sqrt(min d^2) == min sqrt(d^2) bit for bit.  The 5x5x5 window
// is visited in rings of increasing lower bound on the distance from the cell
// centre to any point of a ring cell (sum over axes of max(0,|d|-1/2)^2, in
// h^2); a phase stops once its minimum is below the next ring's bound (with a
// 0.1% margin for rounding), and the 8 corner cells (bound 6.75 h^2 > 2.5^2)
// can never beat the initial 2.5h.  The result equals the full-window minimum.
// The window's 125 cells are bits (25 di + 5 dj + dk, offsets from 0) of two
// words; ring r is the cells set in m[r], its bound lb[r] in h^2 units.
struct Rings {
  uint64_t m[9][2];
  float lb[9];
};
constexpr Rings make_rings() {
  constexpr float lbs[9] = {0.0f, 0.25f, 0.5f, 0.75f, 2.25f, 2.5f, 2.75f, 4.5f, 4.75f};
  Rings r{};
  for (int q = 0; q < 9; ++q) r.lb[q] = lbs[q];
  for (int b = 0; b < 125; ++b) {
    const int d[3] = {b / 25 - 2, (b / 5) % 5 - 2, b % 5 - 2};
    float lb = 0;
    for (int a = 0; a < 3; ++a) {
      const float v = (float)(d[a] < 0 ? -d[a] : d[a]) - 0.5f;
      if (v > 0) lb += v * v;  // multiples of 1/4: exact
    }
    for (int q = 0; q < 9; ++q)
      if (lb == lbs[q]) r.m[q][b >> 6] |= 1ull << (b & 63);
  }
  return r;
}
__constant__ Rings c_rings = make_rings();

__global__ void k_row_bits(Grid g, const uint8_t* __restrict__ cmask, uint64_t* __restrict__ fb,
                           uint64_t* __restrict__ ab, int nw, uint32_t* __restrict__ odd) {
  const int64_t w = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;  // a wave per word
  if (blockIdx.x == 0 && threadIdx.x == 0) *odd = 0;
  if (w >= (int64_t)(g.nx + 4) * (g.ny + 4) * nw) return;
  const int64_t row = w / nw;
  const int i = (int)(row / (g.ny + 4)) - 2, j = (int)(row % (g.ny + 4)) - 2;
  const int k = (int)(w % nw) * 64 + (int)__lane_id() - 2;
  const uint8_t m = valid(g, i, j, k) ? cmask[cid(g, i, j, k)] : (uint8_t)0;
  const uint64_t f = __ballot(m & M_FLUIDSOLID), a = __ballot(m & (M_AIR | M_AIRSOLO));
  if (__lane_id() == 0) {
    fb[w] = f;
    ab[w] = a;
  }
}
// *odd = 1 if an air particle's position, velocity or mass is not finite or its
// position lies off the grid (it is then listed in a cell it is not in).
__global__ void k_air_regular(Grid g, int64_t P, const f3* __restrict__ pos, const f3* __restrict__ vel,
                              const float* __restrict__ mass, const int8_t* __restrict__ flag,
                              uint32_t* __restrict__ odd) {
  const int64_t p0 = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 16;
  if (p0 >= P) return;
  int8_t fl[16];
  if (p0 + 16 <= P) __builtin_memcpy(fl, __builtin_assume_aligned(flag + p0, 16), 16);
  else
    for (int u = 0; u < 16; ++u) fl[u] = p0 + u < P ? flag[p0 + u] : (int8_t)-1;
  bool air = false;
#pragma unroll
  for (int u = 0; u < 16; ++u) air = air || fl[u] == AIR;
  if (!air) return;
  const float lim = 3.4e38f;
  bool bad = false;
#pragma unroll
  for (int u = 0; u < 16; ++u) {
    if (fl[u] != AIR) continue;
    const f3 x = pos[p0 + u], v = vel[p0 + u];
    const float qx = (x.x - g.gx0) / g.h, qy = (x.y - g.gy0) / g.h, qz = (x.z - g.gz0) / g.h;
    const bool in = qx >= 0 && qx < (float)g.nx && qy >= 0 && qy < (float)g.ny && qz >= 0 && qz < (float)g.nz;
    const bool fin = fabsf(v.x) < lim && fabsf(v.y) < lim && fabsf(v.z) < lim && fabsf(mass[p0 + u]) < lim;
    bad = bad || !in || !fin;
  }
  if (bad) *odd = 1;
}

// The 125 bits of the window around (i, j, k).
__device__ __forceinline__ void window_bits(const uint64_t* __restrict__ rows, const RowBits& rb, int i, int j, int k,
                                            uint64_t& lo, uint64_t& hi) {
  uint32_t w[5];
#pragma unroll
  for (int di = 0; di < 5; ++di) {
    w[di] = 0;
    __builtin_amdgcn_sched_barrier(0);  // five reads in flight, not 25 addresses in registers
#pragma unroll
    for (int dj = 0; dj < 5; ++dj) w[di] |= row_window(rows, rb, i + di, j + dj, k) << (5 * dj);
  }
  lo = (uint64_t)w[0] | (uint64_t)w[1] << 25 | (uint64_t)w[2] << 50;
  hi = (uint64_t)(w[2] >> 14) | (uint64_t)w[3] << 11 | (uint64_t)w[4] << 36;
}

// Phases present in each 4x4x4 brick of cells (OR of the occupancy masks),
// then, per brick, in the 3x3x3 bricks around it: a superset of the phases
// in the 5x5x5 window of any cell of the brick.
__global__ void k_brick_or(Grid g, const uint8_t* __restrict__ cmask, uint8_t* __restrict__ bm, int bx, int by,
                           int bz) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= (int64_t)bx * by * bz) return;
  const int bk = (int)(b % bz), bj = (int)((b / bz) % by), bi = (int)(b / ((int64_t)by * bz));
  uint8_t m = 0;
  for (int di = 0; di < 4; ++di)
    for (int dj = 0; dj < 4; ++dj)
      for (int dk = 0; dk < 4; ++dk) {
        const int ci = 4 * bi + di, cj = 4 * bj + dj, ck = 4 * bk + dk;
        if (valid(g, ci, cj, ck)) m |= cmask[cid(g, ci, cj, ck)];
      }
  bm[b] = m;
}
__global__ void k_brick_dilate(const uint8_t* __restrict__ bm, uint8_t* __restrict__ dm, int bx, int by, int bz) {
  const int64_t b = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= (int64_t)bx * by * bz) return;
  const int bk = (int)(b % bz), bj = (int)((b / bz) % by), bi = (int)(b / ((int64_t)by * bz));
  uint8_t m = 0;
  for (int di = -1; di <= 1; ++di)
    for (int dj = -1; dj <= 1; ++dj)
      for (int dk = -1; dk <= 1; ++dk) {
        const int i = bi + di, j = bj + dj, k = bk + dk;
        if (i >= 0 && i < bx && j >= 0 && j < by && k >= 0 && k < bz) m |= bm[((int64_t)i * by + j) * bz + k];
      }
  dm[b] = m;
}

// A phase absent from the cell's brick neighbourhood is absent from its
// window: its search is skipped, with the same result (the 2.5h cap).  Inside
// the liquid a cell's own particles, or those across its faces, decide; near
// a surface or a bubble the window is searched for the other phase, mostly in
// vain, so the cells that hold it are found as bits first.  Testing the mask
// of each of the 117 cells took 0.76 ms at 128^3 with 8 bubbles, now 0.41;
// 256^3 without air 1.7 -> 1.26 ms (one address for eight particles' loads).
__global__ void __launch_bounds__(256, 8) k_genlevelset(Grid g, const f3* __restrict__ pos, const int8_t* __restrict__ flag,
                              const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
                              const uint8_t* __restrict__ cmask, const uint8_t* __restrict__ dm, RowBits rb,
                              float* __restrict__ lsfluid, float* __restrict__ lsair, int8_t* __restrict__ mark) {
  const int64_t idx = xcd_block() * blockDim.x + threadIdx.x;  // XCD-contiguous cells
  if (idx >= g.G) return;
  int i, j, k;
  ijk_of(g, idx, i, j, k);
  const float h = g.h;
  mark[idx] = VACUUM;
  float r = 0.5f * h;
  f3 gp = mk3(((float)i + 0.5f) * h + g.gx0, ((float)j + 0.5f) * h + g.gy0, ((float)k + 0.5f) * h + g.gz0);
  float ma2 = INFINITY, mf2 = INFINITY;
  const float h2 = h * h;
  const int by = (g.ny + 3) / 4, bz = (g.nz + 3) / 4;
  const uint8_t near = dm[((int64_t)(i >> 2) * by + (j >> 2)) * bz + (k >> 2)];
  const bool has_f = (near & M_FLUIDSOLID) != 0, has_a = (near & (M_AIR | M_AIRSOLO)) != 0;
  // particles [s, e), eight at a time, their loads issued together from one
  // address (the arrays are eight longer than their particles; what lies past
  // the range is dropped)
  auto visit = [&](uint32_t s, uint32_t e) {
    for (uint32_t p = s; p < e; p += 8) {
      const f3* __restrict__ xp = pos + p;
      f3 x[8];
      uint32_t fw[2];
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = xp[u];
      __builtin_memcpy(fw, flag + p, 8);
      const uint32_t n = e - p;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const f3 d = sub3(x[u], gp);
        const float d2 = (uint32_t)u < n ? dot3(d, d) : INFINITY;
        const uint32_t fl = (fw[u >> 2] >> (8 * (u & 3))) & 0xffu;
        ma2 = (fl == AIR || fl == AIRSOLO) ? fminf(ma2, d2) : ma2;
        mf2 = (fl == FLUID || fl == SOLID) ? fminf(mf2, d2) : mf2;
      }
    }
  };
  const uint8_t own = cmask[idx];
  if (own) visit(cstart[idx], cend[idx]);
  const int64_t sx = (int64_t)g.ny * g.nz;
  // up to N ranges, one copy of the visit: the ranges move up
  auto visit_all = [&](auto& S, auto& E) {
    constexpr int N = sizeof(S) / sizeof(S[0]);
#pragma unroll 1
    for (int w = 0; w < N; ++w) {
      if (S[0] < E[0]) visit(S[0], E[0]);
#pragma unroll
      for (int v = 0; v + 1 < N; ++v) {
        S[v] = S[v + 1];
        E[v] = E[v + 1];
      }
    }
  };
  // ring 1, the cells across the six faces, read directly: inside the liquid
  // a few cells of every wave go this far, and none further
  {
    const float lb = 0.999f * c_rings.lb[1] * h2;
    const bool need_f = has_f && mf2 > lb, need_a = has_a && ma2 > lb;
    const uint8_t want = (need_f ? M_FLUIDSOLID : 0) | (need_a ? (M_AIR | M_AIRSOLO) : 0);
    if (want) {
      uint32_t S[6], E[6];
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        const int ax = f >> 1, d = (f & 1) ? 1 : -1;
        const int n = ax == 0 ? i : (ax == 1 ? j : k), lim = ax == 0 ? g.nx : (ax == 1 ? g.ny : g.nz);
        const bool v = (unsigned)(n + d) < (unsigned)lim;
        const int64_t c = idx + (v ? d * (ax == 0 ? sx : (ax == 1 ? (int64_t)g.nz : (int64_t)1)) : 0);
        const uint8_t m = cmask[c];
        S[f] = cstart[c];
        E[f] = cend[c];
        if (!(v && (m & want))) E[f] = 0;
      }
      visit_all(S, E);
    }
  }
  // the further rings, over the cells that hold a needed phase
  uint64_t fw[2] = {0, 0}, aw[2] = {0, 0};
  {
    const float lb = 0.999f * c_rings.lb[2] * h2;
    if (has_f && mf2 > lb) window_bits(rb.f, rb, i, j, k, fw[0], fw[1]);
    if (has_a && ma2 > lb) window_bits(rb.a, rb, i, j, k, aw[0], aw[1]);
  }
  for (int ring = 2; ring < 9; ++ring) {
    const float lb = 0.999f * c_rings.lb[ring] * h2;
    const bool need_f = has_f && mf2 > lb, need_a = has_a && ma2 > lb;
    if (!need_f && !need_a) break;
    uint64_t lo = ((need_f ? fw[0] : 0) | (need_a ? aw[0] : 0)) & c_rings.m[ring][0];
    uint64_t hi = ((need_f ? fw[1] : 0) | (need_a ? aw[1] : 0)) & c_rings.m[ring][1];
    // four cells at a time: their ranges read together
    while (lo | hi) {
      uint32_t S4[4], E4[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const bool any = (lo | hi) != 0, first = lo != 0;
        const uint64_t v = first ? lo : hi;
        const uint32_t b = any ? (uint32_t)(__ffsll((unsigned long long)v) - 1) + (first ? 0u : 64u) : 62u;
        if (first) lo &= lo - 1;
        else if (any) hi &= hi - 1;
        const uint32_t di = (b * 41u) >> 10, r = b - 25u * di, dj = (r * 13u) >> 6, dk = r - 5u * dj;
        const int64_t c = idx + ((int)di - 2) * sx + ((int)dj - 2) * g.nz + ((int)dk - 2);  // 62: the cell itself
        S4[w] = cstart[c];
        E4[w] = any ? cend[c] : 0u;
      }
      visit_all(S4, E4);
    }
  }
  float mair = 2.5f * h, mfl = 2.5f * h;
  float da = sqrtf(ma2), df = sqrtf(mf2);
  mair = (da < mair) ? da : mair;
  mfl = (df < mfl) ? df : mfl;
  lsfluid[idx] = mfl - r;
  lsair[idx] = mair - r;
}

// markLS_bigpositive spray_k.cu:3683-3697 (outward, from the distances) /
// setLSback_bigpositive and preparels 3699-3722 (inward, from the outward
// result; the distances between are not kept: the inward passes write all of
// ls), of both level sets.
struct LsPair {
  float* ls[2];
  float* out[2];
  int8_t* mark[2];
};
template <bool INWARD>
__global__ void k_ls_prepare(int64_t G, LsPair p, float h) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= G) return;
  const float* __restrict__ ls = blockIdx.y ? p.ls[1] : p.ls[0];
  float* __restrict__ out = blockIdx.y ? p.out[1] : p.out[0];
  int8_t* __restrict__ mark = blockIdx.y ? p.mark[1] : p.mark[0];
  float v = ls[idx];
  if (!INWARD) {
    v = v / h;
    if (v > 1.99f) { v = 5.0f; mark[idx] = AIR; }
    else mark[idx] = FLUID;
  } else {
    v = -(v * h) / h;
    if (v > 0) { v = 5.0f; mark[idx] = AIR; }
    else mark[idx] = FLUID;
  }
  out[idx] = v;
}

// One triple of solvedistance (spray_k.cu:746-754: d = min(a,b,c) + 1, or
// (a + b + c + sqrt(3 - (a-b)^2 - (a-c)^2 - (b-c)^2)) / 3 when that d exceeds
// max(a,b,c); x = min(x, d)) with the division of its three-axis branch left
// out: those candidates enter x only through a minimum and x/3 rounded
// to nearest is non-decreasing in x, so the smallest numerator s divided once
// at the end (solvedistance_end) gives the same float as dividing each.
__device__ __forceinline__ void solvedistance_acc(float a, float b, float c, float& x, float& s) {
  const float d = fminf(a, fminf(b, c)) + 1.0f;
  if (d > fmaxf(a, fmaxf(b, c)))
    s = fminf(s, a + b + c + sqrtf(3.0f - (a - b) * (a - b) - (a - c) * (a - c) - (b - c) * (b - c)));
  else if (d < x)
    x = d;
}
__device__ __forceinline__ void solvedistance_end(float s, float& x) {
  const float d = s / 3.0f;  // infinity when no triple took the branch
  if (d < x) x = d;
}
// sweepphibytype (spray_k.cu:771-789) / sweepphi (755-770, typeflag < 0), two
// buffers, on 1 x SW_J x SW_K cell tiles of one wave's cells (lane = row *
// SW_K + column), with change flags.  A Jacobi pass changes a cell only when
// a value of its 7-point neighbourhood changed in the pass before.  cur[tile]
// records which cells of the tile got a smaller value: SF_ANY for any, and
// the j-low, j-high, k-low and k-high bits for a change on that face of the
// tile.  A tile whose own flags, those of its x neighbours and the facing bits
// of its y and z neighbours of the previous pass (prev) are clear would
// recompute its previous values, which the output buffer (the previous pass's
// input) already holds, so it is skipped and gets a clear flag.  The first
// pass of a series (prev == nullptr) computes every tile.  A wave owns
// SW_L consecutive tiles: its first SW_L lanes read their flags together and
// the wave then visits the active ones.
constexpr uint8_t SF_ANY = 1, SF_JLO = 2, SF_JHI = 4, SF_KLO = 8, SF_KHI = 16;
constexpr int SW_L = 16;
constexpr int SW_U1 = 4;
static_assert(SW_J * SW_K == 64 && SW_L <= 64, "one wave's cells per eikonal tile");
// whether tile t (of a ntx x ntj x ntk tile grid, x slowest) must be computed:
// always without previous flags, else when it or an x neighbour changed or a
// y or z neighbour changed on the facing side (the seven flags are read
// together: indices clamped, then masked)
__device__ __forceinline__ bool tile_active(const uint8_t* __restrict__ prev, uint32_t t, bool mine, uint32_t ntj,
                                            uint32_t ntk, uint32_t ntx) {
  if (!mine) return false;
  if (!prev) return true;
  const uint32_t sxt = ntj * ntk;
  const uint32_t tk = t % ntk, tj = (t / ntk) % ntj, i = t / sxt;
  const uint8_t f0 = prev[t];
  const uint8_t fx0 = prev[i > 0 ? t - sxt : t], fx1 = prev[i + 1 < ntx ? t + sxt : t];
  const uint8_t fy0 = prev[tj > 0 ? t - ntk : t], fy1 = prev[tj + 1 < ntj ? t + ntk : t];
  const uint8_t fz0 = prev[tk > 0 ? t - 1 : t], fz1 = prev[tk + 1 < ntk ? t + 1 : t];
  const int a = (f0 & SF_ANY) | ((i > 0) ? (fx0 & SF_ANY) : 0) | ((i + 1 < ntx) ? (fx1 & SF_ANY) : 0) |
                ((tj > 0) ? (fy0 & SF_JHI) : 0) | ((tj + 1 < ntj) ? (fy1 & SF_JLO) : 0) |
                ((tk > 0) ? (fz0 & SF_KHI) : 0) | ((tk + 1 < ntk) ? (fz1 & SF_KLO) : 0);
  return a != 0;
}
// the flags of a tile from its lanes' change bits (lane = row * SW_K + column)
__device__ __forceinline__ uint8_t tile_flags(bool changed) {
  const uint64_t bal = __ballot(changed);
  constexpr uint64_t JLO = (1ull << SW_K) - 1, JHI = JLO << (64 - SW_K);
  constexpr uint64_t KLO = 0x0001000100010001ull, KHI = KLO << (SW_K - 1);
  static_assert(SW_K == 16 && SW_J == 4, "face masks of a 4 x 16 tile");
  return (uint8_t)((bal ? SF_ANY : 0) | ((bal & JLO) ? SF_JLO : 0) | ((bal & JHI) ? SF_JHI : 0) |
                   ((bal & KLO) ? SF_KLO : 0) | ((bal & KHI) ? SF_KHI : 0));
}
// One pass over one field, or over two at once (blockIdx.y): most passes of a
// series find few tiles to compute and cost little more than their launch.
struct SweepPass {
  const float* in;
  float* out;
  const int8_t* mark;
  int typeflag;
  const uint8_t* prev;
  uint8_t* cur;
};
__global__ void __launch_bounds__(256)
    k_sweep(Grid g, SweepPass p0, SweepPass p1, uint32_t ntj, uint32_t ntk, uint32_t ntiles) {
  const bool second = blockIdx.y != 0;
  const float* __restrict__ in = second ? p1.in : p0.in;
  float* __restrict__ out = second ? p1.out : p0.out;
  const int8_t* __restrict__ mark = second ? p1.mark : p0.mark;
  const int typeflag = second ? p1.typeflag : p0.typeflag;
  const uint8_t* __restrict__ prev = second ? p1.prev : p0.prev;
  uint8_t* __restrict__ cur = second ? p1.cur : p0.cur;
  const uint32_t t0 = (blockIdx.x * 4u + threadIdx.x / 64u) * SW_L;
  if (t0 >= ntiles) return;
  const int lane = threadIdx.x & 63;
  const uint32_t sxt = ntj * ntk;
  const uint32_t tl = t0 + lane;
  const bool mine = lane < SW_L && tl < ntiles;
  const bool act = tile_active(prev, tl, mine, ntj, ntk, (uint32_t)g.nx);
  uint64_t todo = __ballot(act);
  uint8_t myflag = 0;
  const int jl = lane / SW_K, kl = lane % SW_K;
  const int64_t sx = (int64_t)g.ny * g.nz, sy = g.nz;
  while (todo) {
    const int q = __builtin_ctzll(todo);
    todo &= todo - 1;
    const uint32_t t = t0 + q;
    const int tk = (int)(t % ntk), tj = (int)((t / ntk) % ntj), i = (int)(t / sxt);
    const int j = tj * SW_J + jl, k = tk * SW_K + kl;
    bool changed = false;
    if (j < g.ny && k < g.nz) {
      const int64_t idx = ((int64_t)i * g.ny + j) * g.nz + k;
      // the cell, its mark and its six neighbours (x-, x+, y-, y+, z-, z+)
      // are loaded together (a neighbour outside the grid reads the cell
      // itself and is replaced by infinity)
      const bool vx0 = i > 0, vx1 = i < g.nx - 1, vy0 = j > 0, vy1 = j < g.ny - 1, vz0 = k > 0, vz1 = k < g.nz - 1;
      const float c0 = in[idx];
      float res = c0;
      const int8_t m = (typeflag >= 0) ? mark[idx] : (int8_t)0;
      const float lx0 = in[vx0 ? idx - sx : idx], lx1 = in[vx1 ? idx + sx : idx];
      const float ly0 = in[vy0 ? idx - sy : idx], ly1 = in[vy1 ? idx + sy : idx];
      const float lz0 = in[vz0 ? idx - 1 : idx], lz1 = in[vz1 ? idx + 1 : idx];
      if (!(typeflag >= 0 && m == typeflag)) {
        const float nx0 = vx0 ? lx0 : INFINITY, nx1 = vx1 ? lx1 : INFINITY;
        const float ny0 = vy0 ? ly0 : INFINITY, ny1 = vy1 ? ly1 : INFINITY;
        const float nz0 = vz0 ? lz0 : INFINITY, nz1 = vz1 ? lz1 : INFINITY;
        // an update needs a neighbour below the current value (every
        // candidate is at least min(a, b, c)), so cells without one keep
        // their value without evaluating the 8 triples
        const float mn = fminf(fminf(fminf(nx0, nx1), fminf(ny0, ny1)), fminf(nz0, nz1));
        if (mn < res) {
          float s3 = INFINITY;
          for (int di = -1; di <= 1; di += 2)
            for (int dj = -1; dj <= 1; dj += 2)
              for (int dk = -1; dk <= 1; dk += 2)
                if ((di < 0 ? vx0 : vx1) && (dj < 0 ? vy0 : vy1) && (dk < 0 ? vz0 : vz1))
                  solvedistance_acc(di < 0 ? nx0 : nx1, dj < 0 ? ny0 : ny1, dk < 0 ? nz0 : nz1, res, s3);
          solvedistance_end(s3, res);
        }
      }
      // res only ever takes strictly smaller values: unchanged means bitwise equal
      changed = res < c0;
      out[idx] = res;
    }
    const uint8_t f = tile_flags(changed);
    if (lane == q) myflag = f;
  }
  if (mine) cur[tl] = myflag;
}

// setLSback spray_k.cu:3724-3731 of both level sets, and mergeLSAndMarkGrid
// 3733-3777
__global__ void k_merge(Grid g, float* __restrict__ lsfluid, float* __restrict__ lsair, float* __restrict__ lsmerge,
                        int8_t* __restrict__ mark) {
  CELL_LOOP_HEAD
  const float h = g.h;
  float lf = -lsfluid[idx] * h, la = -lsair[idx] * h, lm;
  lsfluid[idx] = lf;
  lsair[idx] = la;
  int8_t m;
  if (la > 4.99f * h) { lm = lf; m = (lf > 0) ? VACUUM : FLUID; }
  else if (lf > 4.99f * h) { lm = la; m = (la > 0) ? VACUUM : AIR; }
  else if (la > 0.8f * h && lf > 0.8f * h) { m = VACUUM; lm = fminf(lf, la); }
  else { lm = (lf - la) * 0.5f; m = (lm > 0) ? AIR : FLUID; }
  if (i == 0 || i == g.nx - 1 || j == 0 || j == g.ny - 1 || k == 0 || k == g.nz - 1) {
    m = BOUNDARY;
    lm = -0.5f * h;
  }
  lsmerge[idx] = lm;
  mark[idx] = m;
}

// computePhigra spray_k.cu:3994-4019
__global__ void k_phigrad(Grid g, const float* __restrict__ ls, float* __restrict__ gx, float* __restrict__ gy,
                          float* __restrict__ gz) {
  CELL_LOOP_HEAD
  float c0 = ls[idx];
  float x1 = valid(g, i + 1, j, k) ? ls[cid(g, i + 1, j, k)] : c0;
  float x0 = valid(g, i - 1, j, k) ? ls[cid(g, i - 1, j, k)] : c0;
  float y1 = valid(g, i, j + 1, k) ? ls[cid(g, i, j + 1, k)] : c0;
  float y0 = valid(g, i, j - 1, k) ? ls[cid(g, i, j - 1, k)] : c0;
  float z1 = valid(g, i, j, k + 1) ? ls[cid(g, i, j, k + 1)] : c0;
  float z0 = valid(g, i, j, k - 1) ? ls[cid(g, i, j, k - 1)] : c0;
  gx[idx] = ((x1 - x0) * 0.5f) / g.h;
  gy[idx] = ((y1 - y0) * 0.5f) / g.h;
  gz[idx] = ((z1 - z0) * 0.5f) / g.h;
}

// markfluid_dense + markBoundaryCell spray_k.cu:506-545 (all cells)
__global__ void k_mark_counts(Grid g, const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
                              const int8_t* __restrict__ flag, int8_t* __restrict__ mark) {
  CELL_LOOP_HEAD
  int cfs = 0, ca = 0;
  uint32_t s = cstart[idx];
  if (s != MPF_CELL_UNDEF)
    for (uint32_t p = s; p < cend[idx]; ++p) {
      int8_t f = flag[p];
      if (f == FLUID || f == SOLID) cfs++;
      else if (f == AIR) ca++;
    }
  int8_t m = (cfs == 0 && ca == 0) ? VACUUM : (cfs > ca ? FLUID : AIR);
  if (i == 0 || i == g.nx - 1 || j == 0 || j == g.ny - 1 || k == 0 || k == g.nz - 1) m = BOUNDARY;
  mark[idx] = m;
}

// Solid constraint: non-boundary cells whose particles are at least half SOLID.
__global__ void k_mark_solid(Grid g, const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
                             const int8_t* __restrict__ flag, const uint8_t* __restrict__ cmask,
                             int8_t* __restrict__ mark) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= g.G) return;
  if (!(cmask[idx] & M_SOLID) || mark[idx] == BOUNDARY) return;
  int cs = 0, co = 0;
  for (uint32_t p = cstart[idx]; p < cend[idx]; ++p) {
    if (flag[p] == SOLID) cs++;
    else co++;
  }
  if (cs > 0 && cs >= co) mark[idx] = SOLID;
}

// ---------------- P2G (a9) ----------------
// Air P2G: mapvelp2g_k_air with sumcell_* and sharp_kernel, spray_k.cu:255-258,
// 2809-2937.  One thread per face, the three axes in one launch; window normal
// [-2,1] x transverse [-2,2], in the reference's order.  Faces without air in
// the bricks around them are done at once; the others are few (bubbles) and
// walk many particles in a fixed order, so the kernel is bound by the latency
// of that chain.  The rows that hold air come from the row bits; of the 100
// cells only the 36 within the kernel's radius are visited when that changes
// nothing (AirWindow); with the library's own sort a row's cells (consecutive
// along k) are one range of particles, read eight at a time, and the next
// row's range is fetched meanwhile.  At 128^3 with 8 bubbles 1.38 ms as three
// launches that walked 100 cells, particle by particle; 0.56 with rows and
// bits; 0.23 with the near cells alone.
template <int A, bool ROWS>
__device__ __forceinline__ void p2g_air_face(const Grid& g, const f3* __restrict__ pos, const f3* __restrict__ vel,
                                             const float* __restrict__ mass, const int8_t* __restrict__ flag,
                                             const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
                                             const RowBits& rb, const uint8_t* __restrict__ dm,
                                             float* __restrict__ out, float* __restrict__ out2, int64_t f) {
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  {
    // the window (offsets -2..2 from cell (i,j,k)) lies in the 3x3x3 bricks
    // around that cell's brick: no particle of the phase there, no weight
    const int by = (g.ny + 3) / 4, bz = (g.nz + 3) / 4;
    const int64_t b = ((int64_t)(min(i, g.nx - 1) >> 2) * by + (min(j, g.ny - 1) >> 2)) * bz + (min(k, g.nz - 1) >> 2);
    if (!(dm[b] & M_AIR)) {
      out[f] = 0.0f;
      if (out2) out2[f] = 0.0f;
      return;
    }
  }
  const float scale = 1.0f / g.h;
  const f3 gp = mk3((float)i + (A == 0 ? 0.0f : 0.5f), (float)j + (A == 1 ? 0.0f : 0.5f), (float)k + (A == 2 ? 0.0f : 0.5f));
  constexpr int NB = 8;
  float weight = 0, usum = 0;
  const float RE = 1.4f;
  const float RE2 = RE * RE;
  // particles [s, e) in order
  auto visit = [&](uint32_t s, uint32_t e) {
    for (uint32_t p0 = s; p0 < e; p0 += NB) {
      int8_t fl[NB];
      f3 x[NB];
      float mp[NB], va[NB];
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const uint32_t p = min(p0 + (uint32_t)u, e - 1u);
        fl[u] = flag[p];
        x[u] = pos[p];
        mp[u] = mass[p];
        va[u] = (&vel[p].x)[A];
      }
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        if (p0 + (uint32_t)u >= e || fl[u] != AIR) continue;
        const f3 dv = mk3((x[u].x - g.gx0) * scale - gp.x, (x[u].y - g.gy0) * scale - gp.y, (x[u].z - g.gz0) * scale - gp.z);
        const float r2 = dot3(dv, dv);
        // from the kernel's radius on RE2 / r2 - 1 is not positive: no division
        // (the far two cells of a transverse row are all beyond it)
        float q = 0.0f;
        if (!(r2 >= RE2)) q = fmaxf(RE2 / fmaxf(r2, 0.0001f) - 1.0f, 0.0f);
        const float w = mp[u] * q;
        weight += w;
        usum += w * va[u];
      }
    }
  };
  // the window's rows that hold air, NK bits each, in the reference's order
  using AW = AirWindow<A>;
  constexpr int NJ = AW::NJ, NK = AW::NK, RW = AW::RW;
  uint64_t w[2] = {0, 0};
#pragma unroll
  for (int di = 0; di < AW::NI; ++di) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int dj = 0; dj < NJ; ++dj) {
      const int r = di * NJ + dj;
      w[r / RW] |= (uint64_t)(row_window(rb.a, rb, i + di, j + dj, k) & AW::ROW) << (NK * (r % RW));
    }
  }
  if (ROWS && *rb.odd == 0) {  // the library's own sort, every air particle finite and on the grid
    w[0] &= AW::near_word(0);
    w[1] &= AW::near_word(1);
  }
  // the next row's range (ROWS) or cells: offset of its cell k - 2, its bits
  auto pop = [&](int64_t& c0, uint32_t& bits) {
    const bool lo = w[0] != 0;
    const uint64_t v = lo ? w[0] : w[1];
    const int q = (__ffsll((unsigned long long)v) - 1) / NK, r = q + (lo ? 0 : RW);
    bits = (uint32_t)(v >> (NK * q)) & AW::ROW;
    const uint64_t keep = ~((uint64_t)AW::ROW << (NK * q));
    if (lo) w[0] &= keep;
    else w[1] &= keep;
    c0 = cid(g, i + r / NJ - 2, j + r % NJ - 2, k - 2);
  };
  if (ROWS) {
    uint32_t s = 0, e = 0;
    auto next = [&]() {
      s = e = 0;
      if (!(w[0] | w[1])) return;
      int64_t c0;
      uint32_t bits;
      pop(c0, bits);
      s = cstart[c0 + __ffs(bits) - 1];
      e = cend[c0 + 31 - __clz(bits)];
    };
    next();
    while (s < e) {
      const uint32_t cs = s, ce = e;
      next();  // in flight during this row's particles
      visit(cs, ce);
    }
  } else {
    while (w[0] | w[1]) {
      int64_t c0;
      uint32_t bits;
      pop(c0, bits);
      for (; bits; bits &= bits - 1u) {
        const int64_t c = c0 + __ffs(bits) - 1;
        visit(cstart[c], cend[c]);
      }
    }
  }
  const float u = (weight > 0) ? (usum / weight) : 0.0f;
  out[f] = u;
  if (out2) out2[f] = u;
}
struct P2GOut {
  float* u[3];
  float* u2[3];
};
template <bool ROWS>
__global__ void __launch_bounds__(256)
    k_p2g_air(Grid g, const f3* __restrict__ pos, const f3* __restrict__ vel, const float* __restrict__ mass,
              const int8_t* __restrict__ flag, const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
              RowBits rb, const uint8_t* __restrict__ dm, P2GOut o) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int A = blockIdx.y;
  if (f >= (A == 0 ? g.FX : A == 1 ? g.FY : g.FZ)) return;
  if (A == 0) p2g_air_face<0, ROWS>(g, pos, vel, mass, flag, cstart, cend, rb, dm, o.u[0], o.u2[0], f);
  else if (A == 1) p2g_air_face<1, ROWS>(g, pos, vel, mass, flag, cstart, cend, rb, dm, o.u[1], o.u2[1], f);
  else p2g_air_face<2, ROWS>(g, pos, vel, mass, flag, cstart, cend, rb, dm, o.u[2], o.u2[2], f);
}

// Liquid+solid P2G, tile scatter (the hot path).  A block owns a 4x8x8 cell
// tile with one thread per cell and the cell's particles in registers.  Its
// cells contribute to the faces of a per-axis region (the tile's faces plus
// the ring its windows reach); the 27 window offsets are visited as phases in
// the gather's lexicographic order, and in phase o every thread adds its
// particles, in index order, to face c - o of each axis whose window holds o
// -- one-to-one within a phase, so LDS accumulates without atomics.  Each
// tile stores its region's (sum w, sum w v); a second kernel adds, per face,
// the regions of the (at most 8) tiles that cover it in tile order and
// divides.  Every particle-face pair is evaluated once and every thread holds
// a tile cell (no halo threads); sums are deterministic, associated per tile
// (a face inside one tile's region sums exactly like the gather).
constexpr int ST_X = 4, ST_Y = 8, ST_Z = 8;
constexpr int ST_CELLS = ST_X * ST_Y * ST_Z;  // 256 threads
__host__ __device__ constexpr int st_t(int d) { return d == 0 ? ST_X : (d == 1 ? ST_Y : ST_Z); }
// region of axis a: faces [t0_d - (d != a), t0_d + T_d] along d
__host__ __device__ constexpr int st_r(int a, int d) { return st_t(d) + (d == a ? 1 : 2); }
__host__ __device__ constexpr int st_rsz(int a) { return st_r(a, 0) * st_r(a, 1) * st_r(a, 2); }
__host__ __device__ constexpr int st_roff(int a) { return a == 0 ? 0 : (a == 1 ? st_rsz(0) : st_rsz(0) + st_rsz(1)); }
constexpr int ST_RTOT = st_rsz(0) + st_rsz(1) + st_rsz(2);  // 1580 faces
constexpr int SCH = 8;   // particles of a cell in registers in the first pass
constexpr int SCH2 = 4;  // particles per cell in each overflow pass

// A cell's next ns particles [base, base + cnt) in registers (an empty slot
// loads the chunk's last particle, or particle 0 when the chunk is empty, so
// all loads are in flight together; its weight is 0).
template <int NS>
__device__ __forceinline__ void p2g_load(const f3* __restrict__ pos, const f3* __restrict__ vel,
                                         const float* __restrict__ mass, const int8_t* __restrict__ flag,
                                         const Grid& g, float scale, uint32_t base, uint32_t cnt, float (&X)[NS],
                                         float (&Y)[NS], float (&Z)[NS], float (&VX)[NS], float (&VY)[NS],
                                         float (&VZ)[NS], float (&M)[NS]) {
#pragma unroll
  for (int q = 0; q < NS; ++q) {
    const uint32_t p = (cnt > 0) ? base + min((uint32_t)q, cnt - 1) : 0u;
    const int8_t fl = flag[p];
    const f3 x = pos[p], v = vel[p];
    const float m = mass[p];
    X[q] = (x.x - g.gx0) * scale;
    Y[q] = (x.y - g.gy0) * scale;
    Z[q] = (x.z - g.gz0) * scale;
    VX[q] = v.x; VY[q] = v.y; VZ[q] = v.z;
    M[q] = ((uint32_t)q < cnt && (fl == FLUID || fl == SOLID)) ? m : 0.0f;
  }
}

// The 27 phases of one pass: in phase o every active thread adds its NS
// register particles (of cell (ci, cj, ck)) to face c - o of each axis whose
// window holds o.  Within a pass the active cells are distinct, so a face
// takes at most one thread per phase (no atomics).  Inactive threads only
// meet the barriers.
// The sums of the first two squared differences serve three phases; with them
// formed in each phase the tiles took 0.52 ms (11.3M particles, 128^3), now
// 0.43, bound by issuing vector instructions (11 per weight, an exact quotient
// among them).
template <int NS>
__device__ __forceinline__ void p2g_phases(int x0, int y0, int z0, int ci, int cj, int ck, bool act,
                                           const float (&X)[NS], const float (&Y)[NS], const float (&Z)[NS],
                                           const float (&VX)[NS], const float (&VY)[NS], const float (&VZ)[NS],
                                           const float (&M)[NS], float* sW, float* sU) {
  // The faces of the three axes in a phase share the cell c - o: axis a's face
  // sits at that cell's corner along a and at its centre along the others, so
  // a particle's coordinate differences to the corner and the centre and their
  // squares serve all three distances, summed in the gather's order; the sums
  // of the first two directions serve the three phases along k.
  const float RE = 1.4f, RE2 = RE * RE;
  for (int oo = 0; oo < 9; ++oo) {
    const int o0 = oo / 3 - 1, o1 = oo % 3 - 1;
    const int f0 = ci - o0, f1 = cj - o1;
    float s0[NS], s1[NS], s2[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) {
      const float fx = (float)f0, fy = (float)f1;
      const float ax = X[q] - fx, bx = X[q] - (fx + 0.5f), ay = Y[q] - fy, by = Y[q] - (fy + 0.5f);
      const float ax2 = ax * ax, bx2 = bx * bx, ay2 = ay * ay, by2 = by * by;
      s0[q] = ax2 + by2;
      s1[q] = bx2 + ay2;
      s2[q] = bx2 + by2;
    }
    int li[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      const int r0 = x0 - (a != 0), r1 = y0 - (a != 1), r2 = z0 - (a != 2);
      li[a] = st_roff(a) + ((f0 - r0) * st_r(a, 1) + (f1 - r1)) * st_r(a, 2) + (ck - r2);
    }
#pragma unroll
    for (int o2 = -1; o2 <= 1; ++o2) {
      if (act) {
        const float fz = (float)(ck - o2), hz = fz + 0.5f;
        // one face's share: the particles in index order
        auto face = [&](int l, const float (&s)[NS], float z, const float (&V)[NS]) {
          float W = sW[l], U = sU[l];
#pragma unroll
          for (int q = 0; q < NS; ++q) {
            const float d = Z[q] - z;
            const float w = M[q] * fmaxf(div_nr(RE2, fmaxf(s[q] + d * d, 0.0001f)) - 1.0f, 0.0f);
            W += w;
            U += w * V[q];
          }
          sW[l] = W;
          sU[l] = U;
        };
        if (o0 <= 0) face(li[0] - o2, s0, hz, VX);  // normal window is {-1, 0}
        if (o1 <= 0) face(li[1] - o2, s1, hz, VY);
        if (o2 <= 0) face(li[2] - o2, s2, fz, VZ);
      }
      __syncthreads();
    }
  }
}

// Overflow passes of a tile: pass p takes particles [thr, thr + SCH2) of
// every cell holding more than thr = SCH + (p-1) SCH2, the cells compacted
// onto the first threads (a wave without such a cell skips the arithmetic).
// Returns after the pass that finds no cell left; block-uniform.
template <class PassFn>
__device__ __forceinline__ void overflow_passes(uint32_t n, uint32_t* sList, int* sWc, PassFn pass) {
  const int wv = threadIdx.x >> 6, ln = threadIdx.x & 63;
  for (uint32_t thr = SCH;; thr += SCH2) {
    const bool pred = n > thr;
    const unsigned long long bal = __ballot(pred);
    if (ln == 0) sWc[wv] = __popcll(bal);
    __syncthreads();
    int off = 0, tot = 0;
#pragma unroll
    for (int w2 = 0; w2 < ST_CELLS / 64; ++w2) {
      off += (w2 < wv) ? sWc[w2] : 0;
      tot += sWc[w2];
    }
    if (pred) sList[off + __popcll(bal & ((1ull << ln) - 1ull))] = threadIdx.x;
    __syncthreads();
    if (tot == 0) return;
    const bool act = (int)threadIdx.x < tot;
    pass(act, act ? sList[threadIdx.x] : 0u, thr);
  }
}

__global__ void __launch_bounds__(ST_CELLS, 4)
    k_p2g_tile(Grid g, const f3* __restrict__ pos, const f3* __restrict__ vel, const float* __restrict__ mass,
               const int8_t* __restrict__ flag, const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
               const uint8_t* __restrict__ cmask, float* __restrict__ parts, int ntx, int nty, int ntz,
               const float* __restrict__ band, float big, const uint8_t* __restrict__ dmask) {
  __shared__ float sW[ST_RTOT];
  __shared__ float sU[ST_RTOT];
  __shared__ uint32_t sS[ST_CELLS], sN[ST_CELLS], sList[ST_CELLS];
  __shared__ int sWc[ST_CELLS / 64];
  const int tl = (int)xcd_block();  // XCD-contiguous tiles
  int t = tl;
  const int tz = t % ntz;
  t /= ntz;
  const int ty = t % nty;
  const int tx = t / nty;
  const int x0 = tx * ST_X, y0 = ty * ST_Y, z0 = tz * ST_Z;
  for (int q = threadIdx.x; q < ST_RTOT; q += ST_CELLS) {
    sW[q] = 0.0f;
    sU[q] = 0.0f;
  }
  const int b = threadIdx.x;
  const int ci = x0 + b / (ST_Y * ST_Z), cj = y0 + (b / ST_Z) % ST_Y, ck = z0 + b % ST_Z;
  uint32_t s = 0, e = 0;
  if (valid(g, ci, cj, ck)) {
    const int64_t c = cid(g, ci, cj, ck);
    if (cmask[c] & M_FLUIDSOLID) {
      s = cstart[c];
      e = cend[c];
    }
  }
  // band mode: a tile whose cells and ring hold no cell with band < big maps nothing
  bool near = true;
  if (band) {
    // band cells lie within 3 cells of a solid cell, and the region's cells
    // within one cell of the tile, so a tile whose bricks (1 x 2 x 2 of the
    // 4x4x4 bricks, each with its 3x3x3 neighbourhood in dmask) hold no solid
    // cell has none in its region: its band scan is skipped
    static_assert(ST_X == 4 && ST_Y == 8 && ST_Z == 8, "a tile spans 1 x 2 x 2 bricks");
    const int nby = (g.ny + 3) / 4, nbz = (g.nz + 3) / 4;
    uint8_t bm = 0;
#pragma unroll
    for (int dj = 0; dj < 2; ++dj)
#pragma unroll
      for (int dk = 0; dk < 2; ++dk) {
        const int bj = (y0 >> 2) + dj, bk = (z0 >> 2) + dk;
        if (bj < nby && bk < nbz) bm |= dmask[((int64_t)(x0 >> 2) * nby + bj) * nbz + bk];
      }
    near = (bm & M_SOLID) != 0;
  }
  if (band && near) {
    bool mine = false;
    for (int q = threadIdx.x; q < (ST_X + 2) * (ST_Y + 2) * (ST_Z + 2); q += ST_CELLS) {
      const int bi = x0 - 1 + q / ((ST_Y + 2) * (ST_Z + 2)), bj = y0 - 1 + (q / (ST_Z + 2)) % (ST_Y + 2),
                bk = z0 - 1 + q % (ST_Z + 2);
      if (valid(g, bi, bj, bk) && band[cid(g, bi, bj, bk)] < big) mine = true;
    }
    near = __syncthreads_or(mine);
  }
  const int any = __syncthreads_or(e > s) && near;
  if (any) {
    const float scale = 1.0f / g.h;
    const uint32_t n = e - s;
    sS[b] = s;
    sN[b] = n;
    {
      float X[SCH], Y[SCH], Z[SCH], VX[SCH], VY[SCH], VZ[SCH], M[SCH];
      p2g_load<SCH>(pos, vel, mass, flag, g, scale, s, min(n, (uint32_t)SCH), X, Y, Z, VX, VY, VZ, M);
      p2g_phases<SCH>(x0, y0, z0, ci, cj, ck, n > 0, X, Y, Z, VX, VY, VZ, M, sW, sU);
    }
    // cells with more than SCH particles: the rest in compacted passes
    overflow_passes(n, sList, sWc, [&](bool act, uint32_t cb, uint32_t thr) {
      const int oi = x0 + (int)cb / (ST_Y * ST_Z), oj = y0 + ((int)cb / ST_Z) % ST_Y, ok = z0 + (int)cb % ST_Z;
      const uint32_t os = act ? sS[cb] + thr : 0u;
      const uint32_t oc = act ? min(sN[cb] - thr, (uint32_t)SCH2) : 0u;
      float X[SCH2], Y[SCH2], Z[SCH2], VX[SCH2], VY[SCH2], VZ[SCH2], M[SCH2];
      if (act) p2g_load<SCH2>(pos, vel, mass, flag, g, scale, os, oc, X, Y, Z, VX, VY, VZ, M);
      p2g_phases<SCH2>(x0, y0, z0, oi, oj, ok, act, X, Y, Z, VX, VY, VZ, M, sW, sU);
    });
  } else {
    __syncthreads();
  }
  float* dst = parts + (int64_t)tl * (2 * ST_RTOT);
  for (int q = threadIdx.x; q < ST_RTOT; q += ST_CELLS) {
    dst[q] = sW[q];
    dst[ST_RTOT + q] = sU[q];
  }
}

// u = (sum w v) / (sum w) per face from the tile regions covering it, added in
// tile order (also into out2 when given: the copy the FLIP update keeps).
// Band mode: faces without a cell of band < big beside them are 0.
template <int A>
__device__ __forceinline__ void p2g_collect_face(const Grid& g, const float* __restrict__ parts, int ntx, int nty,
                                                 int ntz, float* __restrict__ out, float* __restrict__ out2, int64_t f,
                                                 const float* __restrict__ band, float big) {
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  if (band) {
    const int n3a = (A == 0) ? g.nx : (A == 1) ? g.ny : g.nz;
    const int na = (A == 0) ? i : (A == 1) ? j : k;
    bool in_band = false;
    if (na < n3a) in_band = in_band || band[cid(g, i, j, k)] < big;
    if (na > 0) in_band = in_band || band[cid(g, i - (A == 0), j - (A == 1), k - (A == 2))] < big;
    if (!in_band) {
      out[f] = 0.0f;
      return;
    }
  }
  const int fv[3] = {i, j, k};
  const int nt[3] = {ntx, nty, ntz};
  int qlo[3], qhi[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    // tiles q with q*T - (d != A) <= f <= q*T + T
    const int T = st_t(d);
    int lo = (fv[d] - T + T - 1) / T;  // ceil((f - T) / T) for f >= 0
    if (fv[d] - T < 0) lo = 0;
    int hi = (fv[d] + (d != A ? 1 : 0)) / T;
    if (hi > nt[d] - 1) hi = nt[d] - 1;
    qlo[d] = lo;
    qhi[d] = hi;
  }
  float W = 0.0f, U = 0.0f;
  for (int qx = qlo[0]; qx <= qhi[0]; ++qx)
    for (int qy = qlo[1]; qy <= qhi[1]; ++qy)
      for (int qz = qlo[2]; qz <= qhi[2]; ++qz) {
        const int r0 = qx * ST_X - (A != 0), r1 = qy * ST_Y - (A != 1), r2 = qz * ST_Z - (A != 2);
        const int li = st_roff(A) + ((fv[0] - r0) * st_r(A, 1) + (fv[1] - r1)) * st_r(A, 2) + (fv[2] - r2);
        const float* src = parts + ((int64_t)(qx * nty + qy) * ntz + qz) * (2 * ST_RTOT);
        W += src[li];
        U += src[ST_RTOT + li];
      }
  const float u = (W > 0) ? (U / W) : 0.0f;
  out[f] = u;
  if (out2) out2[f] = u;
}

__global__ void k_p2g_collect(Grid g, const float* __restrict__ parts, int ntx, int nty, int ntz, P2GOut o,
                              const float* __restrict__ band, float big) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int A = blockIdx.y;
  if (f >= (A == 0 ? g.FX : A == 1 ? g.FY : g.FZ)) return;
  if (A == 0) p2g_collect_face<0>(g, parts, ntx, nty, ntz, o.u[0], o.u2[0], f, band, big);
  else if (A == 1) p2g_collect_face<1>(g, parts, ntx, nty, ntz, o.u[1], o.u2[1], f, band, big);
  else p2g_collect_face<2>(g, parts, ntx, nty, ntz, o.u[2], o.u2[2], f, band, big);
}

// ---------------- extrapolation + wall conditions (a10) ----------------
// initphi, spray_k.cu:712-723
// (both phases)
__global__ void k_initphi(int64_t G, const int8_t* __restrict__ mark, float* __restrict__ phi0, int8_t type0,
                          float* __restrict__ phi1, int8_t type1, float big) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= G) return;
  const int8_t m = mark[idx];
  phi0[idx] = (m == type0) ? -0.5f : big;
  phi1[idx] = (m == type1) ? -0.5f : big;
}

// sweepu_k_bubble spray_k.cu:3779-3880 (one axis, out-of-place): the new
// value of face (i, j, k) of axis A (index f); u0 returns its old value
template <int A>
__device__ __forceinline__ float sweep_u_face(const Grid& g, const float* __restrict__ u,
                                              const float* __restrict__ ls, const int8_t* __restrict__ mark, int8_t sf,
                                              int i, int j, int k, int64_t f, float& u0) {
  const int n[3] = {i, j, k};
  const int lim = (A == 0) ? g.nx : (A == 1) ? g.ny : g.nz;
  const bool inner = n[A] > 1 && n[A] < lim - 1;
  // first round of loads: the face, the marks and level sets of its two cells
  // (cell indices clamped for the faces the rule leaves as they are)
  const int ci = min(i, g.nx - 1), cj = min(j, g.ny - 1), ck = min(k, g.nz - 1);
  const int bi = max(i - (A == 0), 0), bj = max(j - (A == 1), 0), bk = max(k - (A == 2), 0);
  float res = u[f];
  u0 = res;
  const int8_t mc = mark[cid(g, ci, cj, ck)], mb = mark[cid(g, bi, bj, bk)];
  const float lsc = ls[cid(g, ci, cj, ck)], lsb = ls[cid(g, bi, bj, bk)];
  if (inner && mc != sf && mb != sf) {
    constexpr int t1 = (A == 0) ? 1 : (A == 1) ? 0 : 1;
    constexpr int t2 = (A == 0) ? 2 : (A == 1) ? 2 : 0;
    const int lims[3] = {g.nx, g.ny, g.nz};
    // second round: the level sets beside both cells across each transverse
    // axis and the face's six neighbours, all issued together (indices
    // clamped; a value outside the grid is not used)
    float lt[2][2][2];  // [transverse t][sign][cell c / cell b]
    bool in[2][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int ax = t == 0 ? t1 : t2;
#pragma unroll
      for (int sg = 0; sg < 2; ++sg) {
        const int dd = sg ? 1 : -1;
        in[t][sg] = n[ax] + dd >= 0 && n[ax] + dd <= lims[ax] - 1;
        int o[3] = {0, 0, 0};
        o[ax] = in[t][sg] ? dd : 0;
        lt[t][sg][0] = ls[cid(g, i + o[0], j + o[1], k + o[2])];
        lt[t][sg][1] = ls[cid(g, i - (A == 0) + o[0], j - (A == 1) + o[1], k - (A == 2) + o[2])];
      }
    }
    float un[3][2];  // u of the face's neighbours along x, y, z (sign -1, +1)
    const int fl[3] = {(A == 0) ? g.nx : g.nx - 1, (A == 1) ? g.ny : g.ny - 1, (A == 2) ? g.nz : g.nz - 1};
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
      for (int sg = 0; sg < 2; ++sg) {
        int q[3] = {i, j, k};
        q[d] = min(max(q[d] + (sg ? 1 : -1), 0), fl[d]);
        un[d][sg] = u[fid(g, A, q[0], q[1], q[2])];
      }
    // The reference visits the 8 octants (di, dj, dk in {-1, +1}, di
    // outermost) and the last one whose three weights are all >= 0 sets the
    // value.  Each weight depends on its own axis' sign only, so that octant
    // takes, per axis, +1 if its weight passes there, else -1.
    const float dl = lsc - lsb;
    const float wa[2] = {(float)(1) * dl, (float)(-1) * dl};  // sign -1, +1
    float wt[2][2];
    bool ok[3][2];
    ok[A][0] = !(wa[0] < 0);
    ok[A][1] = !(wa[1] < 0);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int ax = t == 0 ? t1 : t2;
#pragma unroll
      for (int sg = 0; sg < 2; ++sg) {
        float w = 0.0f;
        if (in[t][sg]) w = (lsc + lsb - lt[t][sg][0] - lt[t][sg][1]) * 0.5f;
        wt[t][sg] = w;
        ok[ax][sg] = in[t][sg] && !(w < 0);
      }
    }
    if ((ok[0][0] || ok[0][1]) && (ok[1][0] || ok[1][1]) && (ok[2][0] || ok[2][1])) {
      const int sgn[3] = {ok[0][1] ? 1 : 0, ok[1][1] ? 1 : 0, ok[2][1] ? 1 : 0};
      float wv[3];
      wv[A] = wa[sgn[A]];
      wv[t1] = wt[0][sgn[t1]];
      wv[t2] = wt[1][sgn[t2]];
      float wx = wv[0], wy = wv[1], wz = wv[2];
      float wsum = wx + wy + wz;
      if (wsum == 0) wx = wy = wz = 1.0f / 3;
      else { wx /= wsum; wy /= wsum; wz /= wsum; }
      res = wx * un[0][sgn[0]] + wy * un[1][sgn[1]] + wz * un[2][sgn[2]];
    }
  }
  return res;
}

// One extrapolation pass of axis A on 1 x SW_J x SW_K tiles of its faces,
// with the change flags of the eikonal passes: a face's new value reads its
// own and its six neighbours' values (level sets and marks are fixed over the
// passes), so a tile whose neighbourhood did not change in the previous pass
// (prev) is skipped, its values being in the output buffer already.  cur (may
// be null) records the changes of this pass; prev == nullptr computes every
// tile.  A change is a different bit pattern.
template <int A>
__device__ __forceinline__ void
    sweep_u_tiles(const Grid& g, const float* __restrict__ u, float* __restrict__ out, const float* __restrict__ ls,
                  const int8_t* __restrict__ mark, int8_t sf, const uint8_t* __restrict__ prev,
                  uint8_t* __restrict__ cur, uint32_t ntj, uint32_t ntk, uint32_t ntiles, int per_wave) {
  const uint32_t t0 = (blockIdx.x * 4u + threadIdx.x / 64u) * (uint32_t)per_wave;
  if (t0 >= ntiles) return;
  const int lane = threadIdx.x & 63;
  const int nfx = g.nx + (A == 0), nfy = g.ny + (A == 1), nfz = g.nz + (A == 2);
  const bool act = tile_active(prev, t0 + lane, lane < per_wave && t0 + lane < ntiles, ntj, ntk, (uint32_t)nfx);
  uint64_t todo = __ballot(act);
  uint8_t myflag = 0;
  const int jl = lane / SW_K, kl = lane % SW_K;
  const uint32_t sxt = ntj * ntk;
  while (todo) {
    const int q = __builtin_ctzll(todo);
    todo &= todo - 1;
    const uint32_t t = t0 + q;
    const int tk = (int)(t % ntk), tj = (int)((t / ntk) % ntj), i = (int)(t / sxt);
    const int j = tj * SW_J + jl, k = tk * SW_K + kl;
    bool changed = false;
    if (j < nfy && k < nfz) {
      const int64_t f = fid(g, A, i, j, k);
      float u0;
      const float res = sweep_u_face<A>(g, u, ls, mark, sf, i, j, k, f, u0);
      changed = __float_as_uint(res) != __float_as_uint(u0);
      out[f] = res;
    }
    const uint8_t fl = tile_flags(changed);
    if (lane == q) myflag = fl;
  }
  if (cur && lane < per_wave && t0 + lane < ntiles) cur[t0 + lane] = myflag;
}

// The six fields (phase and axis: blockIdx.y = 3 phase + axis) in one launch:
// one by one their passes took 19 us each at 128^3, most of it the launch and
// its last waves.
struct SweepU {
  const float* u[6];
  float* out[6];
  const float* ls[2];
  int8_t sf[2];
  uint8_t* flags[6];
};
template <bool FIRST>
__global__ void __launch_bounds__(256) k_sweep_u(Grid g, SweepU s, const int8_t* __restrict__ mark, int per_wave) {
  const int ph = blockIdx.y / 3, A = blockIdx.y % 3, q = blockIdx.y;
  const int64_t nfx = g.nx + (A == 0), nfy = g.ny + (A == 1), nfz = g.nz + (A == 2);
  const uint32_t ntj = (uint32_t)((nfy + SW_J - 1) / SW_J), ntk = (uint32_t)((nfz + SW_K - 1) / SW_K);
  const uint32_t nt = (uint32_t)nfx * ntj * ntk;
  const uint8_t* prev = FIRST ? nullptr : s.flags[q];
  uint8_t* cur = FIRST ? s.flags[q] : nullptr;
  if (A == 0) sweep_u_tiles<0>(g, s.u[q], s.out[q], s.ls[ph], mark, s.sf[ph], prev, cur, ntj, ntk, nt, per_wave);
  else if (A == 1) sweep_u_tiles<1>(g, s.u[q], s.out[q], s.ls[ph], mark, s.sf[ph], prev, cur, ntj, ntk, nt, per_wave);
  else sweep_u_tiles<2>(g, s.u[q], s.out[q], s.ls[ph], mark, s.sf[ph], prev, cur, ntj, ntk, nt, per_wave);
}

// setWaterBoundaryU_k spray_k.cu:956-995 (in place).  The ceiling rule reads
// uz(k-1) after that face's own rule.
__device__ __forceinline__ bool isb(const Grid& g, const int8_t* mark, int i, int j, int k) {
  return mark[cid(g, i, j, k)] == BOUNDARY;
}
template <int A>
__device__ __forceinline__ void bc_face(const Grid& g, float* __restrict__ u, const int8_t* __restrict__ mark, int64_t f) {
  const int hh = g.ny + (A == 1), d = g.nz + (A == 2);
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  if (A == 0) {
    if (i <= 1 || i >= (g.nx + 1) - 2) u[f] = 0.0f;
    else if (i > 1 && i < g.nx - 1 && (isb(g, mark, i, j, k) != isb(g, mark, i - 1, j, k))) u[f] = 0.0f;
  } else if (A == 1) {
    if (j <= 1 || j >= (g.ny + 1) - 2) u[f] = 0.0f;
    else if (j > 0 && j < g.ny && (isb(g, mark, i, j, k) != isb(g, mark, i, j - 1, k))) u[f] = 0.0f;
  } else {
    const int zn = g.nz + 1;
    if (k <= 1 || k >= zn - 1) u[f] = 0.0f;
    else if (k == zn - 2) {
      // post-rule value of uz(k-1): k-1 >= 2 is neither wall nor ceiling here
      int kb = k - 1;
      float b = u[f - 1];
      if (kb <= 1) b = 0.0f;
      else if (kb > 0 && kb < g.nz && (isb(g, mark, i, j, kb) != isb(g, mark, i, j, kb - 1))) b = 0.0f;
      u[f] = (b < 0) ? b : 0.0f;
    } else if (k > 0 && k < g.nz && (isb(g, mark, i, j, k) != isb(g, mark, i, j, k - 1))) u[f] = 0.0f;
  }
}

struct Faces6 {
  float* u[6];  // water x, y, z, air x, y, z
};
__global__ void k_bc(Grid g, Faces6 fs, const int8_t* __restrict__ mark) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int A = blockIdx.y % 3;
  if (f >= (A == 0 ? g.FX : A == 1 ? g.FY : g.FZ)) return;
  float* u = fs.u[blockIdx.y];
  if (A == 0) bc_face<0>(g, u, mark, f);
  else if (A == 1) bc_face<1>(g, u, mark, f);
  else bc_face<2>(g, u, mark, f);
}

// ---------------- divergence (a11) and gradient (a13) ----------------
__device__ __forceinline__ int8_t mark_at(const Grid& g, const int8_t* mark, int i, int j, int k) {
  return valid(g, i, j, k) ? mark[cid(g, i, j, k)] : BOUNDARY;
}
// cptdivergence_bubble2, spray_k.cu:3138-3263, in arithmetic R.
template <class R>
__global__ void k_divergence(Grid g, const float* __restrict__ wux, const float* __restrict__ wuy,
                             const float* __restrict__ wuz, const float* __restrict__ aux,
                             const float* __restrict__ auy, const float* __restrict__ auz,
                             const int8_t* __restrict__ mark, const float* __restrict__ ls, int solid_c,
                             R* __restrict__ div) {
  CELL_LOOP_HEAD
  R dv = 0;
  const int8_t m = mark[idx];
  if (m == FLUID || m == AIR) {
    const float* wu[3] = {wux, wuy, wuz};
    const float* au[3] = {aux, auy, auz};
    R uu[6];
    int q = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a)
#pragma unroll
      for (int s = 1; s >= 0; --s) {
        int ni = i + (a == 0 ? (s ? 1 : -1) : 0), nj = j + (a == 1 ? (s ? 1 : -1) : 0), nk = k + (a == 2 ? (s ? 1 : -1) : 0);
        int64_t fx = fid(g, a, i + (a == 0 && s), j + (a == 1 && s), k + (a == 2 && s));
        int8_t mn = mark_at(g, mark, ni, nj, nk);
        R v;
        if (solid_c && mn == SOLID) v = R(0);
        else if (m == FLUID && mn != AIR) v = (R)wu[a][fx];
        else if (m == AIR && mn != FLUID) v = (R)au[a][fx];
        else {
          R lc = (R)ls[idx], ln = (R)ls[cid(g, ni, nj, nk)];
          R th = (R(0.0f) - lc) / (ln - lc);
          if (m == FLUID) v = th * (R)wu[a][fx] + (R(1) - th) * (R)au[a][fx];
          else v = th * (R)au[a][fx] + (R(1) - th) * (R)wu[a][fx];
        }
        uu[q++] = v;
      }
    dv = (uu[0] - uu[1] + uu[2] - uu[3] + uu[4] - uu[5]) / (R)g.h;
  }
  div[idx] = dv;
}

// subGradPress spray_k.cu:198-224 (unit form, in R) or the 1/rho form (double).
template <int A, class R>
__device__ __forceinline__ void subgrad_face(const Grid& g, float* __restrict__ u, const R* __restrict__ p,
                                             const int8_t* __restrict__ mark, int vardens, double inv_rho, int solid_c,
                                             int64_t f) {
  const int hh = g.ny + (A == 1), d = g.nz + (A == 2);
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  const int n[3] = {i, j, k};
  const int lim = (A == 0) ? g.nx : (A == 1) ? g.ny : g.nz;
  if (!(n[A] > 0 && n[A] < lim)) return;
  const int bi = i - (A == 0), bj = j - (A == 1), bk = k - (A == 2);
  const int64_t c0 = cid(g, i, j, k), c1 = cid(g, bi, bj, bk);
  if (solid_c && (mark[c0] == SOLID || mark[c1] == SOLID)) {
    u[f] = 0.0f;
    return;
  }
  if (!vardens) u[f] = (float)((R)u[f] - (p[c0] - p[c1]) / (R)g.h);
  else u[f] = (float)((double)u[f] - inv_rho * (((double)p[c0] - (double)p[c1]) / (double)g.h));
}

template <class R>
__global__ void k_subgrad(Grid g, Faces6 fs, const R* __restrict__ p, const int8_t* __restrict__ mark, int vardens,
                          double inv_rho_liquid, double inv_rho_air, int solid_c) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int A = blockIdx.y % 3;
  if (f >= (A == 0 ? g.FX : A == 1 ? g.FY : g.FZ)) return;
  float* u = fs.u[blockIdx.y];
  const double inv_rho = blockIdx.y < 3 ? inv_rho_liquid : inv_rho_air;
  if (A == 0) subgrad_face<0, R>(g, u, p, mark, vardens, inv_rho, solid_c, f);
  else if (A == 1) subgrad_face<1, R>(g, u, p, mark, vardens, inv_rho, solid_c, f);
  else subgrad_face<2, R>(g, u, p, mark, vardens, inv_rho, solid_c, f);
}

// ---------------- heat grid stages (a16) ----------------
// Heat P2G (mapHeatp2g_hash + sumHeat, spray_k.cu:4619-4653) as a tile
// scatter like the liquid P2G: one thread per cell of a 4x8x8 tile, 27
// phases in the gather's order adding each particle to the cell c - o of the
// tile's region (the tile grown by one cell), per-tile sums combined per cell
// in tile order by k_heat_collect.
constexpr int HR_X = ST_X + 2, HR_Y = ST_Y + 2, HR_Z = ST_Z + 2;
constexpr int HR = HR_X * HR_Y * HR_Z;  // 600 cells

// NS particles of cell (ci, cj, ck) in registers, and the phases that add
// them to cell c - o in phase o (the liquid P2G's pass structure; 0.35 ms with
// every square formed in each phase, 0.23 now, 128^3).
template <int NS>
__device__ __forceinline__ void heat_load(const f3* __restrict__ pos, const float* __restrict__ temp, const Grid& g,
                                          float scale, uint32_t base, uint32_t cnt, float (&X)[NS], float (&Y)[NS],
                                          float (&Z)[NS], float (&TT)[NS], float (&ON)[NS]) {
  f3 xr[NS];
#pragma unroll
  for (int q = 0; q < NS; ++q) {
    const uint32_t p = (cnt > 0) ? base + min((uint32_t)q, cnt - 1) : 0u;
    xr[q] = pos[p];
    TT[q] = temp[p];
  }
  __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of their uses
#pragma unroll
  for (int q = 0; q < NS; ++q) {
    const bool on = (uint32_t)q < cnt;
    X[q] = on ? (xr[q].x - g.gx0) * scale : 0.0f;
    Y[q] = on ? (xr[q].y - g.gy0) * scale : 0.0f;
    Z[q] = on ? (xr[q].z - g.gz0) * scale : 0.0f;
    TT[q] = on ? TT[q] : 0.0f;
    ON[q] = on ? 1.0f : 0.0f;
  }
}

template <int NS>
__device__ __forceinline__ void heat_phases(int x0, int y0, int z0, int ci, int cj, int ck, bool act,
                                            const float (&X)[NS], const float (&Y)[NS], const float (&Z)[NS],
                                            const float (&TT)[NS], const float (&ON)[NS], float* sW, float* sH) {
  const float RE = 1.4f, RE2 = RE * RE;
  for (int oo = 0; oo < 9; ++oo) {
    const int f0 = ci - (oo / 3 - 1), f1 = cj - (oo % 3 - 1);
    const int l0 = ((f0 - (x0 - 1)) * HR_Y + (f1 - (y0 - 1))) * HR_Z + (ck - (z0 - 1));
    float s[NS];
#pragma unroll
    for (int q = 0; q < NS; ++q) {
      const float dx = X[q] - ((float)f0 + 0.5f), dy = Y[q] - ((float)f1 + 0.5f);
      s[q] = dx * dx + dy * dy;
    }
#pragma unroll
    for (int o2 = -1; o2 <= 1; ++o2) {
      if (act) {
        const int li = l0 - o2;
        float W = sW[li], Hs = sH[li];
        const float gz = (float)(ck - o2) + 0.5f;
#pragma unroll
        for (int q = 0; q < NS; ++q) {
          const float dz = Z[q] - gz;
          const float w = ON[q] * fmaxf(div_nr(RE2, fmaxf(s[q] + dz * dz, 0.0001f)) - 1.0f, 0.0f);
          W += w;
          Hs += w * TT[q];
        }
        sW[li] = W;
        sH[li] = Hs;
      }
      __syncthreads();
    }
  }
}

__global__ void __launch_bounds__(ST_CELLS)
    k_heat_tile(Grid g, const f3* __restrict__ pos, const float* __restrict__ temp,
                const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
                const uint8_t* __restrict__ cmask, float* __restrict__ parts, int ntx, int nty, int ntz) {
  __shared__ float sW[HR];
  __shared__ float sH[HR];
  __shared__ uint32_t sS[ST_CELLS], sN[ST_CELLS], sList[ST_CELLS];
  __shared__ int sWc[ST_CELLS / 64];
  const int tl = (int)xcd_block();  // XCD-contiguous tiles
  int t = tl;
  const int tz = t % ntz;
  t /= ntz;
  const int ty = t % nty;
  const int tx = t / nty;
  const int x0 = tx * ST_X, y0 = ty * ST_Y, z0 = tz * ST_Z;
  for (int q = threadIdx.x; q < HR; q += ST_CELLS) {
    sW[q] = 0.0f;
    sH[q] = 0.0f;
  }
  const int b = threadIdx.x;
  const int ci = x0 + b / (ST_Y * ST_Z), cj = y0 + (b / ST_Z) % ST_Y, ck = z0 + b % ST_Z;
  uint32_t s = 0, e = 0;
  if (valid(g, ci, cj, ck)) {
    const int64_t c = cid(g, ci, cj, ck);
    if (cmask[c]) {
      s = cstart[c];
      e = cend[c];
    }
  }
  const int any = __syncthreads_or(e > s);
  if (any) {
    const float scale = 1.0f / g.h;
    const uint32_t n = e - s;
    sS[b] = s;
    sN[b] = n;
    {
      float X[SCH], Y[SCH], Z[SCH], TT[SCH], ON[SCH];
      heat_load<SCH>(pos, temp, g, scale, s, min(n, (uint32_t)SCH), X, Y, Z, TT, ON);
      heat_phases<SCH>(x0, y0, z0, ci, cj, ck, n > 0, X, Y, Z, TT, ON, sW, sH);
    }
    overflow_passes(n, sList, sWc, [&](bool act, uint32_t cb, uint32_t thr) {
      const int oi = x0 + (int)cb / (ST_Y * ST_Z), oj = y0 + ((int)cb / ST_Z) % ST_Y, ok = z0 + (int)cb % ST_Z;
      const uint32_t os = act ? sS[cb] + thr : 0u;
      const uint32_t oc = act ? min(sN[cb] - thr, (uint32_t)SCH2) : 0u;
      float X[SCH2], Y[SCH2], Z[SCH2], TT[SCH2], ON[SCH2];
      if (act) heat_load<SCH2>(pos, temp, g, scale, os, oc, X, Y, Z, TT, ON);
      heat_phases<SCH2>(x0, y0, z0, oi, oj, ok, act, X, Y, Z, TT, ON, sW, sH);
    });
  } else {
    __syncthreads();
  }
  float* dst = parts + (int64_t)tl * (2 * HR);
  for (int q = threadIdx.x; q < HR; q += ST_CELLS) {
    dst[q] = sW[q];
    dst[HR + q] = sH[q];
  }
}

// T of a cell from the regions of the (at most 8) tiles covering it, in tile
// order; cells without particle weight keep the default temperature.
__global__ void k_heat_collect(Grid g, const float* __restrict__ parts, int ntx, int nty, int ntz, float deft,
                               float* __restrict__ tp) {
  CELL_LOOP_HEAD
  const int cv[3] = {i, j, k};
  const int nt[3] = {ntx, nty, ntz};
  int qlo[3], qhi[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int T = st_t(d);  // region [qT - 1, qT + T]
    qlo[d] = (cv[d] - T < 0) ? 0 : (cv[d] - 1) / T;
    const int hi = (cv[d] + 1) / T;
    qhi[d] = hi > nt[d] - 1 ? nt[d] - 1 : hi;
  }
  float W = 0.0f, Hs = 0.0f;
  for (int qx = qlo[0]; qx <= qhi[0]; ++qx)
    for (int qy = qlo[1]; qy <= qhi[1]; ++qy)
      for (int qz = qlo[2]; qz <= qhi[2]; ++qz) {
        const int li = ((i - (qx * ST_X - 1)) * HR_Y + (j - (qy * ST_Y - 1))) * HR_Z + (k - (qz * ST_Z - 1));
        const float* src = parts + ((int64_t)(qx * nty + qy) * ntz + qz) * (2 * HR);
        W += src[li];
        Hs += src[HR + li];
      }
  tp[idx] = (W > 0) ? (Hs / W) : deft;
}

// addHeatAtBottom spray_k.cu:4492-4504, then save T and form b (compb_heat
// 4507-4523) for the implicit solve.
__global__ void k_heat_pre(Grid g, float* __restrict__ tp, float* __restrict__ tsave, float* __restrict__ b,
                           const int8_t* __restrict__ mark, int add_bottom, float inc, float clampv, float a0, float a1,
                           float a2, float a3, float a4, float a5, float dt) {
  CELL_LOOP_HEAD
  float t = tp[idx];
  if (add_bottom) {
    if (i >= 1 && i < g.nx - 1 && j >= 1 && j < g.ny - 1 && k <= 3) t += inc;
    t = fminf(clampv, t);
  }
  tp[idx] = t;
  tsave[idx] = t;
  const float al[6] = {a0, a1, a2, a3, a4, a5};
  int8_t m = mark[idx];
  b[idx] = (m == BOUNDARY) ? 0.0f : (float)((double)t * ((double)g.h * (double)g.h) / (double)al[m] / (double)dt);
}

// One Jacobi sweep of the heat operator (computeAx_heat, spray_k.cu:4526-4567).
// Per cell, once per Jacobi solve: its type (7 = BOUNDARY) and the 6-bit
// mask of neighbours that are not Neumann, in the order +x, +y, +z, -x, -y, -z.
__global__ void k_heat_code(Grid g, const int8_t* __restrict__ mark, uint16_t* __restrict__ code, int vac_neumann) {
  CELL_LOOP_HEAD
  const int8_t m = mark[idx];
  if (m == BOUNDARY) {
    code[idx] = 7;
    return;
  }
  const int off[6][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {-1, 0, 0}, {0, -1, 0}, {0, 0, -1}};
  unsigned mask = 0;
#pragma unroll
  for (int q = 0; q < 6; ++q) {
    const int8_t mn = mark_at(g, mark, i + off[q][0], j + off[q][1], k + off[q][2]);
    if (!(mn == BOUNDARY || (vac_neumann && mn == VACUUM))) mask |= 1u << q;
  }
  code[idx] = (uint16_t)((unsigned)m | (mask << 3));
}

// One Jacobi pass: the diagonal h^2/(alpha_m dt) + 6, less one per Neumann
// neighbour (subtracted at once: below 2^53 every subtraction of 1 is exact);
// x of the open neighbours added to b in face order.  Four cells per
// thread, their loads in flight together, and the six diagonals from the host:
// 256^3 72 -> 59 us a pass, where every block of 256 cells had formed a
// table of them.
struct HeatDiag {
  double d[6];
};
constexpr int HJ = 4;
__global__ void __launch_bounds__(256)
    k_heat_jacobi(Grid g, const float* __restrict__ x, float* __restrict__ xn, const float* __restrict__ b,
                  const uint16_t* __restrict__ code, HeatDiag hd) {
  const int64_t i0 = (int64_t)blockIdx.x * (256 * HJ) + threadIdx.x;
  const int64_t sx = (int64_t)g.ny * g.nz, sy = g.nz;
  const int64_t st[6] = {sx, sy, 1, -sx, -sy, -1};
  unsigned cd[HJ];
  float bv[HJ];
#pragma unroll
  for (int u = 0; u < HJ; ++u) {
    const int64_t idx = i0 + u * 256;
    cd[u] = idx < g.G ? code[idx] : 7u;
    bv[u] = idx < g.G ? b[idx] : 0.0f;
  }
  // the neighbour loads issued together (a closed face reads the cell)
  float xv[HJ][6];
#pragma unroll
  for (int u = 0; u < HJ; ++u) {
    const unsigned mask = (cd[u] & 7u) == 7u ? 0u : cd[u] >> 3;
    const int64_t idx = min(i0 + u * 256, g.G - 1);
#pragma unroll
    for (int q = 0; q < 6; ++q) xv[u][q] = x[(mask & (1u << q)) ? idx + st[q] : idx];
  }
#pragma unroll
  for (int u = 0; u < HJ; ++u) {
    const int64_t idx = i0 + u * 256;
    if (idx >= g.G) return;
    const unsigned m = cd[u] & 7u, mask = cd[u] >> 3;
    double s = (double)bv[u];
#pragma unroll
    for (int q = 0; q < 6; ++q)
      if (mask & (1u << q)) s += (double)xv[u][q];
    double d = hd.d[0];
#pragma unroll
    for (int t = 1; t < 6; ++t) d = m == (unsigned)t ? hd.d[t] : d;
    d -= (double)(6 - __popc(mask));
    xn[idx] = m == 7u ? 0.0f : (float)(s / d);
  }
}

__global__ void k_heat_start(int64_t G, const float* __restrict__ tsave, const int8_t* __restrict__ mark,
                             float* __restrict__ x) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < G) x[idx] = (mark[idx] == BOUNDARY) ? 0.0f : tsave[idx];
}

// setBoundaryHeat spray_k.cu:4585-4605 (reads the pass's input) ; compTpChange 4607-4617
__global__ void k_heat_post(Grid g, const float* __restrict__ tin, float* __restrict__ tp,
                            const float* __restrict__ tsave, float* __restrict__ tch, const int8_t* __restrict__ mark,
                            int extend) {
  CELL_LOOP_HEAD
  float t = tin[idx];
  if (extend) {
    if (i == g.nx - 1) t = tin[cid(g, i - 1, j, k)];
    else if (i == 0) t = tin[cid(g, i + 1, j, k)];
    else if (j == g.ny - 1) t = tin[cid(g, i, j - 1, k)];
    else if (j == 0) t = tin[cid(g, i, j + 1, k)];
    else if (k == g.nz - 1) t = tin[cid(g, i, j, k - 1)];
    else if (k == 0) t = tin[cid(g, i, j, k + 1)];
  }
  tp[idx] = t;
  tch[idx] = (mark[idx] != BOUNDARY) ? t - tsave[idx] : 0.0f;
}

// ---------------- solid distance + velocity (a15 support) ----------------
// initSolidPhi spray_k.cu:724-744
__global__ void k_init_solid_phi(int64_t G, const uint8_t* __restrict__ cmask, float* __restrict__ phi, float big) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx < G) phi[idx] = (cmask[idx] & M_SOLID) ? -0.5f : big;
}

// ---------------- marching cubes (a18) ----------------
// A node lattice: nodes (nx, ny, nz), voxels one fewer per axis; node
// (i,j,k) at index (i*ny + j)*nz + k, position (i + off) * h + origin.  The
// level-set source uses cell centres of the N grid (off 0.5); the particle
// sources the (2N+1)^3 nodes of spacing dx/2 (off 0, spray_k.cu:1649).
struct McGrid {
  int nx, ny, nz;
  int64_t N, V;
  float h, off, x0, y0, z0;
};
__device__ __forceinline__ int64_t nid(const McGrid& m, int i, int j, int k) {
  return ((int64_t)i * m.ny + j) * m.nz + k;
}

// Cube edges as (di, dj, dk, slot): the edge starts at node (i+di, j+dj, k+dk)
// and runs along +x (slot 1), +y (slot 0) or +z (slot 2); its id is
// 3 * node + slot, the numbering of GetEdgeID (spray_k.cu:1920-1957).
__constant__ int c_eo[12][4] = {{0, 0, 0, 1}, {1, 0, 0, 0}, {0, 1, 0, 1}, {0, 0, 0, 0}, {0, 0, 1, 1}, {1, 0, 1, 0},
                                {0, 1, 1, 1}, {0, 0, 1, 0}, {0, 0, 0, 2}, {1, 0, 0, 2}, {1, 1, 0, 2}, {0, 1, 0, 2}};
__constant__ signed char c_tri[256][16];
__constant__ unsigned char c_nv[256];

// classifyVoxel, spray_k.cu:1853-1888 (isoValue 0)
__device__ __forceinline__ uint32_t mc_case_of(const McGrid& m, const float* f, int i, int j, int k) {
  const int64_t si = (int64_t)m.ny * m.nz, sj = m.nz;
  const float* b = f + nid(m, i, j, k);
  float v[8] = {b[0], b[si], b[si + sj], b[sj], b[1], b[si + 1], b[si + sj + 1], b[sj + 1]};
  uint32_t ci = 0;
#pragma unroll
  for (int q = 0; q < 8; ++q) ci += (uint32_t)(v[q] < 0.0f) << q;
  return ci;
}

// Case index, triangle count and the edges its triangles use
// (markActiveEdge_MC, spray_k.cu:2172-2220).
__global__ void k_mc_classify(McGrid m, const float* __restrict__ f, uint8_t* __restrict__ cases,
                              uint32_t* __restrict__ tcount, uint32_t* __restrict__ edge_used,
                              uint32_t* __restrict__ active) {
  int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int nv = 0;
  if (v < m.V) {
    int i, j, k;
    ijk3(v, m.ny - 1, m.nz - 1, i, j, k);
    uint32_t ci = mc_case_of(m, f, i, j, k);
    cases[v] = (uint8_t)ci;
    nv = c_nv[ci];
    tcount[v] = (uint32_t)(nv / 3);
    for (int t = 0; t < nv; ++t) {
      int e = c_tri[ci][t];
      edge_used[3 * nid(m, i + c_eo[e][0], j + c_eo[e][1], k + c_eo[e][2]) + c_eo[e][3]] = 1u;
    }
  }
  // active voxels: one add per block, spread over NSPREAD counters
  const int cnt = __syncthreads_count(nv > 0);
  if (threadIdx.x == 0 && cnt) atomicAdd(active + (blockIdx.x % NSPREAD) * SPREAD_STRIDE, (uint32_t)cnt);
}

// vertexInterp (spray_k.cu:1903-1908) along each used edge, from its start
// node p0 to p1 = p0 + h along the edge (generateTriangles_indices,
// spray_k.cu:2092-2117); vid holds the exclusive scan of the used flags.  The
// reference writes a shared edge's vertex from whichever voxel comes last;
// here every edge is interpolated once, in the + direction.
__global__ void k_mc_verts(McGrid m, const float* __restrict__ f, const uint32_t* __restrict__ used,
                           const uint32_t* __restrict__ vid, float* __restrict__ verts,
                           uint32_t* __restrict__ vedge) {
  int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= 3 * m.N || !used[e]) return;
  const int64_t n = e / 3;
  const int slot = (int)(e % 3);
  const int a = slot == 1 ? 0 : (slot == 0 ? 1 : 2);
  int i, j, k;
  ijk3(n, m.ny, m.nz, i, j, k);
  const int i2 = i + (a == 0), j2 = j + (a == 1), k2 = k + (a == 2);
  const float f0 = f[n], f1 = f[nid(m, i2, j2, k2)];
  const float t = (0.0f - f0) / (f1 - f0);
  const float h = m.h;
  const float p0x = ((float)i + m.off) * h + m.x0, p0y = ((float)j + m.off) * h + m.y0,
              p0z = ((float)k + m.off) * h + m.z0;
  const float p1x = a == 0 ? p0x + h : p0x, p1y = a == 1 ? p0y + h : p0y, p1z = a == 2 ? p0z + h : p0z;
  const uint32_t o = vid[e];
  vedge[o] = (uint32_t)e;
  verts[3 * (int64_t)o + 0] = p0x + t * (p1x - p0x);
  verts[3 * (int64_t)o + 1] = p0y + t * (p1y - p0y);
  verts[3 * (int64_t)o + 2] = p0z + t * (p1z - p0z);
}

// generateTriangles_indices spray_k.cu:2074-2170 (indices = scanned edge ids)
__global__ void k_mc_tris(McGrid m, const uint8_t* __restrict__ cases, const uint32_t* __restrict__ toff,
                          const uint32_t* __restrict__ vid, uint32_t* __restrict__ tris) {
  int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= m.V) return;
  uint32_t ci = cases[v];
  int nv = c_nv[ci];
  if (!nv) return;
  int i, j, k;
  ijk3(v, m.ny - 1, m.nz - 1, i, j, k);
  int64_t w = 3 * (int64_t)toff[v];
  for (int t = 0; t < nv; ++t) {
    int e = c_tri[ci][t];
    tris[w + t] = vid[3 * nid(m, i + c_eo[e][0], j + c_eo[e][1], k + c_eo[e][2]) + c_eo[e][3]];
  }
}

// The triangles around one vertex, in the order of the triangle list: the
// vertex lies on edge e, which the (at most) 4 voxels around it share; their
// index order is the list's order, and within a voxel its triangles follow
// the table.  fn(i1, i2, i3) sees every triangle that holds the vertex.
template <class Fn>
__device__ __forceinline__ void mc_vertex_triangles(const McGrid& m, uint32_t e, const uint8_t* __restrict__ cases,
                                                    const uint32_t* __restrict__ toff,
                                                    const uint32_t* __restrict__ tris, uint32_t v, Fn fn) {
  const int64_t n = e / 3;
  const int slot = (int)(e % 3);
  int i, j, k;
  ijk3(n, m.ny, m.nz, i, j, k);
  const int VX = m.nx - 1, VY = m.ny - 1, VZ = m.nz - 1;
  for (int q = 0; q < 4; ++q) {
    const int a = q >> 1, b = q & 1;
    int vi, vj, vk;
    if (slot == 1) { vi = i; vj = j - 1 + a; vk = k - 1 + b; }       // x edge
    else if (slot == 0) { vi = i - 1 + a; vj = j; vk = k - 1 + b; }  // y edge
    else { vi = i - 1 + a; vj = j - 1 + b; vk = k; }                  // z edge
    if (vi < 0 || vi >= VX || vj < 0 || vj >= VY || vk < 0 || vk >= VZ) continue;
    const int64_t vox = ((int64_t)vi * VY + vj) * VZ + vk;
    const int nt = c_nv[cases[vox]] / 3;
    const int64_t t0 = toff[vox];
    for (int t = 0; t < nt; ++t) {
      const uint32_t i1 = tris[3 * (t0 + t)], i2 = tris[3 * (t0 + t) + 1], i3 = tris[3 * (t0 + t) + 2];
      if (i1 == v || i2 == v || i3 == v) fn(i1, i2, i3);
    }
  }
}

// calNormals, spray.cu:981-997: the sum of cross(p2 - p1, p3 - p1) over the
// vertex's triangles (calnormal_k, spray_k.cu:2223-2250, adds them with
// atomics; here in the list's order), normalised when nonzero
// (normalizeTriangleNor_k, 2252-2261).
__global__ void k_mc_normals(McGrid m, const uint32_t* __restrict__ vedge, const uint8_t* __restrict__ cases,
                             const uint32_t* __restrict__ toff, const uint32_t* __restrict__ tris,
                             const float* __restrict__ verts, float* __restrict__ nrm, int64_t nv) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  float nx = 0.0f, ny = 0.0f, nz = 0.0f;
  mc_vertex_triangles(m, vedge[v], cases, toff, tris, (uint32_t)v, [&](uint32_t i1, uint32_t i2, uint32_t i3) {
    const float* a = verts + 3 * (int64_t)i1;
    const float* b = verts + 3 * (int64_t)i2;
    const float* c = verts + 3 * (int64_t)i3;
    const float ux = b[0] - a[0], uy = b[1] - a[1], uz = b[2] - a[2];
    const float wx = c[0] - a[0], wy = c[1] - a[1], wz = c[2] - a[2];
    nx = nx + (uy * wz - uz * wy);
    ny = ny + (uz * wx - ux * wz);
    nz = nz + (ux * wy - uy * wx);
  });
  const float len = sqrtf(nx * nx + ny * ny + nz * nz);
  if (len > 0.0f) {
    const float inv = 1.0f / len;
    nx = nx * inv;
    ny = ny * inv;
    nz = nz * inv;
  }
  nrm[3 * v] = nx;
  nrm[3 * v + 1] = ny;
  nrm[3 * v + 2] = nz;
}

// smoothMesh, spray.cu:1271-1288, one iteration: each vertex gathers the
// edge vectors to the other two corners of its triangles (in the order of
// smooth_computedisplacement, spray_k.cu:2408-2427) and moves by
// lambda * sum / count (smooth_addDisplacement, 2429-2440).  The
// reference's second, mu = -0.53 pass finds the sums already cleared by the
// first and does nothing; so here.  Positions of the pass's input are read.
__global__ void k_mc_smooth(McGrid m, const uint32_t* __restrict__ vedge, const uint8_t* __restrict__ cases,
                            const uint32_t* __restrict__ toff, const uint32_t* __restrict__ tris,
                            const float* __restrict__ vin, float* __restrict__ vout, int64_t nv, float lambda) {
  const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (v >= nv) return;
  float dx = 0.0f, dy = 0.0f, dz = 0.0f;
  int w = 0;
  const float* pv = vin + 3 * v;
  mc_vertex_triangles(m, vedge[v], cases, toff, tris, (uint32_t)v, [&](uint32_t i1, uint32_t i2, uint32_t i3) {
    const uint32_t o1 = (i1 == (uint32_t)v) ? i2 : i1;
    const uint32_t o2 = (i3 == (uint32_t)v) ? i2 : i3;
    const float* a = vin + 3 * (int64_t)o1;
    const float* b = vin + 3 * (int64_t)o2;
    dx = dx + (a[0] - pv[0]);
    dy = dy + (a[1] - pv[1]);
    dz = dz + (a[2] - pv[2]);
    dx = dx + (b[0] - pv[0]);
    dy = dy + (b[1] - pv[1]);
    dz = dz + (b[2] - pv[2]);
    w += 2;
  });
  float x = pv[0], y = pv[1], z = pv[2];
  if (w > 0) {
    const float fw = (float)w;
    x = x + lambda * dx / fw;
    y = y + lambda * dy / fw;
    z = z + lambda * dz / fw;
  }
  vout[3 * v] = x;
  vout[3 * v + 1] = y;
  vout[3 * v + 2] = z;
}

// Node field of a particle source, one thread per node of the (2N+1)^3
// lattice, reading the 4x4x4 cells of the 2N lists around it (di, dj, dk in
// [-2, 1]):
//  MPF_MC_LIQUID_GAS  genWaterDensfield_liquidAndGas + sumcelldens_liquidAndGas
//                     (spray_k.cu:1595-1686): FLUID/AIR/AIRSOLO within R = 2h,
//                     w = (R^2 - d^2)^3, phi = h/2 - |x - centre| (-h/2 when
//                     no particle), lattice faces -1000;
//  MPF_MC_GAS         genWaterDensfield_Gas + sumcelldens_Gas (1528-1593): AIR
//                     and, when airsolo, AIRSOLO; r = 0.8h;
//  MPF_MC_SOLID       genWaterDensfield_GY + sumcelldens3 (1688-1772): SOLID
//                     within R = h, w = max((1 - (d/4h)^2)^3, 0), phi =
//                     |x - centre| - 0.75h f(Ev) with the centre measured
//                     from the origin (the reference's centertmp is zero),
//                     lattice faces min(phi, -10).
// Per cell the weighted positions are summed from zero and added to the
// centre, the weights accumulate directly (the reference's order).
template <int SRC>
__global__ void k_mc_density(McGrid m, Grid g2, const f3* __restrict__ pos, const int8_t* __restrict__ flag,
                             const uint32_t* __restrict__ cs, const uint32_t* __restrict__ ce,
                             float* __restrict__ out, int airsolo) {
  const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= m.N) return;
  int i, j, k;
  ijk3(idx, m.ny, m.nz, i, j, k);
  const float h = m.h;
  const float px = ((float)i + m.off) * h + m.x0, py = ((float)j + m.off) * h + m.y0,
              pz = ((float)k + m.off) * h + m.z0;
  const float R = (SRC == MPF_MC_SOLID) ? h : h * 2.0f;
  float cx = 0.0f, cy = 0.0f, cz = 0.0f, wsum = 0.0f;
  for (int di = -2; di <= 1; ++di)
    for (int dj = -2; dj <= 1; ++dj)
      for (int dk = -2; dk <= 1; ++dk) {
        const int a = i + di, b = j + dj, q = k + dk;
        if (a < 0 || a > g2.nx - 1 || b < 0 || b > g2.ny - 1 || q < 0 || q > g2.nz - 1) continue;
        const int64_t cell = ((int64_t)a * g2.ny + b) * g2.nz + q;
        const uint32_t s = cs[cell];
        if (s == MPF_CELL_UNDEF) continue;
        const uint32_t e = ce[cell];
        float rx = 0.0f, ry = 0.0f, rz = 0.0f;
        for (uint32_t p = s; p < e; ++p) {
          const int8_t fl = flag[p];
          bool take;
          if (SRC == MPF_MC_LIQUID_GAS) take = fl == AIR || fl == AIRSOLO || fl == FLUID;
          else if (SRC == MPF_MC_GAS) take = fl == AIR || (fl == AIRSOLO && airsolo);
          else take = fl == SOLID;
          if (!take) continue;
          const f3 x = pos[p];
          const float dx = x.x - px, dy = x.y - py, dz = x.z - pz;
          const float dis = sqrtf(dx * dx + dy * dy + dz * dz);
          if (dis < R) {
            float w;
            if (SRC == MPF_MC_SOLID) {
              w = dis / (4.0f * h);
              w = 1.0f - w * w;
              w = fmaxf(w * w * w, 0.0f);
            } else {
              w = R * R - dis * dis;
              w = w * w * w;
            }
            rx = rx + x.x * w;
            ry = ry + x.y * w;
            rz = rz + x.z * w;
            wsum = wsum + w;
          }
        }
        cx = cx + rx;
        cy = cy + ry;
        cz = cz + rz;
      }
  const float r = (SRC == MPF_MC_LIQUID_GAS) ? 0.5f * h : (SRC == MPF_MC_GAS ? 0.8f * h : 0.75f * h);
  float phi;
  if (wsum > 0.0f) {
    cx = cx / wsum;
    cy = cy / wsum;
    cz = cz / wsum;
    const float ex = px - cx, ey = py - cy, ez = pz - cz;
    const float len = sqrtf(ex * ex + ey * ey + ez * ez);
    if (SRC == MPF_MC_SOLID) {
      const float thigh = 0.51f, tlow = 0.49f;
      const float Ev = fmaxf(cx, fmaxf(cy, cz)) / (4.0f * h);
      const float gamma = (thigh - Ev) / (thigh - tlow);
      const float fr = (Ev < tlow) ? 1.0f : gamma * gamma * gamma - 3.0f * gamma * gamma + 3.0f * gamma;
      phi = len - r * fr;
    } else {
      phi = r - len;
    }
  } else {
    phi = -r;
  }
  const bool face = i == 0 || j == 0 || k == 0 || i == m.nx - 1 || j == m.ny - 1 || k == m.nz - 1;
  if (face) phi = (SRC == MPF_MC_SOLID) ? fminf(phi, -10.0f) : -1000.0f;
  out[idx] = phi;
}

}  // namespace

// ================= host stage drivers =================
// N two-buffer passes over one field or two: from tmp into phi and back, an odd
// number so that the last is into phi.  flags: two sets of tile flags.
struct SweepJob {
  float* phi;
  float* tmp;
  const int8_t* mark;
  int typeflag;
  uint8_t* flags;
};
template <int N>
static void sweep_n(Ctx& c, const SweepJob* jobs, int njobs) {
  static_assert(N % 2 == 1, "the last pass writes phi");
  const uint32_t ntj = (uint32_t)((c.g.ny + SW_J - 1) / SW_J), ntk = (uint32_t)((c.g.nz + SW_K - 1) / SW_K);
  const int64_t nt = sweep_tiles(c.g);
  const int64_t nwaves = (nt + SW_L - 1) / SW_L;
  for (int it = 0; it < N; ++it) {
    SweepPass p[2];
    for (int q = 0; q < 2; ++q) {
      const SweepJob& j = jobs[q < njobs ? q : 0];
      p[q] = SweepPass{(it & 1) ? j.phi : j.tmp, (it & 1) ? j.tmp : j.phi, j.mark, j.typeflag,
                       it == 0 ? nullptr : j.flags + ((it - 1) & 1) * nt, j.flags + (it & 1) * nt};
    }
    launch(c, njobs == 1 ? "sweep_one" : "sweep", dim3((unsigned)((nwaves + 3) / 4), njobs), dim3(256), 0, k_sweep,
           c.g, p[0], p[1], ntj, ntk, (uint32_t)nt);
  }
}

// Both level sets together; the second takes its scratch values from a face
// field's scratch, its marks from the liquid P2G's (free here) and its flags
// from the extrapolation's (at least three sets of face tiles).
static void redistance(Ctx& c) {
  const int64_t G = c.g.G;
  int8_t* mark2 = (int8_t*)c.p2g_parts;
  const LsPair p{{c.lsfluid, c.lsair}, {c.ctmp, c.ftmp[0]}, {c.mark, mark2}};
  const SweepJob jobs[2] = {{c.lsfluid, c.ctmp, c.mark, FLUID, c.sflag},
                            {c.lsair, c.ftmp[0], mark2, FLUID, c.sflag + 2 * sweep_tiles(c.g)}};
  launch(c, "ls_prepare", dim3(nblocks(G, 256), 2), dim3(256), 0, k_ls_prepare<false>, G, p, c.g.h);
  sweep_n<5>(c, jobs, 2);
  launch(c, "ls_prepare", dim3(nblocks(G, 256), 2), dim3(256), 0, k_ls_prepare<true>, G, p, c.g.h);
  sweep_n<5>(c, jobs, 2);
}

// Brick summary of the occupancy masks (after every change of the masks).
void run_bricks(Ctx& c) {
  const int bx = (c.g.nx + 3) / 4, by = (c.g.ny + 3) / 4, bz = (c.g.nz + 3) / 4;
  const int64_t NB = nbricks(c.g);
  launch(c, "bricks", dim3(nblocks(NB, 256)), dim3(256), 0, k_brick_or, c.g, (const uint8_t*)c.cmask, c.bmask, bx, by,
         bz);
  launch(c, "bricks", dim3(nblocks(NB, 256)), dim3(256), 0, k_brick_dilate, (const uint8_t*)c.bmask, c.bmask + NB, bx,
         by, bz);
}

// Row bits of the current masks, in the scratch of the liquid P2G (a quarter
// byte a cell and the border; it holds 49 bytes a cell of 4x8x8 tiles): valid
// until the next P2G or solve.
RowBits run_row_bits(Ctx& c) {
  const int nw = (c.g.nz + 4 + 63) / 64;
  const int64_t words = (int64_t)(c.g.nx + 4) * (c.g.ny + 4) * nw;
  uint64_t* fb = (uint64_t*)c.p2g_parts;
  uint64_t* ab = fb + words;
  launch(c, "row_bits", dim3(nblocks(words * 64, 256)), dim3(256), 0, k_row_bits, c.g, (const uint8_t*)c.cmask, fb, ab,
         nw, (uint32_t*)(ab + words));
  return RowBits{fb, ab, nw, c.g.ny + 4, (uint32_t*)(ab + words)};
}
void run_air_regular(Ctx& c, const RowBits& rb) {
  const int cur = c.cur;
  launch(c, "air_regular", dim3(nblocks((c.P + 15) / 16, 256)), dim3(256), 0, k_air_regular, c.g, c.P,
         (const f3*)c.pos[cur], (const f3*)c.vel[cur], (const float*)c.mass[cur], (const int8_t*)c.flag[cur], rb.odd);
}

void run_levelset(Ctx& c) {
  const int64_t G = c.g.G;
  const int cur = c.cur;
  const int64_t NB = nbricks(c.g);
  const RowBits rb = run_row_bits(c);
  launch(c, "genlevelset", dim3(nblocks(G, 256)), dim3(256), 0, k_genlevelset, c.g, (const f3*)c.pos[cur],
         (const int8_t*)c.flag[cur], (const uint32_t*)c.cstart, (const uint32_t*)c.cend, (const uint8_t*)c.cmask,
         (const uint8_t*)(c.bmask + NB), rb, c.lsfluid, c.lsair, c.mark);
  redistance(c);
  launch(c, "merge_mark", dim3(nblocks(G, 256)), dim3(256), 0, k_merge, c.g, c.lsfluid, c.lsair, c.lsmerge, c.mark);
  launch(c, "phigrad", dim3(nblocks(G, 256)), dim3(256), 0, k_phigrad, c.g, (const float*)c.lsmerge, c.phig[0],
         c.phig[1], c.phig[2]);
  if (c.cfg.flags_from_counts)
    launch(c, "mark_counts", dim3(nblocks(G, 256)), dim3(256), 0, k_mark_counts, c.g, (const uint32_t*)c.cstart,
           (const uint32_t*)c.cend, (const int8_t*)c.flag[cur], c.mark);
  if (c.cfg.solid_constraint)
    launch(c, "mark_solid", dim3(nblocks(G, 256)), dim3(256), 0, k_mark_solid, c.g, (const uint32_t*)c.cstart,
           (const uint32_t*)c.cend, (const int8_t*)c.flag[cur], (const uint8_t*)c.cmask, c.mark);
}

static unsigned face_blocks(const Grid& g) { return nblocks(std::max(g.FX, std::max(g.FY, g.FZ)), 256); }

static void p2g_air(Ctx& c, float* const* out, float* const* out2) {
  const int cur = c.cur;
  P2GOut o;
  for (int a = 0; a < 3; ++a) {
    o.u[a] = out[a];
    o.u2[a] = out2 ? out2[a] : nullptr;
  }
  const RowBits rb = run_row_bits(c);
  if (c.own_sort) run_air_regular(c, rb);
  // lists given by the caller need not be consecutive along a row
  auto kern = c.own_sort ? k_p2g_air<true> : k_p2g_air<false>;
  launch(c, "p2g_air", dim3(face_blocks(c.g), 3), dim3(256), 0, kern, c.g,
         (const f3*)c.pos[cur], (const f3*)c.vel[cur], (const float*)c.mass[cur], (const int8_t*)c.flag[cur],
         (const uint32_t*)c.cstart, (const uint32_t*)c.cend, rb, (const uint8_t*)(c.bmask + nbricks(c.g)), o);
}

static void p2g_liquid(Ctx& c, float* const* out, float* const* out2 = nullptr, const float* band = nullptr,
                       float big = 0.0f) {
  const int cur = c.cur;
  const int ntx = (c.g.nx + ST_X - 1) / ST_X, nty = (c.g.ny + ST_Y - 1) / ST_Y, ntz = (c.g.nz + ST_Z - 1) / ST_Z;
  launch(c, band ? "p2g_solid_band" : "p2g_liquid", dim3((unsigned)(ntx * nty * ntz)), dim3(ST_CELLS), 0,
         k_p2g_tile, c.g, (const f3*)c.pos[cur], (const f3*)c.vel[cur], (const float*)c.mass[cur],
         (const int8_t*)c.flag[cur], (const uint32_t*)c.cstart, (const uint32_t*)c.cend, (const uint8_t*)c.cmask,
         c.p2g_parts, ntx, nty, ntz, band, big, (const uint8_t*)(c.bmask + nbricks(c.g)));
  P2GOut o;
  for (int a = 0; a < 3; ++a) {
    o.u[a] = out[a];
    o.u2[a] = out2 ? out2[a] : nullptr;
  }
  launch(c, band ? "p2g_solid_collect" : "p2g_collect", dim3(face_blocks(c.g), 3), dim3(256), 0, k_p2g_collect, c.g,
         (const float*)c.p2g_parts, ntx, nty, ntz, o, band, big);
}

static_assert(2 * ST_RTOT >= 12 * ST_CELLS, "the solver's slow-row weights (six FP64 values a cell) fit as well");
int64_t p2g_parts_floats(const Grid& g) {
  const int64_t nt = (int64_t)((g.nx + ST_X - 1) / ST_X) * ((g.ny + ST_Y - 1) / ST_Y) * ((g.nz + ST_Z - 1) / ST_Z);
  return nt * 2 * ST_RTOT;
}

void run_p2g(Ctx& c) {
  p2g_liquid(c, c.wu, c.wuo);
  p2g_air(c, c.au, c.auo);
}

void run_solid_phi_and_velocity(Ctx& c) {
  const int64_t G = c.g.G;
  launch(c, "init_solid_phi", dim3(nblocks(G, 256)), dim3(256), 0, k_init_solid_phi, G, (const uint8_t*)c.cmask,
         c.ctmp, (float)(3 * c.g.nx));
  const SweepJob job{c.phisolid, c.ctmp, c.mark, -1, c.sflag};
  sweep_n<3>(c, &job, 1);
  // solid velocity only where the collision response can read it
  p2g_liquid(c, c.su, nullptr, c.phisolid, (float)(3 * c.g.nx));
}

static Faces6 faces6(Ctx& c) { return Faces6{{c.wu[0], c.wu[1], c.wu[2], c.au[0], c.au[1], c.au[2]}}; }

void run_extrapolate_bc(Ctx& c, bool recompute_phi) {
  const int64_t G = c.g.G;
  const int64_t fc[3] = {c.g.FX, c.g.FY, c.g.FZ};
  if (recompute_phi) {
    float* tmp2 = c.ftmp[0];
    launch(c, "initphi", dim3(nblocks(G, 256)), dim3(256), 0, k_initphi, G, (const int8_t*)c.mark, c.ctmp, (int8_t)AIR,
           tmp2, (int8_t)FLUID, (float)(c.g.nx * 3));
    const SweepJob jobs[2] = {{c.phiair, c.ctmp, c.mark, AIR, c.sflag},
                              {c.phifluid, tmp2, c.mark, FLUID, c.sflag + 2 * sweep_tiles(c.g)}};
    sweep_n<3>(c, jobs, 2);
  }
  // Two passes: u -> scratch, scratch -> u; the first records per-tile changes
  // (a flag set per field), the second skips the tiles they leave unchanged.
  // The air faces' scratch is the liquid P2G's (12 floats a cell, three face
  // fields are at most 6).  A pass that computes every tile gives each wave
  // SW_U1 tiles (more waves in flight for its two rounds of loads); a pass
  // that skips reads the flags of SW_L tiles per wave.
  const Faces6 u = faces6(c);
  SweepU s;
  float* air = c.p2g_parts;
  uint8_t* fl = c.sflag + 2 * sweep_tiles(c.g);
  float* tmp[6];
  int64_t most = 0;
  for (int q = 0; q < 6; ++q) {
    const int a = q % 3;
    tmp[q] = q < 3 ? c.ftmp[a] : air;
    if (q >= 3) air += fc[a];
    s.flags[q] = fl;
    fl += face_tiles(c.g, a);
    most = std::max(most, face_tiles(c.g, a));
  }
  s.ls[0] = c.phifluid;
  s.sf[0] = FLUID;
  s.ls[1] = c.phiair;
  s.sf[1] = AIR;
  for (int it = 0; it < 2; ++it) {
    for (int q = 0; q < 6; ++q) {
      s.u[q] = it == 0 ? u.u[q] : tmp[q];
      s.out[q] = it == 0 ? tmp[q] : u.u[q];
    }
    const int per_wave = it ? SW_L : SW_U1;
    const int64_t nwaves = (most + per_wave - 1) / per_wave;
    launch(c, "sweep_u", dim3((unsigned)((nwaves + 3) / 4), 6), dim3(256), 0,
           it == 0 ? k_sweep_u<true> : k_sweep_u<false>, c.g, s, (const int8_t*)c.mark, per_wave);
  }
  launch(c, "bc", dim3(face_blocks(c.g), 6), dim3(256), 0, k_bc, c.g, u, (const int8_t*)c.mark);
}

void run_divergence(Ctx& c) {
  const int64_t G = c.g.G;
  if (c.cfg.precision == MPF_FP64)
    launch(c, "divergence", dim3(nblocks(G, 256)), dim3(256), 0, k_divergence<double>, c.g, (const float*)c.wu[0],
           (const float*)c.wu[1], (const float*)c.wu[2], (const float*)c.au[0], (const float*)c.au[1],
           (const float*)c.au[2], (const int8_t*)c.mark, (const float*)c.lsmerge, c.cfg.solid_constraint,
           (double*)c.div);
  else
    launch(c, "divergence", dim3(nblocks(G, 256)), dim3(256), 0, k_divergence<float>, c.g, (const float*)c.wu[0],
           (const float*)c.wu[1], (const float*)c.wu[2], (const float*)c.au[0], (const float*)c.au[1],
           (const float*)c.au[2], (const int8_t*)c.mark, (const float*)c.lsmerge, c.cfg.solid_constraint,
           (float*)c.div);
}

template <class R>
static void subgrad_t(Ctx& c) {
  launch(c, "subgrad", dim3(face_blocks(c.g), 6), dim3(256), 0, k_subgrad<R>, c.g, faces6(c), (const R*)c.press,
         (const int8_t*)c.mark, (int)(c.cfg.op == MPF_OPERATOR_VARDENS), 1.0 / (double)c.cfg.rho_liquid,
         1.0 / (double)c.cfg.rho_air, (int)c.cfg.solid_constraint);
}

void run_subgrad(Ctx& c) {
  if (c.cfg.precision == MPF_FP32) subgrad_t<float>(c);
  else subgrad_t<double>(c);
}

void run_heat_grid_pre(Ctx& c) {
  const mpf_config& k = c.cfg;
  const int64_t G = c.g.G;
  const int ntx = (c.g.nx + ST_X - 1) / ST_X, nty = (c.g.ny + ST_Y - 1) / ST_Y, ntz = (c.g.nz + ST_Z - 1) / ST_Z;
  static_assert(HR <= ST_RTOT, "heat regions fit the P2G tile buffer");
  launch(c, "heat_p2g", dim3((unsigned)(ntx * nty * ntz)), dim3(ST_CELLS), 0, k_heat_tile, c.g,
         (const f3*)c.pos[c.cur], (const float*)c.temp[c.cur], (const uint32_t*)c.cstart, (const uint32_t*)c.cend,
         (const uint8_t*)c.cmask, c.p2g_parts, ntx, nty, ntz);
  launch(c, "heat_collect", dim3(nblocks(G, 256)), dim3(256), 0, k_heat_collect, c.g, (const float*)c.p2g_parts, ntx,
         nty, ntz, k.default_temperature, c.tp);
  launch(c, "heat_pre", dim3(nblocks(G, 256)), dim3(256), 0, k_heat_pre, c.g, c.tp, c.tsave, c.ctmp,
         (const int8_t*)c.mark, k.heat_add_bottom, k.heat_increase_bottom, k.heat_bottom_clamp, k.heat_alpha[0],
         k.heat_alpha[1], k.heat_alpha[2], k.heat_alpha[3], k.heat_alpha[4], k.heat_alpha[5], k.dt);
}

void run_heat_jacobi(Ctx& c, int iters) {
  const mpf_config& k = c.cfg;
  const int64_t G = c.g.G;
  float* x = (float*)c.vx;
  float* xn = (float*)c.vr;
  uint16_t* code = (uint16_t*)c.ctmp_u32;
  HeatDiag hd;
  for (int t = 0; t < 6; ++t) hd.d[t] = (double)c.g.h * (double)c.g.h / (double)k.heat_alpha[t] / (double)k.dt + 6.0;
  launch(c, "heat_start", dim3(nblocks(G, 256)), dim3(256), 0, k_heat_start, G, (const float*)c.tsave,
         (const int8_t*)c.mark, iters > 0 ? x : c.tp);
  launch(c, "heat_code", dim3(nblocks(G, 256)), dim3(256), 0, k_heat_code, c.g, (const int8_t*)c.mark, code,
         k.heat_vacuum_neumann);
  for (int it = 0; it < iters; ++it) {
    if (it == iters - 1) xn = c.tp;
    launch(c, "heat_jacobi", dim3(nblocks(G, 256 * HJ)), dim3(256), 0, k_heat_jacobi, c.g, (const float*)x, xn,
           (const float*)c.ctmp, (const uint16_t*)code, hd);
    float* t = x; x = xn; xn = t;
  }
}

void run_heat_grid_post(Ctx& c) {
  const int64_t G = c.g.G;
  hipMemcpyAsync(c.ctmp, c.tp, (size_t)G * 4, hipMemcpyDeviceToDevice, c.stream);
  launch(c, "heat_post", dim3(nblocks(G, 256)), dim3(256), 0, k_heat_post, c.g, (const float*)c.ctmp, c.tp,
         (const float*)c.tsave, c.tpchange, (const int8_t*)c.mark, c.cfg.heat_extend_boundary);
}

int run_marching_cubes(Ctx& c, mpf_mc_info* info) {
  static bool tables_loaded[64] = {};  // per device; the tables are constants
  const int dslot = c.device >= 0 && c.device < 64 ? c.device : 0;
  if (!tables_loaded[dslot]) {
    if (hipMemcpyToSymbol(HIP_SYMBOL(c_tri), MC_TRI_TABLE, sizeof(MC_TRI_TABLE)) != hipSuccess ||
        hipMemcpyToSymbol(HIP_SYMBOL(c_nv), MC_NUM_VERTS, sizeof(MC_NUM_VERTS)) != hipSuccess) {
      c.err = "marching cubes tables: hipMemcpyToSymbol failed";
      return MPF_HIP_ERROR;
    }
    tables_loaded[dslot] = true;
  }
  const int src = c.cfg.mc_source;
  McGrid m{};
  const float* f;
  if (src == MPF_MC_LEVELSET) {
    m.nx = c.g.nx; m.ny = c.g.ny; m.nz = c.g.nz;
    m.h = c.g.h;
    m.off = 0.5f;
    f = c.lsfluid;
  } else {
    m.nx = c.g2.nx + 1; m.ny = c.g2.ny + 1; m.nz = c.g2.nz + 1;
    m.h = c.cfg.dx / 2.0f;  // cellsize.x / (NXMC / NX), spray_k.cu:1640
    m.off = 0.0f;
    f = c.mc_field;
  }
  m.x0 = c.g.gx0; m.y0 = c.g.gy0; m.z0 = c.g.gz0;
  m.N = (int64_t)m.nx * m.ny * m.nz;
  m.V = (int64_t)(m.nx - 1) * (m.ny - 1) * (m.nz - 1);
  if (src != MPF_MC_LEVELSET) {
    const f3* pos = (const f3*)c.pos[c.cur];
    const int8_t* fl = (const int8_t*)c.flag[c.cur];
    const uint32_t *cs = c.mc_cstart, *ce = c.mc_cend;
    const dim3 gd(nblocks(m.N, 256));
    if (src == MPF_MC_LIQUID_GAS)
      launch(c, "mc_density_liquid_gas", gd, dim3(256), 0, k_mc_density<MPF_MC_LIQUID_GAS>, m, c.g2, pos, fl, cs, ce,
             c.mc_field, c.cfg.mc_gas_airsolo);
    else if (src == MPF_MC_GAS)
      launch(c, "mc_density_gas", gd, dim3(256), 0, k_mc_density<MPF_MC_GAS>, m, c.g2, pos, fl, cs, ce, c.mc_field,
             c.cfg.mc_gas_airsolo);
    else
      launch(c, "mc_density_solid", gd, dim3(256), 0, k_mc_density<MPF_MC_SOLID>, m, c.g2, pos, fl, cs, ce,
             c.mc_field, c.cfg.mc_gas_airsolo);
    c.mc_field_valid = true;
  }
  const int64_t V = m.V, N = m.N;
  c.mc_nvox = V;
  hipMemsetAsync(c.mc_edge, 0, (size_t)3 * N * 4, c.stream);
  uint32_t* spread = c.counters + 64;
  hipMemsetAsync(spread, 0, NSPREAD * SPREAD_STRIDE * 4, c.stream);
  launch(c, "mc_classify", dim3(nblocks(V, 256)), dim3(256), 0, k_mc_classify, m, f, c.mc_case, c.mc_tcount,
         c.mc_edge, spread);
  // vertex ids = exclusive scan of the used-edge flags (second half of mc_edge)
  uint32_t* vid = c.mc_edge + 3 * N;
  int64_t nv = run_scan_u32(c, c.mc_edge, vid, 3 * N, true);
  // triangle offsets = exclusive scan of per-voxel triangle counts (second half of mc_tcount)
  int64_t nt = run_scan_u32(c, c.mc_tcount, c.mc_tcount + V, V, true);
  if (nv < 0 || nt < 0) return MPF_HIP_ERROR;
  hipMemcpyAsync(c.counters_host + 64, spread, NSPREAD * SPREAD_STRIDE * 4, hipMemcpyDeviceToHost, c.stream);
  if (!hip_ok(c, hipStreamSynchronize(c.stream), "marching_cubes")) return MPF_HIP_ERROR;
  if (nv > c.cfg.mc_max_verts || nt > c.cfg.mc_max_tris) {
    c.err = "marching cubes mesh exceeds mc_max_verts/mc_max_tris";
    return MPF_CAPACITY;
  }
  launch(c, "mc_verts", dim3(nblocks(3 * N, 256)), dim3(256), 0, k_mc_verts, m, f, (const uint32_t*)c.mc_edge,
         (const uint32_t*)vid, c.mc_verts, c.mc_vedge);
  launch(c, "mc_tris", dim3(nblocks(V, 256)), dim3(256), 0, k_mc_tris, m, (const uint8_t*)c.mc_case,
         (const uint32_t*)(c.mc_tcount + V), (const uint32_t*)vid, c.mc_tris);
  // runMC_smooth step 8 (spray.cu:948-951): smoothing, then vertex normals
  // (the normal buffer is the smoothing's second vertex buffer before that)
  {
    const uint32_t* toff = c.mc_tcount + V;
    float* a = c.mc_verts;
    float* b = c.mc_normals;
    for (int it = 0; it < c.cfg.mc_smooth_iters; ++it) {
      launch(c, "mc_smooth", dim3(nblocks(nv, 256)), dim3(256), 0, k_mc_smooth, m, (const uint32_t*)c.mc_vedge,
             (const uint8_t*)c.mc_case, toff, (const uint32_t*)c.mc_tris, (const float*)a, b, nv, 0.5f);
      std::swap(a, b);
    }
    if (a != c.mc_verts && nv > 0)
      hipMemcpyAsync(c.mc_verts, a, (size_t)nv * 12, hipMemcpyDeviceToDevice, c.stream);
    launch(c, "mc_normals", dim3(nblocks(nv, 256)), dim3(256), 0, k_mc_normals, m, (const uint32_t*)c.mc_vedge,
           (const uint8_t*)c.mc_case, toff, (const uint32_t*)c.mc_tris, (const float*)c.mc_verts, c.mc_normals, nv);
  }
  c.mc_nv = nv;
  c.mc_nt = nt;
  if (info) {
    info->verts = nv;
    info->tris = nt;
    int64_t act = 0;
    for (int q = 0; q < NSPREAD; ++q) act += c.counters_host[64 + q * SPREAD_STRIDE];
    info->active_voxels = act;
  }
  return MPF_OK;
}

}  // namespace mpf
