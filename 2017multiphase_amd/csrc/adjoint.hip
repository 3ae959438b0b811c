// Hand-written adjoints (reverse-mode products) of the projection, P2G, G2P
// and advection stages.  The reference has no counterpart; these serve
// gradient computations through the step.  Each adjoint is evaluated at the
// state of the stage's forward call (flags, level sets, cell lists, particle
// order, positions) and holds every discrete decision of that call fixed.
// Cotangents are FP64.
#include "interp.h"
#include "row_bits.h"
#include "mpf_internal.h"

#include <algorithm>

namespace mpf {

namespace {

__device__ __forceinline__ int8_t mark_at(const Grid& g, const int8_t* mark, int i, int j, int k) {
  return valid(g, i, j, k) ? mark[cid(g, i, j, k)] : BOUNDARY;
}

struct Faces6 {
  double* f[6];  // water ux, uy, uz, air ux, uy, uz
};
struct CFaces6 {
  const double* f[6];
};

// ---------------- projection ----------------
// Forward (cspray::project_CG_bubble, spray.cu:1590-1611):
//   b = D(u_w, u_a) on FLUID|AIR cells (cptdivergence_bubble2, theta blend at
//   liquid/air faces; 0 at faces of constrained SOLID cells), p = A^-1 b,
//   u'_phase[f] = u_phase[f] - beta_phase (p[c1] - p[c0]) / h on interior faces
//   (subGradPress), 0 on faces touching a constrained SOLID cell.
// Adjoint: gp = -G^T g' (cell gather), lambda = A^-1 gp (A symmetric),
//   g_in = (identity part of g') + D^T lambda (face gather).

// gp[c] = sum over the 6 faces of c of (+-beta g'[f] / h), unknown cells only.
__global__ void k_adj_gradT(Grid g, const int8_t* __restrict__ mark, CFaces6 go, double bw, double ba, int solid_c,
                            double* __restrict__ gp) {
  int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= g.G) return;
  int i, j, k;
  ijk_of(g, idx, i, j, k);
  const int8_t m = mark[idx];
  double s = 0.0;
  if (m == FLUID || m == AIR) {
    const int n3[3] = {g.nx, g.ny, g.nz};
    const int c3[3] = {i, j, k};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
      // face below (c is its upper cell c1): u' -= beta (p[c] - p[below]) / h -> gp[c] -= beta g / h
      if (c3[a] > 0) {
        int o[3] = {0, 0, 0};
        o[a] = -1;
        bool solid = solid_c && (m == SOLID || mark_at(g, mark, i + o[0], j + o[1], k + o[2]) == SOLID);
        if (!solid) {
          int64_t f = fid(g, a, i, j, k);
          s -= (bw * go.f[a][f] + ba * go.f[3 + a][f]) / (double)g.h;
        }
      }
      // face above (c is its lower cell c0): gp[c] += beta g / h
      if (c3[a] + 1 < n3[a]) {
        int o[3] = {0, 0, 0};
        o[a] = 1;
        bool solid = solid_c && (m == SOLID || mark_at(g, mark, i + o[0], j + o[1], k + o[2]) == SOLID);
        if (!solid) {
          int64_t f = fid(g, a, i + o[0], j + o[1], k + o[2]);
          s += (bw * go.f[a][f] + ba * go.f[3 + a][f]) / (double)g.h;
        }
      }
    }
  }
  gp[idx] = s;
}

// Coefficients of face velocity (water, air) in the divergence of cell c for
// its face towards neighbour n (cptdivergence_bubble2 cases).
__device__ __forceinline__ void div_coef(const Grid& g, const int8_t* mark, const float* ls, int64_t c, int8_t m,
                                         int64_t n, int8_t mn, int solid_c, double& cw, double& ca) {
  cw = ca = 0.0;
  if (solid_c && mn == SOLID) return;
  if (m == FLUID && mn != AIR) { cw = 1.0; return; }
  if (m == AIR && mn != FLUID) { ca = 1.0; return; }
  double th = (0.0 - (double)ls[c]) / ((double)ls[n] - (double)ls[c]);
  if (m == FLUID) { cw = th; ca = 1.0 - th; }
  else { ca = th; cw = 1.0 - th; }
}

template <int A>
__global__ void k_adj_divT(Grid g, const int8_t* __restrict__ mark, const float* __restrict__ ls,
                           const double* __restrict__ lam, CFaces6 go, Faces6 gi, int solid_c, int64_t nf) {
  int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f >= nf) return;
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  const int n3[3] = {i, j, k};
  const int lim = (A == 0) ? g.nx : (A == 1) ? g.ny : g.nz;
  // cells on either side: c1 = (i,j,k) (upper), c0 = one step down along A
  const bool has1 = n3[A] < lim, has0 = n3[A] > 0;
  const int bi = i - (A == 0), bj = j - (A == 1), bk = k - (A == 2);
  const int8_t m1 = has1 ? mark[cid(g, i, j, k)] : BOUNDARY;
  const int8_t m0 = has0 ? mark[cid(g, bi, bj, bk)] : BOUNDARY;
  const bool interior = has0 && has1;
  const bool solid = solid_c && (m0 == SOLID || m1 == SOLID);
  double w = 0.0, a = 0.0;
  if (!(interior && solid)) {  // identity part (interior faces keep u; domain faces are unchanged)
    w = go.f[A][f];
    a = go.f[3 + A][f];
  }
  const double ih = 1.0 / (double)g.h;
  if (has1 && (m1 == FLUID || m1 == AIR)) {  // f is the lower face of c1: div -= u0 / h
    double cw, ca;
    const int64_t c1 = cid(g, i, j, k);
    div_coef(g, mark, ls, c1, m1, has0 ? cid(g, bi, bj, bk) : c1, m0, solid_c, cw, ca);
    w -= lam[c1] * cw * ih;
    a -= lam[c1] * ca * ih;
  }
  if (has0 && (m0 == FLUID || m0 == AIR)) {  // f is the upper face of c0: div += u1 / h
    double cw, ca;
    const int64_t c0 = cid(g, bi, bj, bk);
    div_coef(g, mark, ls, c0, m0, has1 ? cid(g, i, j, k) : c0, m1, solid_c, cw, ca);
    w += lam[c0] * cw * ih;
    a += lam[c0] * ca * ih;
  }
  gi.f[A][f] = w;
  gi.f[3 + A][f] = a;
}

// ---------------- P2G ----------------
// Forward (mapvelp2g_k_fluidSolid / _air, spray_k.cu:2809-2937):
//   u_f = sum_p w_pf v_p / W_f,  W_f = sum_p w_pf,  w_pf = m_p max(RE^2/max(r^2,1e-4) - 1, 0)
// Adjoint per particle p (gather over the faces whose window holds p's cell):
//   g_v[p] += (w_pf / W_f) g_u[f]
//   g_x[p] += (dw_pf/dx)(v_p - u_f) / W_f g_u[f]

// The air window's rows are dealt to AIR_LANES lanes per face: few faces have
// air near them, and one lane's walk over 25 rows is a chain of loads.
constexpr int AIR_LANES = 8;
// Marks a face without weight, or whose weight is not a number, in place of
// g_u / W: a NaN whose payload arithmetic does not make.  Such a face passes
// nothing on, whatever a particle beside it holds.
constexpr long long NO_WEIGHT = 0x7ff8a5c3f00d1e2dll;
// W_f and u_f recomputed in FP64 (face gather with the forward's windows, one
// launch for the three axes).  Bound by FP64 arithmetic: about 30 operations
// at half rate, a division among them, for each of a face's 144 particles.
// The occupancy masks of the sort, which the forward call goes by too, leave
// out the cells and bricks without a particle of the phase: the air window
// (100 cells) was walked on every face before, 4.1 ms at 96^3 for the six
// launches with 2.9M particles and 6 bubbles; 0.97 (liquid) + 0.36 ms (air: row
// bits, the 36 cells within the radius) now.
struct FaceOut {
  const double* gu[3];
  double* B[3];  // g_u / W (NO_WEIGHT without weight)
  double* U[3];
};
template <int A, bool AIRPH, bool ROWS>
__device__ __forceinline__ void adj_p2g_face(const Grid& g, const f3* __restrict__ pos, const f3* __restrict__ vel,
                                             const float* __restrict__ mass, const int8_t* __restrict__ flag,
                                             const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
                                             const uint8_t* __restrict__ cmask, const RowBits& rb,
                                             const uint8_t* __restrict__ dm, const double* __restrict__ gu,
                                             double* __restrict__ Bout, double* __restrict__ Uout, int64_t f, int sub) {
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  constexpr uint8_t need = AIRPH ? M_AIR : M_FLUIDSOLID;
  {
    // the bricks around the face's cell hold every cell of the window
    const int by = (g.ny + 3) / 4, bz = (g.nz + 3) / 4;
    const int64_t b = ((int64_t)(min(i, g.nx - 1) >> 2) * by + (min(j, g.ny - 1) >> 2)) * bz + (min(k, g.nz - 1) >> 2);
    if (!(dm[b] & need)) {  // the same for all lanes of a face
      if (sub == 0) {
        Bout[f] = __longlong_as_double(NO_WEIGHT);
        Uout[f] = 0.0;
      }
      return;
    }
  }
  const double gx = (double)i + (A == 0 ? 0.0 : 0.5), gy = (double)j + (A == 1 ? 0.0 : 0.5),
               gz = (double)k + (A == 2 ? 0.0 : 0.5);
  constexpr int lo = AIRPH ? -2 : -1, hin = AIRPH ? 1 : 0, lot = AIRPH ? -2 : -1, hit = AIRPH ? 2 : 1;
  const double RE2 = (double)1.4f * (double)1.4f, scale = 1.0 / (double)g.h;
  constexpr int NP = AIRPH ? 8 : 4;  // particles whose loads are in flight together
  double W = 0, U = 0;
  auto visit = [&](uint32_t s, uint32_t e) {
    for (uint32_t p0 = s; p0 < e; p0 += NP) {
      int8_t fl[NP];
      f3 x[NP];
      float mp[NP], va[NP];
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        const uint32_t p = min(p0 + (uint32_t)u, e - 1u);
        fl[u] = flag[p];
        x[u] = pos[p];
        mp[u] = mass[p];
        va[u] = (&vel[p].x)[A];
      }
#pragma unroll
      for (int u = 0; u < NP; ++u) {
        const bool take = p0 + (uint32_t)u < e && (AIRPH ? (fl[u] == AIR) : (fl[u] == FLUID || fl[u] == SOLID));
        if (!take) continue;
        const double dx = ((double)x[u].x - g.gx0) * scale - gx, dy = ((double)x[u].y - g.gy0) * scale - gy,
                     dz = ((double)x[u].z - g.gz0) * scale - gz;
        const double r2 = dx * dx + dy * dy + dz * dz;
        double q = 0.0;  // not positive from the kernel's radius on: no division
        if (!(r2 >= RE2)) q = fmax(RE2 / fmax(r2, (double)0.0001f) - 1.0, 0.0);
        const double w = (double)mp[u] * q;
        W += w;
        U += w * (double)va[u];
      }
    }
  };
  constexpr int i0 = A == 0 ? lo : lot, j0 = A == 1 ? lo : lot;
  constexpr int NJ = (A == 1 ? hin : hit) - j0 + 1, NR = ((A == 0 ? hin : hit) - i0 + 1) * NJ;
  constexpr int k0 = A == 2 ? lo : lot, NK = (A == 2 ? hin : hit) - k0 + 1;
  for (int r = sub; r < NR; r += AIRPH ? AIR_LANES : 1) {
    const int ci = i + i0 + r / NJ, cj = j + j0 + r % NJ;
    if (AIRPH) {  // the row's cells that hold air, from their bits
      using AW = AirWindow<A>;
      const bool near = ROWS && *rb.odd == 0;
      if (near && !AW::row_near(r)) continue;
      uint32_t bits = row_window(rb.a, rb, ci + 2, cj + 2, k) & (near ? AW::bits_near : AW::ROW);
      if (!bits) continue;
      const int64_t c0 = cid(g, ci, cj, k + k0);
      if (ROWS) visit(cstart[c0 + __ffs(bits) - 1], cend[c0 + 31 - __clz(bits)]);
      else
        for (; bits; bits &= bits - 1u) visit(cstart[c0 + __ffs(bits) - 1], cend[c0 + __ffs(bits) - 1]);
    } else {
      if (ci < 0 || ci >= g.nx || cj < 0 || cj >= g.ny) continue;
      // the row's masks and ranges together, then its particles (ROWS: one range)
      uint32_t S[NK], E[NK];
      bool take_cell[NK];
#pragma unroll
      for (int q = 0; q < NK; ++q) {
        const int ck = k + k0 + q;
        const bool in = ck >= 0 && ck < g.nz;
        const int64_t c = cid(g, ci, cj, in ? ck : min(max(ck, 0), g.nz - 1));
        const uint8_t m = cmask[c];
        S[q] = cstart[c];
        E[q] = cend[c];
        take_cell[q] = in && (m & need);
      }
      uint32_t s = MPF_CELL_UNDEF, e = 0;
#pragma unroll
      for (int q = 0; q < NK; ++q) {
        if (!take_cell[q]) continue;
        if (ROWS) {
          s = min(s, S[q]);
          e = max(e, E[q]);
        } else {
          visit(S[q], E[q]);
        }
      }
      if (ROWS && s < e) visit(s, e);
    }
  }
  if (AIRPH) {
#pragma unroll
    for (int o = 1; o < AIR_LANES; o <<= 1) {
      W += __shfl_xor(W, o);
      U += __shfl_xor(U, o);
    }
  }
  if (sub == 0) {
    Bout[f] = (W > 0) ? gu[f] / W : __longlong_as_double(NO_WEIGHT);
    Uout[f] = (W > 0) ? U / W : 0.0;
  }
}
template <bool AIRPH, bool ROWS>
__global__ void __launch_bounds__(256) k_adj_p2g_faces(Grid g, const f3* __restrict__ pos, const f3* __restrict__ vel,
                                const float* __restrict__ mass, const int8_t* __restrict__ flag,
                                const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend,
                                const uint8_t* __restrict__ cmask, RowBits rb, const uint8_t* __restrict__ dm, FaceOut out) {
  const int64_t u = xcd_block() * blockDim.x + threadIdx.x;
  const int64_t f = AIRPH ? u / AIR_LANES : u;
  const int sub = AIRPH ? (int)(u % AIR_LANES) : 0;
  const int A = blockIdx.y;
  if (f >= (A == 0 ? g.FX : A == 1 ? g.FY : g.FZ)) return;
  if (A == 0) adj_p2g_face<0, AIRPH, ROWS>(g, pos, vel, mass, flag, cstart, cend, cmask, rb, dm, out.gu[0], out.B[0], out.U[0], f, sub);
  else if (A == 1) adj_p2g_face<1, AIRPH, ROWS>(g, pos, vel, mass, flag, cstart, cend, cmask, rb, dm, out.gu[1], out.B[1], out.U[1], f, sub);
  else adj_p2g_face<2, AIRPH, ROWS>(g, pos, vel, mass, flag, cstart, cend, cmask, rb, dm, out.gu[2], out.B[2], out.U[2], f, sub);
}

struct P2GFaceData {
  const double* B[3];  // g_u / W
  const double* U[3];
};

// The liquid launch writes every particle (0 off its phase), the air launch
// adds.  Bound by FP64 arithmetic and the gathers: with g_u / W formed once per
// face and one reciprocal of r^2 a pair takes one division where it took four
// (0.60 -> 0.40 ms at 96^3, liquid; 0.23 -> 0.11 air).
template <bool AIRPH>
__global__ void k_adj_p2g_part(Grid g, int64_t P, const f3* __restrict__ pos, const f3* __restrict__ vel,
                               const float* __restrict__ mass, const int8_t* __restrict__ flag, P2GFaceData fd,
                               double* __restrict__ gv, double* __restrict__ gx) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const int8_t fl = flag[p];
  const bool take = AIRPH ? (fl == AIR) : (fl == FLUID || fl == SOLID);
  if (!take) {
    if (!AIRPH)
      for (int d = 0; d < 3; ++d) gv[3 * p + d] = gx[3 * p + d] = 0.0;
    return;
  }
  const f3 x = pos[p];
  const float* vp = &vel[p].x;
  // the particle's cell, as the hash assigns it (getijkfrompos)
  float qx = (x.x - g.gx0) / g.h, qy = (x.y - g.gy0) / g.h, qz = (x.z - g.gz0) / g.h;
  const int ci = (qx >= 0 && qx < (float)g.nx) ? (int)qx : 0;
  const int cj = (qy >= 0 && qy < (float)g.ny) ? (int)qy : 0;
  const int ck = (qz >= 0 && qz < (float)g.nz) ? (int)qz : 0;
  const double RE2 = (double)1.4f * (double)1.4f, scale = 1.0 / (double)g.h;
  const double X = ((double)x.x - g.gx0) * scale, Y = ((double)x.y - g.gy0) * scale, Z = ((double)x.z - g.gz0) * scale;
  const double m = (double)mass[p];
  constexpr int lo = AIRPH ? -2 : -1, hin = AIRPH ? 1 : 0, lot = AIRPH ? -2 : -1, hit = AIRPH ? 2 : 1;
  double av[3] = {0, 0, 0}, ax[3] = {0, 0, 0};
#pragma unroll
  for (int A = 0; A < 3; ++A) {
    const int dims[3] = {g.nx + (A == 0), g.ny + (A == 1), g.nz + (A == 2)};
    // faces f = c - o for window offsets o
    for (int oi = (A == 0 ? lo : lot); oi <= (A == 0 ? hin : hit); ++oi)
      for (int oj = (A == 1 ? lo : lot); oj <= (A == 1 ? hin : hit); ++oj)
        for (int ok = (A == 2 ? lo : lot); ok <= (A == 2 ? hin : hit); ++ok) {
          const int fi = ci - oi, fj = cj - oj, fk = ck - ok;
          if (fi < 0 || fj < 0 || fk < 0 || fi >= dims[0] || fj >= dims[1] || fk >= dims[2]) continue;
          const int64_t f = fid(g, A, fi, fj, fk);
          const double B = fd.B[A][f], U = fd.U[A][f];
          const double gxf = (double)fi + (A == 0 ? 0.0 : 0.5), gyf = (double)fj + (A == 1 ? 0.0 : 0.5),
                       gzf = (double)fk + (A == 2 ? 0.0 : 0.5);
          const double dx = X - gxf, dy = Y - gyf, dz = Z - gzf;
          const double r2 = dx * dx + dy * dy + dz * dz;
          if (r2 >= RE2) continue;
          const double ir2 = 1.0 / fmax(r2, (double)0.0001f);
          const double s = RE2 * ir2 - 1.0;
          if (!(s > 0) || __double_as_longlong(B) == NO_WEIGHT) continue;
          av[A] += (m * s) * B;
          if (r2 > (double)0.0001f) {
            // dw/dx_d = -2 m RE^2 d_d / r^4 * scale
            const double dwr = -2.0 * m * RE2 * (ir2 * ir2) * scale;
            const double coef = ((double)vp[A] - U) * B * dwr;
            ax[0] += coef * dx;
            ax[1] += coef * dy;
            ax[2] += coef * dz;
          }
        }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    gv[3 * p + d] = AIRPH ? gv[3 * p + d] + av[d] : av[d];
    gx[3 * p + d] = AIRPH ? gx[3 * p + d] + ax[d] : ax[d];
  }
}

// ---------------- G2P ----------------
// Forward (mapvelg2p_flip_bubble spray_k.cu:3525-3540 with blend alpha):
//   v' = (1 - alpha) T(x) u + alpha (v + T(x) du),  du = u - u_old (grid of the particle's phase)
// Adjoint: g_v = alpha g_v';  g_u += T^T g_v' (both terms);  g_uold -= alpha T^T g_v';
//   g_x += (1 - alpha) (dT u/dx)^T g_v' + alpha (dT du/dx)^T g_v'.
// g_uold is -alpha times the scattered g_u, so only g_u is scattered (FP64
// atomics, whose order sets the rounding).  Particles in the order of the
// library's sort are scattered tile by tile (4x8x8 cells): a row of 8 cells is
// one range of particles, a wave's lanes add them into the tile's faces in
// LDS, and the tile adds its sums to the grid once.  48 grid atomics per
// particle took 3.6 ms at 96^3 (2.9M particles), bound by the atomics; by tiles
// 0.47 ms.
struct G2PArgs {
  const float* u[6];   // water u, air u (current)
  const float* du[6];  // water du, air du (forward's u - u_old)
  double* gu[6];
};

// One particle's cotangents (gvi, gx written); scat(slot, axis, i, j, k, value)
// takes the eight corner terms of each axis.
template <class S>
__device__ __forceinline__ void adj_g2p_particle(const Grid& g, int64_t p, const f3* __restrict__ pos,
                                                 const int8_t* __restrict__ flag, const G2PArgs& a, double alpha,
                                                 const double* __restrict__ gvo, double* __restrict__ gvi,
                                                 double* __restrict__ gx, S scat) {
  const int8_t fl = flag[p];
  int ph = -1;
  if (fl == FLUID || fl == SOLID) ph = 0;
  else if (fl == AIR) ph = 1;
  const double gv[3] = {gvo[3 * p], gvo[3 * p + 1], gvo[3 * p + 2]};
  if (ph < 0) {
    for (int d = 0; d < 3; ++d) {
      gvi[3 * p + d] = gv[d];
      gx[3 * p + d] = 0.0;
    }
    return;
  }
  for (int d = 0; d < 3; ++d) gvi[3 * p + d] = alpha * gv[d];
  const f3 x = pos[p];
  const double X = ((double)x.x - g.gx0) / g.h, Y = ((double)x.y - g.gy0) / g.h, Z = ((double)x.z - g.gz0) / g.h;
  double gpos[3] = {0, 0, 0};
#pragma unroll
  for (int A = 0; A < 3; ++A) {
    const int w = g.nx + (A == 0), hh = g.ny + (A == 1), d = g.nz + (A == 2);
    const double qx = X - (A == 0 ? 0.0 : 0.5), qy = Y - (A == 1 ? 0.0 : 0.5), qz = Z - (A == 2 ? 0.0 : 0.5);
    int i, j, k;
    double wt[8];
    trilinear_weights(qx, qy, qz, w, hh, d, i, j, k, wt);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if (wt[c] == 0.0) continue;
      scat(3 * ph + A, A, i + (c & 1), j + ((c >> 1) & 1), k + (c >> 2), wt[c] * gv[A]);
    }
    double g1x, g1y, g1z, g2x, g2y, g2z;
    trilinear_grad(a.u[3 * ph + A], qx, qy, qz, w, hh, d, g1x, g1y, g1z);
    trilinear_grad(a.du[3 * ph + A], qx, qy, qz, w, hh, d, g2x, g2y, g2z);
    const double s1 = (1.0 - alpha) * gv[A], s2 = alpha * gv[A];
    gpos[0] += (s1 * g1x + s2 * g2x) / (double)g.h;
    gpos[1] += (s1 * g1y + s2 * g2y) / (double)g.h;
    gpos[2] += (s1 * g1z + s2 * g2z) / (double)g.h;
  }
  for (int d = 0; d < 3; ++d) gx[3 * p + d] = gpos[d];
}

__global__ void __launch_bounds__(256) k_adj_g2p(Grid g, int64_t P, const f3* __restrict__ pos, const int8_t* __restrict__ flag,
                          G2PArgs a, double alpha, const double* __restrict__ gvo, double* __restrict__ gvi,
                          double* __restrict__ gx) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  adj_g2p_particle(g, p, pos, flag, a, alpha, gvo, gvi, gx, [&](int slot, int A, int i, int j, int k, double v) {
    unsafeAtomicAdd(&a.gu[slot][fid(g, A, i, j, k)], v);
  });
}

// The tile's faces of axis a: [t0_d - (d != a), t0_d + T_d] along d, as in the liquid P2G.
constexpr int GT_X = 4, GT_Y = 8, GT_Z = 8, GT = GT_X * GT_Y * GT_Z;
__host__ __device__ constexpr int gt_t(int d) { return d == 0 ? GT_X : (d == 1 ? GT_Y : GT_Z); }
__host__ __device__ constexpr int gt_r(int a, int d) { return gt_t(d) + (d == a ? 1 : 2); }
__host__ __device__ constexpr int gt_sz(int a) { return gt_r(a, 0) * gt_r(a, 1) * gt_r(a, 2); }
__host__ __device__ constexpr int gt_off(int a) { return a == 0 ? 0 : (a == 1 ? gt_sz(0) : gt_sz(0) + gt_sz(1)); }
constexpr int GT_TOT = gt_sz(0) + gt_sz(1) + gt_sz(2);

__global__ void __launch_bounds__(GT)
    k_adj_g2p_tile(Grid g, const f3* __restrict__ pos, const int8_t* __restrict__ flag,
                   const uint32_t* __restrict__ cstart, const uint32_t* __restrict__ cend, int nty, int ntz, G2PArgs a,
                   double alpha, const double* __restrict__ gvo, double* __restrict__ gvi, double* __restrict__ gx) {
  __shared__ double acc[2 * GT_TOT];  // liquid, then air
  __shared__ uint32_t sS[GT], sE[GT];
  int t = (int)xcd_block();
  const int tz = t % ntz;
  t /= ntz;
  const int ty = t % nty, tx = t / nty;
  const int x0 = tx * GT_X, y0 = ty * GT_Y, z0 = tz * GT_Z;
  const int b = threadIdx.x, lane = b & 63;
  for (int q = b; q < 2 * GT_TOT; q += GT) acc[q] = 0.0;
  {
    const int ci = x0 + b / (GT_Y * GT_Z), cj = y0 + (b / GT_Z) % GT_Y, ck = z0 + b % GT_Z;
    uint32_t s = MPF_CELL_UNDEF, e = 0;
    if (valid(g, ci, cj, ck)) {
      const int64_t c = cid(g, ci, cj, ck);
      s = cstart[c];
      e = s == MPF_CELL_UNDEF ? 0 : cend[c];
    }
    sS[b] = s;
    sE[b] = e;
  }
  __syncthreads();
  for (int row = b >> 6; row < GT_X * GT_Y; row += GT / 64) {
    uint32_t s = MPF_CELL_UNDEF, e = 0;
#pragma unroll
    for (int q = 0; q < GT_Z; ++q) {
      s = min(s, sS[row * GT_Z + q]);
      e = max(e, sE[row * GT_Z + q]);
    }
    for (uint32_t p = s + lane; s < e && p < e; p += 64)
      adj_g2p_particle(g, p, pos, flag, a, alpha, gvo, gvi, gx, [&](int slot, int A, int i, int j, int k, double v) {
        const int ri = i - (x0 - (A != 0)), rj = j - (y0 - (A != 1)), rk = k - (z0 - (A != 2));
        // (a particle outside the domain lies in cell 0 whatever its position)
        if ((unsigned)ri < (unsigned)gt_r(A, 0) && (unsigned)rj < (unsigned)gt_r(A, 1) &&
            (unsigned)rk < (unsigned)gt_r(A, 2))
          unsafeAtomicAdd(&acc[(slot >= 3 ? GT_TOT : 0) + gt_off(A) + (ri * gt_r(A, 1) + rj) * gt_r(A, 2) + rk], v);
        else
          unsafeAtomicAdd(&a.gu[slot][fid(g, A, i, j, k)], v);
      });
  }
  __syncthreads();
  for (int q = b; q < 2 * GT_TOT; q += GT) {
    const double v = acc[q];
    if (v == 0.0) continue;
    const int ph = q >= GT_TOT, r = q - ph * GT_TOT;
    const int A = r < gt_off(1) ? 0 : (r < gt_off(2) ? 1 : 2);
    const int l = r - gt_off(A);
    const int rk = l % gt_r(A, 2), rj = (l / gt_r(A, 2)) % gt_r(A, 1), ri = l / (gt_r(A, 2) * gt_r(A, 1));
    unsafeAtomicAdd(&a.gu[3 * ph + A][fid(g, A, x0 - (A != 0) + ri, y0 - (A != 1) + rj, z0 - (A != 2) + rk)], v);
  }
}

// ---------------- advection ----------------
// Forward (CollisionWithSolid_k, spray_k.cu:5276-5345, away from solids):
//   x' = clamp(x + v dt), v' = v with clamped components zeroed; SOLID fixed.
// Adjoint, per component not clamped: g_x = g_x', g_v = g_v' + dt g_x';
// clamped component: both 0.  The solid-collision response (phi_solid <= 0.5)
// is not differentiated; particles in that band are reported through
// `in_band` (count) so a caller can tell.
__global__ void k_adj_advect(Grid g, int64_t P, const f3* __restrict__ pos, const f3* __restrict__ vel,
                             const int8_t* __restrict__ flag, const float* __restrict__ phis, double dt,
                             const double* __restrict__ gxo, const double* gvo, double* __restrict__ gxi,
                             double* gvi, uint32_t* __restrict__ in_band) {
  int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P) return;
  const int8_t fl = flag[p];
  if (fl == SOLID) {
    for (int d = 0; d < 3; ++d) {
      gxi[3 * p + d] = gxo[3 * p + d];
      gvi[3 * p + d] = gvo[3 * p + d];
    }
    return;
  }
  const f3 x = pos[p], v = vel[p];
  if (phis && scalar_from_grid(g, x, phis) <= 0.5f) atomicAdd(in_band, 1u);
  const float rate = (fl == AIRSOLO) ? 0.8f : 0.5f;
  const float m = g.h + rate * g.h;
  const float lo[3] = {g.gx0 + m, g.gy0 + m, g.gz0 + m}, hi[3] = {g.gx1 - m, g.gy1 - m, g.gz1 - m};
  const float xs[3] = {x.x + v.x * (float)dt, x.y + v.y * (float)dt, x.z + v.z * (float)dt};
  for (int d = 0; d < 3; ++d) {
    const bool cl = xs[d] <= lo[d] || xs[d] >= hi[d];
    gxi[3 * p + d] = cl ? 0.0 : gxo[3 * p + d];
    gvi[3 * p + d] = cl ? 0.0 : gvo[3 * p + d] + dt * gxo[3 * p + d];
  }
}

// ---------------- extrapolation and wall rule ----------------
// Forward (sweepU + setWaterBoundaryU_k, spray_k.cu:900-995): two passes of
// out[f] = u[f], or, for a face with both cells outside phase sf, the blend
// wx u[f+dx e_x] + wy u[f+dy e_y] + wz u[f+dz e_z] of the last qualifying
// diagonal direction; then the wall rule zeroes faces and sets the ceiling
// uz(nz-1) to min(uz(nz-2), 0).  Linear in u for fixed level set and flags.

// The forward's decision for face (i,j,k) of axis A: false = identity.  The
// reference visits the 8 octants and the last one whose three weights are all
// >= 0 decides; each weight depends on its own axis' sign only, so per axis +1
// decides if its weight passes, else -1 (as in the forward's sweep).
template <int A>
__device__ __forceinline__ bool sweep_rule(const Grid& g, const float* __restrict__ ls,
                                           const int8_t* __restrict__ mark, int8_t sf, int i, int j, int k,
                                           int (&dsel)[3], float (&wsel)[3]) {
  const int n[3] = {i, j, k};
  const int lim = (A == 0) ? g.nx : (A == 1) ? g.ny : g.nz;
  if (!(n[A] > 1 && n[A] < lim - 1)) return false;
  const int bi = i - (A == 0), bj = j - (A == 1), bk = k - (A == 2);
  if (mark[cid(g, i, j, k)] == sf || mark[cid(g, bi, bj, bk)] == sf) return false;
  const float lsc = ls[cid(g, i, j, k)], lsb = ls[cid(g, bi, bj, bk)];
  constexpr int t1 = (A == 0) ? 1 : (A == 1) ? 0 : 1;
  constexpr int t2 = (A == 0) ? 2 : (A == 1) ? 2 : 0;
  const int lims[3] = {g.nx, g.ny, g.nz};
  float wv[3][2];
  bool ok[3][2];
#pragma unroll
  for (int sg = 0; sg < 2; ++sg) {
    const int dd = sg ? 1 : -1;
    wv[A][sg] = (float)(-dd) * (lsc - lsb);
    ok[A][sg] = !(wv[A][sg] < 0);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int ax = t == 0 ? t1 : t2;
      const bool in = n[ax] + dd >= 0 && n[ax] + dd <= lims[ax] - 1;
      int o[3] = {0, 0, 0};
      o[ax] = in ? dd : 0;
      const float lc = ls[cid(g, i + o[0], j + o[1], k + o[2])], lb = ls[cid(g, bi + o[0], bj + o[1], bk + o[2])];
      wv[ax][sg] = (lsc + lsb - lc - lb) * 0.5f;
      ok[ax][sg] = in && !(wv[ax][sg] < 0);
    }
  }
  if (!((ok[0][0] || ok[0][1]) && (ok[1][0] || ok[1][1]) && (ok[2][0] || ok[2][1]))) return false;
  float wx[3];
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    dsel[d] = ok[d][1] ? 1 : -1;
    wx[d] = ok[d][1] ? wv[d][1] : wv[d][0];
  }
  const float wsum = wx[0] + wx[1] + wx[2];
#pragma unroll
  for (int d = 0; d < 3; ++d) wsel[d] = wsum == 0 ? 1.0f / 3 : wx[d] / wsum;
  return true;
}

// The decisions of every face of axis A, for both transposed passes: code bit
// 3: blended, bits 0-2: the direction along x, y, z is +1; the three weights.
// (A pass that evaluates the rules of a face and its six readers itself took
// 87 us a launch at 96^3, 12 launches; now 12 us, and 11 us for an axis' rules.)
struct SweepRules {
  float* w[3];
  uint8_t* code;
};
struct SweepRules3 {
  SweepRules a[3];  // by axis
};
template <int A>
__device__ __forceinline__ void adj_sweep_rules_face(const Grid& g, const float* __restrict__ ls,
                                                     const int8_t* __restrict__ mark, int8_t sf, const SweepRules& r,
                                                     int64_t f) {
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  int dsel[3];
  float wsel[3];
  if (!sweep_rule<A>(g, ls, mark, sf, i, j, k, dsel, wsel)) {
    r.code[f] = 0;
    return;
  }
  uint8_t c = 8;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    c |= dsel[d] > 0 ? (uint8_t)(1u << d) : (uint8_t)0;
    r.w[d][f] = wsel[d];
  }
  r.code[f] = c;
}

// One transposed pass, as a gather: face n collects its identity term and the
// weights of the (at most 6) faces whose chosen blend reads it.
template <int A>
__device__ __forceinline__ void adj_sweep_u_face(const Grid& g, const double* __restrict__ gout,
                                                 double* __restrict__ gin, const SweepRules& r, int64_t f) {
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  const int dims[3] = {g.nx + (A == 0), g.ny + (A == 1), g.nz + (A == 2)};
  const int n[3] = {i, j, k};
  const int64_t st[3] = {(int64_t)dims[1] * dims[2], dims[2], 1};
  uint8_t c[3][2];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      // candidate reader: its blend along d with direction s lands on f
      const bool in = s ? n[d] > 0 : n[d] + 1 < dims[d];
      c[d][s] = in ? r.code[s ? f - st[d] : f + st[d]] : (uint8_t)0;
    }
  double acc = r.code[f] ? 0.0 : gout[f];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (!c[d][s] || ((c[d][s] >> d) & 1) != s) continue;
      const int64_t q = s ? f - st[d] : f + st[d];
      acc += (double)r.w[d][q] * gout[q];
    }
  gin[f] = acc;
}

__device__ __forceinline__ bool isb(const Grid& g, const int8_t* mark, int i, int j, int k) {
  return mark[cid(g, i, j, k)] == BOUNDARY;
}
// 0 = kept, 1 = zeroed, 2 = ceiling face (k = nz-1 of uz); same order of tests as the forward.
template <int A>
__device__ __forceinline__ int bc_rule(const Grid& g, const int8_t* mark, int i, int j, int k) {
  if (A == 0) {
    if (i <= 1 || i >= (g.nx + 1) - 2) return 1;
    if (i > 1 && i < g.nx - 1 && (isb(g, mark, i, j, k) != isb(g, mark, i - 1, j, k))) return 1;
    return 0;
  } else if (A == 1) {
    if (j <= 1 || j >= (g.ny + 1) - 2) return 1;
    if (j > 0 && j < g.ny && (isb(g, mark, i, j, k) != isb(g, mark, i, j - 1, k))) return 1;
    return 0;
  } else {
    const int zn = g.nz + 1;
    if (k <= 1 || k >= zn - 1) return 1;
    if (k == zn - 2) return 2;
    if (k > 0 && k < g.nz && (isb(g, mark, i, j, k) != isb(g, mark, i, j, k - 1))) return 1;
    return 0;
  }
}

// Transposed wall rule.  The ceiling's branch (uz(nz-2) < 0) is read from the
// forward's output `u_after`: the output is negative exactly when it copied.
template <int A>
__device__ __forceinline__ void adj_bc_face(const Grid& g, const double* __restrict__ gout, double* __restrict__ gin,
                                            const int8_t* __restrict__ mark, const float* __restrict__ u_after,
                                            int64_t f) {
  int i, j, k;
  ijk_face<A>(g, f, i, j, k);
  const int r = bc_rule<A>(g, mark, i, j, k);
  double acc = (r == 0) ? gout[f] : 0.0;
  if (A == 2 && r == 0 && k + 1 <= g.nz && bc_rule<2>(g, mark, i, j, k + 1) == 2 && u_after[f + 1] < 0.0f)
    acc += gout[f + 1];
  gin[f] = acc;
}

// Three axes (rules, passes: blockIdx.y = axis) or six fields (3 phase + axis)
// in one launch.
struct Grads6 {
  const double* in[6];
  double* out[6];
  const float* u[6];
};
__device__ __forceinline__ int64_t face_n(const Grid& g, int A) { return A == 0 ? g.FX : A == 1 ? g.FY : g.FZ; }
__global__ void k_adj_sweep_rules(Grid g, const float* __restrict__ ls, const int8_t* __restrict__ mark, int8_t sf,
                                  SweepRules3 r) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int A = blockIdx.y;
  if (f >= face_n(g, A)) return;
  if (A == 0) adj_sweep_rules_face<0>(g, ls, mark, sf, r.a[0], f);
  else if (A == 1) adj_sweep_rules_face<1>(g, ls, mark, sf, r.a[1], f);
  else adj_sweep_rules_face<2>(g, ls, mark, sf, r.a[2], f);
}
__global__ void k_adj_sweep_u(Grid g, Grads6 gr, int ph, SweepRules3 r) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int A = blockIdx.y;
  if (f >= face_n(g, A)) return;
  const double* src = gr.in[3 * ph + A];
  double* dst = gr.out[3 * ph + A];
  if (A == 0) adj_sweep_u_face<0>(g, src, dst, r.a[0], f);
  else if (A == 1) adj_sweep_u_face<1>(g, src, dst, r.a[1], f);
  else adj_sweep_u_face<2>(g, src, dst, r.a[2], f);
}
__global__ void k_adj_bc(Grid g, Grads6 gr, const int8_t* __restrict__ mark) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int q = blockIdx.y, A = q % 3;
  if (f >= face_n(g, A)) return;
  if (A == 0) adj_bc_face<0>(g, gr.in[q], gr.out[q], mark, gr.u[q], f);
  else if (A == 1) adj_bc_face<1>(g, gr.in[q], gr.out[q], mark, gr.u[q], f);
  else adj_bc_face<2>(g, gr.in[q], gr.out[q], mark, gr.u[q], f);
}
__global__ void k_zero6(Grid g, Grads6 gr) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (f < face_n(g, blockIdx.y % 3)) gr.out[blockIdx.y][f] = 0.0;
}
// g_uold = -alpha g_u (nothing with alpha = 0, also of an infinite g_u)
__global__ void k_adj_uold(Grid g, Grads6 gr, double alpha) {
  const int64_t f = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int q = blockIdx.y;
  if (f < face_n(g, q % 3)) gr.out[q][f] = alpha != 0.0 ? 0.0 - alpha * gr.in[q][f] : 0.0;
}

__global__ void k_fill_d(int64_t n, double* __restrict__ a, double v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) a[i] = v;
}

}  // namespace

static int64_t face_count(const Ctx& c, int q) {
  const int64_t fc[3] = {c.g.FX, c.g.FY, c.g.FZ};
  return fc[q % 3];
}

// Adjoint scratch, allocated by mpf_create when cfg.adjoint_enabled is set
// (a failure part-way leaves the pointers set so that adj_free releases them).
bool adj_alloc_all(Ctx& c) {
  auto get = [&](double*& p, size_t bytes) {
    void* q = nullptr;
    if (hipMalloc(&q, bytes) != hipSuccess) return false;
    p = (double*)q;
    return true;
  };
  for (int q = 0; q < 6; ++q)
    if (!get(c.adj_fin[q], (size_t)face_count(c, q) * 8) || !get(c.adj_fout[q], (size_t)face_count(c, q) * 8))
      return false;
  for (int q = 0; q < 2; ++q)
    if (!get(c.adj_cell[q], (size_t)c.g.G * 8)) return false;
  for (int q = 0; q < 3; ++q)
    if (!get(c.adj_part[q], (size_t)(c.cap > 0 ? c.cap : 1) * 24)) return false;
  c.adj_ready = true;
  return true;
}

static bool adj_alloc(Ctx& c) {
  if (c.adj_ready) return true;
  c.err = "adjoint entry points need mpf_config.adjoint_enabled = 1 at mpf_create";
  return false;
}

void adj_free(Ctx& c) {
  for (int q = 0; q < 6; ++q) {
    if (c.adj_fin[q]) hipFree(c.adj_fin[q]);
    if (c.adj_fout[q]) hipFree(c.adj_fout[q]);
    c.adj_fin[q] = c.adj_fout[q] = nullptr;
  }
  for (int q = 0; q < 2; ++q) {
    if (c.adj_cell[q]) hipFree(c.adj_cell[q]);
    c.adj_cell[q] = nullptr;
  }
  for (int q = 0; q < 3; ++q) {
    if (c.adj_part[q]) hipFree(c.adj_part[q]);
    c.adj_part[q] = nullptr;
  }
  c.adj_ready = false;
}

static void copy_in(Ctx& c, double* dst, const double* src, int64_t n, int where) {
  if (src) hipMemcpyAsync(dst, src, (size_t)n * 8, where == MPF_HOST ? hipMemcpyHostToDevice : hipMemcpyDeviceToDevice,
                          c.stream);
  else launch(c, "adj_fill", dim3(nblocks(n, 256)), dim3(256), 0, k_fill_d, n, dst, 0.0);
}
static void copy_out(Ctx& c, double* dst, const double* src, int64_t n, int where) {
  if (dst) hipMemcpyAsync(dst, src, (size_t)n * 8, where == MPF_HOST ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice,
                          c.stream);
}
static void zero(Ctx& c, double* a, int64_t n) {
  launch(c, "adj_fill", dim3(nblocks(n, 256)), dim3(256), 0, k_fill_d, n, a, 0.0);
}

int run_project_adjoint(Ctx& c, const double* const* gout, double* const* gin, int where, mpf_solve_info* info) {
  if (!adj_alloc(c)) return MPF_INVALID_ARG;
  for (int q = 0; q < 6; ++q) copy_in(c, c.adj_fin[q], gout ? gout[q] : nullptr, face_count(c, q), where);
  const bool vd = c.cfg.op == MPF_OPERATOR_VARDENS;
  const double bw = vd ? 1.0 / (double)c.cfg.rho_liquid : 1.0, ba = vd ? 1.0 / (double)c.cfg.rho_air : 1.0;
  CFaces6 go;
  Faces6 gi;
  for (int q = 0; q < 6; ++q) {
    go.f[q] = c.adj_fin[q];
    gi.f[q] = c.adj_fout[q];
  }
  const int64_t G = c.g.G;
  launch(c, "adj_gradT", dim3(nblocks(G, 256)), dim3(256), 0, k_adj_gradT, c.g, (const int8_t*)c.mark, go, bw, ba,
         c.cfg.solid_constraint, c.adj_cell[0]);
  int st = run_adjoint_solve(c, c.adj_cell[0], c.adj_cell[1], info);
  if (st == MPF_HIP_ERROR || st == MPF_NONFINITE) return st;
  launch(c, "adj_divT", dim3(nblocks(c.g.FX, 256)), dim3(256), 0, k_adj_divT<0>, c.g, (const int8_t*)c.mark,
         (const float*)c.lsmerge, (const double*)c.adj_cell[1], go, gi, c.cfg.solid_constraint, c.g.FX);
  launch(c, "adj_divT", dim3(nblocks(c.g.FY, 256)), dim3(256), 0, k_adj_divT<1>, c.g, (const int8_t*)c.mark,
         (const float*)c.lsmerge, (const double*)c.adj_cell[1], go, gi, c.cfg.solid_constraint, c.g.FY);
  launch(c, "adj_divT", dim3(nblocks(c.g.FZ, 256)), dim3(256), 0, k_adj_divT<2>, c.g, (const int8_t*)c.mark,
         (const float*)c.lsmerge, (const double*)c.adj_cell[1], go, gi, c.cfg.solid_constraint, c.g.FZ);
  for (int q = 0; q < 6; ++q) copy_out(c, gin[q], c.adj_fout[q], face_count(c, q), where);
  if (!hip_ok(c, hipStreamSynchronize(c.stream), "project_adjoint")) return MPF_HIP_ERROR;
  return st;
}

int run_extrapolate_adjoint(Ctx& c, const double* const* gout, double* const* gin, int where) {
  if (!adj_alloc(c)) return MPF_INVALID_ARG;
  for (int q = 0; q < 6; ++q) copy_in(c, c.adj_fin[q], gout ? gout[q] : nullptr, face_count(c, q), where);
  const int64_t fc[3] = {c.g.FX, c.g.FY, c.g.FZ};
  const unsigned nb = nblocks(std::max(fc[0], std::max(fc[1], fc[2])), 256);
  // the decisions of one phase at a time, in the P2G's tile buffer (over 12
  // floats per cell; they take 13 bytes per face)
  SweepRules3 rules;
  float* at = c.p2g_parts;
  for (int A = 0; A < 3; ++A) {
    for (int d = 0; d < 3; ++d, at += fc[A]) rules.a[A].w[d] = at;
    rules.a[A].code = (uint8_t*)at;
    at += (fc[A] + 3) / 4;
  }
  if (at - c.p2g_parts > p2g_parts_floats(c.g)) {
    c.err = "extrapolation adjoint: scratch too small";
    return MPF_INVALID_ARG;
  }
  // wall rule^T: fin -> fout; then two sweep passes^T: fout -> fin -> fout
  Grads6 to, back;
  for (int q = 0; q < 6; ++q) {
    to.in[q] = back.out[q] = c.adj_fin[q];
    to.out[q] = c.adj_fout[q];
    back.in[q] = c.adj_fout[q];
    to.u[q] = back.u[q] = q < 3 ? c.wu[q] : c.au[q - 3];
  }
  launch(c, "adj_bc", dim3(nb, 6), dim3(256), 0, k_adj_bc, c.g, to, (const int8_t*)c.mark);
  for (int ph = 0; ph < 2; ++ph) {
    launch(c, "adj_sweep_rules", dim3(nb, 3), dim3(256), 0, k_adj_sweep_rules, c.g,
           (const float*)(ph == 0 ? c.phifluid : c.phiair), (const int8_t*)c.mark, (int8_t)(ph == 0 ? FLUID : AIR), rules);
    launch(c, "adj_sweep_u", dim3(nb, 3), dim3(256), 0, k_adj_sweep_u, c.g, back, ph, rules);
    launch(c, "adj_sweep_u", dim3(nb, 3), dim3(256), 0, k_adj_sweep_u, c.g, to, ph, rules);
  }
  for (int q = 0; q < 6; ++q) copy_out(c, gin[q], c.adj_fout[q], face_count(c, q), where);
  return hip_ok(c, hipStreamSynchronize(c.stream), "extrapolate_adjoint") ? MPF_OK : MPF_HIP_ERROR;
}

int run_p2g_adjoint(Ctx& c, const double* const* gfaces, double* gvel, double* gpos, int where) {
  if (!adj_alloc(c)) return MPF_INVALID_ARG;
  const int cur = c.cur;
  const int64_t P = c.P;
  for (int q = 0; q < 6; ++q) copy_in(c, c.adj_fin[q], gfaces ? gfaces[q] : nullptr, face_count(c, q), where);
  const int64_t fc[3] = {c.g.FX, c.g.FY, c.g.FZ};
  const int64_t fm = std::max(fc[0], std::max(fc[1], fc[2]));
  const RowBits rb = run_row_bits(c);
  if (c.own_sort) run_air_regular(c, rb);
  for (int ph = 0; ph < 2; ++ph) {
    // g_u / W in adj_fout[0..2], U in adj_fout[3..5]
    FaceOut fo;
    for (int A = 0; A < 3; ++A) {
      fo.gu[A] = c.adj_fin[3 * ph + A];
      fo.B[A] = c.adj_fout[A];
      fo.U[A] = c.adj_fout[3 + A];
    }
    // with the library's own sort a row's cells are one range of particles
    auto kern = ph == 0 ? (c.own_sort ? k_adj_p2g_faces<false, true> : k_adj_p2g_faces<false, false>)
                        : (c.own_sort ? k_adj_p2g_faces<true, true> : k_adj_p2g_faces<true, false>);
    launch(c, ph == 0 ? "adj_p2g_faces" : "adj_p2g_faces_air",
           dim3(nblocks(ph == 0 ? fm : fm * AIR_LANES, 256), 3), dim3(256), 0, kern, c.g,
           (const f3*)c.pos[cur], (const f3*)c.vel[cur], (const float*)c.mass[cur], (const int8_t*)c.flag[cur],
           (const uint32_t*)c.cstart, (const uint32_t*)c.cend, (const uint8_t*)c.cmask, rb,
           (const uint8_t*)(c.bmask + nbricks(c.g)), fo);
    P2GFaceData fd;
    for (int A = 0; A < 3; ++A) {
      fd.B[A] = c.adj_fout[A];
      fd.U[A] = c.adj_fout[3 + A];
    }
    if (ph == 0)
      launch(c, "adj_p2g_part", dim3(nblocks(P, 256)), dim3(256), 0, k_adj_p2g_part<false>, c.g, P,
             (const f3*)c.pos[cur], (const f3*)c.vel[cur], (const float*)c.mass[cur], (const int8_t*)c.flag[cur], fd,
             c.adj_part[0], c.adj_part[2]);
    else
      launch(c, "adj_p2g_part_air", dim3(nblocks(P, 256)), dim3(256), 0, k_adj_p2g_part<true>, c.g, P,
             (const f3*)c.pos[cur], (const f3*)c.vel[cur], (const float*)c.mass[cur], (const int8_t*)c.flag[cur], fd,
             c.adj_part[0], c.adj_part[2]);
  }
  copy_out(c, gvel, c.adj_part[0], 3 * P, where);
  copy_out(c, gpos, c.adj_part[2], 3 * P, where);
  return hip_ok(c, hipStreamSynchronize(c.stream), "p2g_adjoint") ? MPF_OK : MPF_HIP_ERROR;
}

int run_g2p_adjoint(Ctx& c, const double* gvel_out, double* gvel_in, double* const* gu, double* const* guo,
                    double* gpos, int where) {
  if (!adj_alloc(c)) return MPF_INVALID_ARG;
  const int cur = c.cur;
  const int64_t P = c.P;
  copy_in(c, c.adj_part[0], gvel_out, 3 * P, where);
  Grads6 gr;
  for (int q = 0; q < 6; ++q) {
    gr.in[q] = gr.out[q] = c.adj_fin[q];
    gr.u[q] = nullptr;
  }
  const unsigned nb6 = nblocks(std::max(c.g.FX, std::max(c.g.FY, c.g.FZ)), 256);
  launch(c, "adj_fill", dim3(nb6, 6), dim3(256), 0, k_zero6, c.g, gr);
  G2PArgs a;
  for (int A = 0; A < 3; ++A) {
    a.u[A] = c.wu[A];
    a.u[3 + A] = c.au[A];
    a.du[A] = c.wuo[A];
    a.du[3 + A] = c.auo[A];
  }
  for (int q = 0; q < 6; ++q) a.gu[q] = c.adj_fin[q];
  const double alpha = (double)c.cfg.flip_alpha;
  // tile by tile when the particles lie in the order of this library's sort
  // (lists given by the caller need not be the particles' order)
  if (c.own_sort) {
    const int ntx = (c.g.nx + GT_X - 1) / GT_X, nty = (c.g.ny + GT_Y - 1) / GT_Y, ntz = (c.g.nz + GT_Z - 1) / GT_Z;
    launch(c, "adj_g2p_tile", dim3((unsigned)(ntx * nty * ntz)), dim3(GT), 0, k_adj_g2p_tile, c.g,
           (const f3*)c.pos[cur], (const int8_t*)c.flag[cur], (const uint32_t*)c.cstart, (const uint32_t*)c.cend, nty,
           ntz, a, alpha, (const double*)c.adj_part[0], c.adj_part[1], c.adj_part[2]);
  } else {
    launch(c, "adj_g2p", dim3(nblocks(P, 256)), dim3(256), 0, k_adj_g2p, c.g, P, (const f3*)c.pos[cur],
           (const int8_t*)c.flag[cur], a, alpha, (const double*)c.adj_part[0], c.adj_part[1], c.adj_part[2]);
  }
  if (guo) {
    for (int q = 0; q < 6; ++q) gr.out[q] = c.adj_fout[q];
    launch(c, "adj_uold", dim3(nb6, 6), dim3(256), 0, k_adj_uold, c.g, gr, alpha);
  }
  copy_out(c, gvel_in, c.adj_part[1], 3 * P, where);
  copy_out(c, gpos, c.adj_part[2], 3 * P, where);
  for (int q = 0; q < 6; ++q) {
    copy_out(c, gu ? gu[q] : nullptr, c.adj_fin[q], face_count(c, q), where);
    copy_out(c, guo ? guo[q] : nullptr, c.adj_fout[q], face_count(c, q), where);
  }
  return hip_ok(c, hipStreamSynchronize(c.stream), "g2p_adjoint") ? MPF_OK : MPF_HIP_ERROR;
}

int run_advect_adjoint(Ctx& c, const double* gpos_out, const double* gvel_out, double* gpos_in, double* gvel_in,
                       int where, int64_t* in_band) {
  if (!adj_alloc(c)) return MPF_INVALID_ARG;
  if (c.cfg.integrator != MPF_ADVECT_EULER_COLLIDE) {
    c.err = "advection adjoint is implemented for the Euler/collision integrator";
    return MPF_INVALID_ARG;
  }
  const int cur = c.cur;
  const int64_t P = c.P;
  copy_in(c, c.adj_part[0], gvel_out, 3 * P, where);
  copy_in(c, c.adj_part[2], gpos_out, 3 * P, where);
  // the solid level set of this step's forward call (recomputed from the cell
  // lists, which the entry point requires to be current)
  run_solid_phi_and_velocity(c);
  hipMemsetAsync(c.counters + 4, 0, 4, c.stream);
  // g_x -> adj_part[1]; g_v is updated in place in adj_part[0] (each thread
  // reads its own entries before writing them)
  launch(c, "adj_advect", dim3(nblocks(P, 256)), dim3(256), 0, k_adj_advect, c.g, P, (const f3*)c.pos[cur],
         (const f3*)c.vel[cur], (const int8_t*)c.flag[cur], (const float*)c.phisolid, (double)c.cfg.dt,
         (const double*)c.adj_part[2], (const double*)c.adj_part[0], c.adj_part[1], c.adj_part[0],
         c.counters + 4);
  copy_out(c, gpos_in, c.adj_part[1], 3 * P, where);
  copy_out(c, gvel_in, c.adj_part[0], 3 * P, where);
  hipMemcpyAsync(c.counters_host + 4, c.counters + 4, 4, hipMemcpyDeviceToHost, c.stream);
  if (!hip_ok(c, hipStreamSynchronize(c.stream), "advect_adjoint")) return MPF_HIP_ERROR;
  if (in_band) *in_band = c.counters_host[4];
  return MPF_OK;
}

}  // namespace mpf
