// Resident conjugate gradients: one launch runs a whole solve with the
// vectors in registers (included by pcg.hip, inside its anonymous namespace).
//
// What bounds a solve on a grid of up to a few million cells is not memory:
// an iteration as one to three launches takes 20-45 us there whatever the
// size (launches, partial-sum prologues, filling and draining the plane
// pipeline), while its vectors would fit the register files.  Here a block of
// up to 1024 threads per CU owns a tile of bi x bj rows along k: a thread owns
// a column of bi cells along i, with r, q, x and p in registers and p also in
// LDS for its j and k neighbours.  Blocks exchange the q values of their edge
// rows and seven partial sums once per iteration: ring cells (the neighbours'
// edge rows) carry their own copies of r and p, by the same recurrence from
// the same values as their owner's, so q of the ring is all that a block
// needs to form p_k on tile and ring, and alpha, beta and the stop decision
// come from the sums of k_cgf's expansion.
//
// Meeting: every 8-byte word that goes to another block carries 32 bits of
// data and the meeting's number, stored through to memory; a reader polls the
// words that it needs until they carry the number, so arrival and data come
// in one trip, without fences or counters.  Buffers alternate by the meeting's
// number: a block writes for meeting s + 2 only after meeting s + 1, which no
// block joins before it has read all of meeting s.  The block sums are added
// by every block in the same fixed order, so all derive the same scalars bit
// for bit.  The launch is cooperative: every block is resident before any polls.
// Polls are bounded in time; a block that gives up raises a flag (quit) on
// which all leave.  In the last meeting no later one waits for a block that
// gave up, and the others may end the solve without its tile: the flag outlives
// the launch, and a result counts only while it is down (k_collect_rr).
// Otherwise the launch-per-iteration kernels solve, then and in that context
// from then on: blocks that cannot all run at once (two processes on one GPU,
// half of each one's blocks running) would cost every solve the wait.
//
// Measured per iteration (one MI355X, whole solves to 1e-6, launch form -> this
// one; true residuals included; in brackets with six air balls):
//   FP32   64^3 16.0 -> 4.3 us (19.8 -> 4.5), 128^3 26.2 -> 9.2 (29.4 -> 13.0),
//          144^3 40.0 -> 21.4 (43.2 -> 27.7)
//   FP64   64^3 17.3 -> 6.4 (23.8 -> 6.4), 96^3 25.6 -> 11.0 (33.5 -> 12.5),
//          128^3 36.4 -> 25.0 (45.9 -> 31.5)
//   MIXED  64^3 12.7 -> 5.4 (18.4 -> 5.6), 128^3 20.7 -> 12.0 (27.0 -> 17.7),
//          130^3 29.9 -> 19.3 (37.0 -> 28.2), 133^3 29.9 -> 26.2 (36.6 -> 36.0),
//          120 x 128 x 150 27.2 -> 26.2 (33.9 -> 36.4)
// About 4.5 us is the meeting (two trips through memory, the sums and the
// scalars; 32 or 200 blocks differ by 0.4 us), the rest grows with the cells
// per thread and is vector arithmetic, LDS and, in the larger columns, spilled
// registers (RES_M).  So the rule is that the grid fits (resident_tile).  At
// its upper end, 12 cells a thread in the MIXED form (131^3 to 133^3 and
// ragged grids of as many cells), the two forms are about equal: this one takes
// 3 to 15% less without air, 2% less to 7% more with it, and which of them a
// solve is shows only after the form is chosen.

constexpr int RT = 1024;  // threads per block
constexpr int RG = 256;   // most blocks
constexpr int RWORDS = 16;                         // words of a record: (low, high) half of 8 sums
constexpr uint64_t RES_SPIN_TICKS = 200000000ull;  // 2 s of the 100 MHz clock
constexpr int RES_LDS_MAX = 160 * 1024 - 4096;     // dynamic LDS (the static part is below 4 KB)
constexpr uint32_t RES_NONE = 0xffffffffu;

struct ResTile {
  int bi, bj, nti, ntj, nblk, cols, cells;  // tile rows, tiles, blocks; columns (bj * nz) and cells of a full tile
  int m, mj;                                // compiled cells per thread (>= bi), j ring cells per thread
  int dl, dr;                               // FP64: 1/diag in LDS, of own cells, of ring cells
  size_t lds;
  FastDiv dbi;  // by bi * nz
};

template <class V>
struct ResArgs {
  ResTile t;
  uint64_t* rec;     // [2][RG][RWORDS]
  uint64_t* hq[2];   // q of edge rows by block and tile cell (FP64: low halves, then at +plane the high ones)
  uint64_t plane;
  V* hr;             // r of edge rows after a true residual
  double* hx;        // x64 of edge rows for a true residual
  V* beta[6];        // face weights of the slow rows, by cell
  uint32_t* quit;
  uint32_t seq0;     // number of the first meeting
  double eps_abs;    // reference criterion: r.r < eps_abs (negative: relative residual)
  double bc;         // 1/rho of the fast rows
};

// The solve's scalars, in LDS: written by one lane at each meeting, so that
// no wave holds them in registers.
struct ResShared {
  double al, be, rz, rr, rz_prev, bb, stop2, prev_true;
  int next, restarts, it_done;
  int conv, nonfin, missed, lost;
};
// what follows a meeting
constexpr int N_STEP = 1;   // r and x take alpha q, alpha p
constexpr int N_CHECK = 2;  // the next pass only establishes r.z and r.r
constexpr int N_END = 4;    // the solve ends (with N_STEP: x takes its last step)

// Device-scope accesses: through the XCD's L2 to memory, where every XCD sees them.
template <class T>
__device__ __forceinline__ T ld_dev(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
__device__ __forceinline__ void st_dev(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t tagged(uint32_t seq, uint32_t data) { return ((uint64_t)seq << 32) | data; }

// x, its origin hidden from the compiler: what is derived from it is formed
// again where it is used, not kept in registers across the solve's loop.
__device__ __forceinline__ uint32_t fresh(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

// ---- wave sums of eight values at once ----
// Three exchanges halve the values a lane carries (lanes 1, 2 and 4 apart:
// the lane keeps one half and adds the partner's), then the lanes that carry
// the same value (equal lane & 7) are added 8, 16 and 32 apart: 10 double
// additions where eight separate wave sums take 48.
__device__ __forceinline__ double pack64(uint32_t lo, uint32_t hi) {
  return __builtin_bit_cast(double, ((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ uint32_t lo32(double v) { return (uint32_t)__builtin_bit_cast(uint64_t, v); }
__device__ __forceinline__ uint32_t hi32(double v) { return (uint32_t)(__builtin_bit_cast(uint64_t, v) >> 32); }
template <int CTRL>
__device__ __forceinline__ double dpp64(double v) {
  return pack64((uint32_t)__builtin_amdgcn_update_dpp(0, (int)lo32(v), CTRL, 0xF, 0xF, true),
                (uint32_t)__builtin_amdgcn_update_dpp(0, (int)hi32(v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ uint32_t xor4_32(uint32_t v) {
  const int a = __builtin_amdgcn_update_dpp((int)v, (int)v, 0x104, 0xF, 0x5, false);      // row_shl:4 into banks 0, 2
  return (uint32_t)__builtin_amdgcn_update_dpp(a, (int)v, 0x114, 0xF, 0xA, false);  // row_shr:4 into banks 1, 3
}
__device__ __forceinline__ double xor4(double v) { return pack64(xor4_32(lo32(v)), xor4_32(hi32(v))); }
// lanes 16 and 32 apart by the row swaps of v with itself
__device__ __forceinline__ double add16(double v) {
  const auto a = __builtin_amdgcn_permlane16_swap(lo32(v), lo32(v), false, false);
  const auto b = __builtin_amdgcn_permlane16_swap(hi32(v), hi32(v), false, false);
  return pack64(a[0], b[0]) + pack64(a[1], b[1]);
}
__device__ __forceinline__ double add32(double v) {
  const auto a = __builtin_amdgcn_permlane32_swap(lo32(v), lo32(v), false, false);
  const auto b = __builtin_amdgcn_permlane32_swap(hi32(v), hi32(v), false, false);
  return pack64(a[0], b[0]) + pack64(a[1], b[1]);
}
// sum of v over the lanes with this lane's (lane & 7), in all of them
__device__ __forceinline__ double class_sum(double v) {
  v = v + dpp64<0x128>(v);  // row_ror:8
  return add32(add16(v));
}
// lane's value index = 4 * bit0 + 2 * bit1 + bit2 of the lane
__device__ __forceinline__ int wave8_index(int lane) { return ((lane & 1) << 2) | (lane & 2) | ((lane >> 2) & 1); }
__device__ __forceinline__ double wave_sum8(const double (&v)[8], int lane) {
  const bool b0 = lane & 1, b1 = lane & 2, b2 = lane & 4;
  double a[4], c[2];
#pragma unroll
  for (int q = 0; q < 4; ++q) a[q] = (b0 ? v[4 + q] : v[q]) + dpp64<0xB1>(b0 ? v[q] : v[4 + q]);  // quad_perm 1,0,3,2
#pragma unroll
  for (int q = 0; q < 2; ++q) c[q] = (b1 ? a[2 + q] : a[q]) + dpp64<0x4E>(b1 ? a[q] : a[2 + q]);  // quad_perm 2,3,0,1
  return class_sum((b2 ? c[1] : c[0]) + xor4(b2 ? c[0] : c[1]));
}

// The meeting.  v[]: this thread's eight sums.  `load` issues the loads of the
// ring words that this thread needs, `arrived` says whether all of them carry
// the number; `decide` runs on one lane with the totals.  Returns false when
// the solve was given up.  (The polling loop is left lane by lane: nothing
// uniform that is used after it may be decided on inside it.)
template <class FL, class FA, class FD>
__device__ __forceinline__ bool grid_meet(const double (&v)[8], uint32_t seq, uint64_t* rec, uint32_t* quit, int nblk,
                                          int* block_lost, FL load, FA arrived, FD decide) {
  __shared__ double red[RT / 64][8], red2[RT / 64][8];
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  {
    const double s = wave_sum8(v, lane);
    if (lane < 8) red[w][wave8_index(lane)] = s;
  }
  __syncthreads();
  uint64_t* const slot = rec + (size_t)(seq & 1) * RG * RWORDS;
  if (w == 0) {  // value lane & 7 of wave pair lane >> 3
    const double s = class_sum(red[lane >> 3][lane & 7] + red[(lane >> 3) + 8][lane & 7]);
    if (lane < RWORDS)  // word 2 q + half of value q, from lane (q | half << 3)
      st_dev(slot + (size_t)blockIdx.x * RWORDS + 2 * (lane & 7) + (lane >> 3),
             tagged(seq, (lane >> 3) ? hi32(s) : lo32(s)));
  }
  // value t & 7 of records t >> 3 and (t >> 3) + 128
  double s = 0.0;
  {
    const int r0 = t >> 3, r1 = r0 + RT / 8;
    const bool h0 = r0 < nblk, h1 = r1 < nblk;
    const uint64_t* const p0 = slot + (size_t)r0 * RWORDS + 2 * (t & 7);
    const uint64_t* const p1 = slot + (size_t)r1 * RWORDS + 2 * (t & 7);
    uint64_t t0 = 0;
    for (uint32_t spin = 0;; ++spin) {
      uint64_t a0 = 0, a1 = 0, c0 = 0, c1 = 0;
      if (h0) {
        a0 = ld_dev(p0);
        a1 = ld_dev(p0 + 1);
      }
      if (h1) {
        c0 = ld_dev(p1);
        c1 = ld_dev(p1 + 1);
      }
      load();
      bool ok = arrived();
      ok = ok && (!h0 || ((uint32_t)(a0 >> 32) == seq && (uint32_t)(a1 >> 32) == seq)) &&
           (!h1 || ((uint32_t)(c0 >> 32) == seq && (uint32_t)(c1 >> 32) == seq));
      if (ok) {
        s = pack64((uint32_t)a0, (uint32_t)a1) + pack64((uint32_t)c0, (uint32_t)c1);
        break;
      }
      if ((spin & 255u) == 255u) {
        const uint64_t now = wall_clock64();
        if (t0 == 0) t0 = now;
        if (ld_dev(quit) != 0 || now - t0 > RES_SPIN_TICKS) {
          st_dev(quit, 1u);
          *block_lost = 1;
          break;
        }
      }
    }
  }
  s = class_sum(s);
  if (lane < 8) red2[w][lane] = s;
  __syncthreads();
  if (*block_lost) return false;
  if (w == 0) {
    const double f = class_sum(red2[lane >> 3][lane & 7] + red2[(lane >> 3) + 8][lane & 7]);
    double d[8];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      d[q] = pack64(__builtin_amdgcn_readlane(lo32(f), q), __builtin_amdgcn_readlane(hi32(f), q));
    if (lane == 0) decide(d);
  }
  __syncthreads();
  return true;
}

// Whole solve of A x = b.  V: vector type; MIX: FP32 vectors with x64 and an
// FP64 true residual every R iterations (the MIXED form); M: cells per
// thread; MJ: j ring cells per thread.  Results: x (or x64) of every cell, and sc.
//
// One pass of the loop is an iteration k, or (check) a pass that only
// establishes r.z and r.r: of the start, of the residual whose prediction met
// the criterion (FP32 and FP64 forms), or of the FP64 true residual of x
// (MIXED form).
// Registers are what a larger column runs out of: the FP64 form keeps 1/diag
// in LDS where there is room (T.dl, T.dr; up to six cells) and looks it up by
// the open faces of a cell, or in memory for a slow row, elsewhere, and x lives
// in LDS (XL) in the larger columns, where x64 of the MIXED form (always in
// LDS) leaves the room.  The face weights of a slow row are read res_nbf at a
// time: one by one they were a chain of up to six round trips (FP64 at 96^3
// with bubbles 15.7 us an iteration, 12.9 so, 12.7 with 1/diag in LDS, which at
// 112^3 takes 23.9 to 20.9; MIXED at 128^3 with bubbles 25.4 -> 17.8); all six
// at once spill more in the larger columns (FP64 128^3 24.4 -> 32.3 us).
constexpr bool res_xl(int m, bool d64, bool mix) { return d64 ? m >= 3 : mix ? m == 8 : m >= 8; }
constexpr int res_nbf(int m, bool d64, bool mix) { return m <= (d64 ? 4 : mix ? 6 : 8) ? 6 : 3; }
template <class V, bool MIX, int M, int MJ>
__global__ void __launch_bounds__(RT)
    k_cg_resident(OpArgs o, ResArgs<V> ra, const V* __restrict__ b, V* __restrict__ xout, double* __restrict__ x64out,
                  SolveScalars* sc, double tol, int cap, int R) {
  extern __shared__ __align__(16) char smem[];
  __shared__ ResShared sh;
  __shared__ V dtab[8];
  constexpr bool D64 = sizeof(V) == 8, KD = !D64, XL = res_xl(M, D64, MIX);
  constexpr int NBF = res_nbf(M, D64, MIX);
  constexpr bool DL = D64 && M <= 6, DR = D64 && M <= 4;
  const Grid& g = o.g;
  const ResTile& T = ra.t;
  const int t = threadIdx.x, blk = blockIdx.x;
  const int ti = blk / T.ntj, tj = blk - ti * T.ntj;
  const int i0 = ti * T.bi, j0 = tj * T.bj;
  const int ni = min(T.bi, g.nx - i0), nj = min(T.bj, g.ny - j0);
  const int nz = g.nz, SM = (T.bj + 2) * nz;  // LDS stride along i
  const uint32_t sx = (uint32_t)(g.ny * nz);
  const int rj = (int)fdiv((uint32_t)t, g.dnz), kk = t - rj * nz;
  const bool act = rj < nj;  // this thread owns a column
  const bool jedge = act && (rj == 0 || rj == nj - 1);
  const int Lb = act ? (rj + 1) * nz + kk : nz;  // spare threads read the first cell's neighbourhood
  const uint32_t gidx = ((uint32_t)i0 * (uint32_t)g.ny + (uint32_t)(j0 + rj)) * (uint32_t)nz + (uint32_t)kk;
  const uint32_t hb = (uint32_t)blk * (uint32_t)T.cells + (uint32_t)t;  // halo position of own cell m: hb + m * cols
  const uint32_t cols = (uint32_t)T.cols;
  const bool has_lo = act && i0 > 0, has_hi = act && i0 + ni < g.nx;
  const uint32_t ho_lo = hb - (uint32_t)T.ntj * (uint32_t)T.cells + (uint32_t)(T.bi - 1) * cols;
  const uint32_t ho_hi = hb + (uint32_t)T.ntj * (uint32_t)T.cells;
  double* const lx = (double*)smem;                        // MIX: x64 of the tile and its j ring, laid out as p
  V* const lp = (V*)smem + (MIX ? 2 * T.bi * SM : 0);      // p of the tile and its j ring: [bi][bj + 2][nz]
  V* const xs_ = lp + T.bi * SM + (uint32_t)t;             // XL: x of own cell m at xs_[m * RT]
  V* const ds_ = xs_ + (XL ? M * RT : 0);                  // T.dl: 1/diag of own cell m at ds_[m * RT]
  V* const dr_ = ds_ + (T.dl ? M * RT : 0);                // T.dr: of the i ring below and above, of j ring cell m at 2 + m
  if (t < 8) dtab[t] = (t < 7 && o.precond) ? dinv_tab<V>(o, t) : V(1);
  if (t == 0) sh = ResShared{0, 0, 0, 0, 0, 0, 0, -1.0, 0, 0, 0, 0, 0, 0, 0};
  for (int q = t; q < T.bi * SM; q += RT) {
    lp[q] = V(0);
    if (MIX) lx[q] = 0.0;
  }

  auto face_step = [&](int f) -> int64_t {  // cell index step across face f (order of c_off)
    const int64_t st = f % 3 == 0 ? (int64_t)sx : f % 3 == 1 ? nz : 1;
    return f < 3 ? st : -st;
  };
  // 1/diag of a cell with mask nb (1 off the unknowns, whose r is 0)
  auto dinv_of = [&](uint32_t idx, uint32_t nb) -> V {
    if (!o.precond || !(nb & NB_UNKNOWN)) return V(1);
    return (nb & NB_SLOW) ? dslow_at<V>(o, idx) : dinv_tab<V>(o, __popc(nb & 63u));
  };
  V r[M], q[M], p[M], x[XL ? 1 : M], d[KD ? M : 1];
  uint32_t nbw[(M + 3) / 4];
#pragma unroll
  for (int w = 0; w < (M + 3) / 4; ++w) nbw[w] = 0;
#pragma unroll
  for (int m = 0; m < M; ++m) {
    r[m] = q[m] = p[m] = V(0);
    if constexpr (XL) xs_[m * RT] = V(0);
    else x[m] = V(0);
    if constexpr (KD) d[m] = V(1);
    else if (DL && T.dl) ds_[m * RT] = V(1);
    if (act && m < ni) {
      const uint32_t idx = gidx + (uint32_t)m * sx;
      const uint32_t nb = o.nbm[idx];
      nbw[m / 4] |= nb << (8 * (m & 3));
      if constexpr (KD) d[m] = dinv_of(idx, nb);
      else if (DL && T.dl) ds_[m * RT] = dinv_of(idx, nb);
      if (nb & NB_UNKNOWN) r[m] = b[idx];
      if ((nb & (NB_UNKNOWN | NB_SLOW)) == (NB_UNKNOWN | NB_SLOW)) {
        const int8_t mk = o.mark[idx];
        for (int f = 0; f < 6; ++f) {
          if (!(nb & (1u << f))) continue;
          const int64_t n = (int64_t)idx + face_step(f);
          ra.beta[f][idx] = face_beta<V>(o, idx, n, mk, o.mark[n]);
        }
      }
    }
  }
  // i ring: the cells below and above the column, in this thread
  V rl = V(0), rh = V(0), pl = V(0), ph = V(0), dl = V(1), dh = V(1);
  uint32_t nbr = 0;  // their masks
  if (DR && T.dr) dr_[0] = dr_[RT] = V(1);
  if (has_lo) {
    const uint32_t idx = gidx - sx, nb = o.nbm[idx];
    if constexpr (KD) dl = dinv_of(idx, nb);
    else if (DR && T.dr) dr_[0] = dinv_of(idx, nb);
    nbr = nb;
    if (nb & NB_UNKNOWN) rl = b[idx];
  }
  if (has_hi) {
    const uint32_t idx = gidx + (uint32_t)ni * sx, nb = o.nbm[idx];
    if constexpr (KD) dh = dinv_of(idx, nb);
    else if (DR && T.dr) dr_[RT] = dinv_of(idx, nb);
    nbr |= nb << 8;
    if (nb & NB_UNKNOWN) rh = b[idx];
  }
  // j ring: rows -1 and nj of every plane, spread over the threads
  V rg[MJ], dg[KD ? MJ : 1];
  uint32_t ho[MJ], Lg[MJ];  // halo position; LDS offset | mask << 24
#pragma unroll
  for (int m = 0; m < MJ; ++m) {
    const uint32_t e = (uint32_t)(t + RT * m);
    const uint32_t side = fdiv(e, T.dbi), e2 = e - side * T.dbi.d;
    const uint32_t mi = fdiv(e2, g.dnz), k2 = e2 - mi * (uint32_t)nz;
    rg[m] = V(0);
    if constexpr (KD) dg[m] = V(1);
    ho[m] = RES_NONE;
    Lg[m] = 0;
    if (side < 2 && (int)mi < ni && (side == 0 ? j0 > 0 : j0 + nj < g.ny)) {
      const int j = side == 0 ? j0 - 1 : j0 + nj;
      const uint32_t idx = ((uint32_t)(i0 + (int)mi) * (uint32_t)g.ny + (uint32_t)j) * (uint32_t)nz + k2;
      const uint32_t nb = o.nbm[idx];
      if constexpr (KD) dg[m] = dinv_of(idx, nb);
      else if (DR && T.dr) dr_[(2 + m) * RT] = dinv_of(idx, nb);
      if (nb & NB_UNKNOWN) rg[m] = b[idx];
      Lg[m] = (uint32_t)((int)mi * SM + (side == 0 ? 0 : nj + 1) * nz + (int)k2) | (nb << 24);
      ho[m] = (uint32_t)(side == 0 ? blk - 1 : blk + 1) * (uint32_t)T.cells + mi * cols +
              (uint32_t)((side == 0 ? T.bj - 1 : 0) * nz) + k2;
    }
  }
  __syncthreads();

  // 1/diag from the table by a mask, of cell idx() where the row is slow
  auto d_table = [&](uint32_t nb, auto idx) -> V {
    V dv = dtab[(nb & NB_UNKNOWN) ? __popc(nb & 63u) : 7];
    if ((nb & (NB_UNKNOWN | NB_SLOW)) == (NB_UNKNOWN | NB_SLOW) && o.precond) dv = dslow_at<V>(o, idx());
    return dv;
  };
  auto d_own = [&](int m, uint32_t nb) -> V {
    if constexpr (KD) return d[m];
    else if (DL && T.dl) return ds_[m * RT];
    else return d_table(nb, [&]() { return fresh(gidx) + (uint32_t)m * sx; });
  };
  auto nb_own = [&](int m) -> uint32_t { return (fresh(nbw[m / 4]) >> (8 * (m & 3))) & 0xffu; };
  uint32_t seq = ra.seq0;
  int k = 0, refinements = 0;
  bool start = true;   // the first pass
  bool check = true;   // this pass only establishes r.z and r.r
  bool step = false;   // alpha q_{k-1} and alpha p_{k-1} are owed to r and x
  bool new_r = false;  // a true residual replaced r: ring cells take it from hr
  V al = V(0), be = V(0);
  V hl = V(0), hh = V(0), hg[MJ];  // q of the ring
#pragma unroll
  for (int m = 0; m < MJ; ++m) hg[m] = V(0);
  const V qc = qcoef<V>(o);
  auto acc = [](double a, V y, V z) -> double { return __builtin_fma((double)y, (double)z, a); };
  auto put_q = [&](uint32_t at, V v) {
    uint64_t* const h = ra.hq[seq & 1];
    if constexpr (D64) {
      st_dev(h + at, tagged(seq, lo32(v)));
      st_dev(h + ra.plane + at, tagged(seq, hi32(v)));
    } else {
      st_dev(h + at, tagged(seq, __builtin_bit_cast(uint32_t, v)));
    }
  };
  // the words of one q value
  struct QW {
    uint64_t a, c;
  };
  auto get_q = [&](const uint64_t* h, uint32_t at, QW& w) {
    w.a = ld_dev(h + at);
    if constexpr (D64) w.c = ld_dev(h + ra.plane + at);
  };
  auto q_here = [&](const QW& w, V& v) -> bool {
    if constexpr (D64) {
      v = pack64((uint32_t)w.a, (uint32_t)w.c);
      return (uint32_t)(w.a >> 32) == seq && (uint32_t)(w.c >> 32) == seq;
    } else {
      v = __builtin_bit_cast(V, (uint32_t)w.a);
      return (uint32_t)(w.a >> 32) == seq;
    }
  };
  for (;;) {
    // ---- r and x of the column, r of the ring; p_k of both ----
    if (new_r) {
      if (has_lo) rl = ld_dev(ra.hr + fresh(ho_lo));
      if (has_hi) rh = ld_dev(ra.hr + fresh(ho_hi));
#pragma unroll
      for (int m = 0; m < MJ; ++m)
        if (ho[m] != RES_NONE) rg[m] = ld_dev(ra.hr + fresh(ho[m]));
      new_r = false;
    }
    if (step) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        r[m] = r[m] - al * q[m];
        if constexpr (XL) xs_[m * RT] = xs_[m * RT] + al * p[m];
        else x[m] = x[m] + al * p[m];
      }
      rl = rl - al * hl;
      rh = rh - al * hh;
#pragma unroll
      for (int m = 0; m < MJ; ++m) rg[m] = rg[m] - al * hg[m];
    }
    double v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    const bool resid = MIX && (check ? !start : (k + 1) % R == 0);  // a true residual replaces r in this pass
    if (check) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        v[0] = acc(v[0], r[m], r[m] * d_own(m, nb_own(m)));
        v[1] = acc(v[1], r[m], r[m]);
      }
    } else {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        p[m] = r[m] * d_own(m, nb_own(m)) + be * p[m];
        if (act && m < ni) lp[(int)fresh((uint32_t)Lb) + m * SM] = p[m];
        if (M > 4) __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (KD) {
        pl = rl * dl + be * pl;
        ph = rh * dh + be * ph;
      } else if (DR && T.dr) {
        pl = rl * dr_[0] + be * pl;
        ph = rh * dr_[RT] + be * ph;
      } else {
        pl = rl * d_table(fresh(nbr) & 0xffu, [&]() { return fresh(gidx) - sx; }) + be * pl;
        ph = rh * d_table(fresh(nbr) >> 8, [&]() { return fresh(gidx) + (uint32_t)ni * sx; }) + be * ph;
      }
#pragma unroll
      for (int m = 0; m < MJ; ++m)
        if (ho[m] != RES_NONE) {
          const uint32_t lg = fresh(Lg[m]), L = lg & 0xffffffu;
          V dv;
          if constexpr (KD) dv = dg[m];
          else if (DR && T.dr) dv = dr_[(2 + m) * RT];
          else dv = d_table(lg >> 24, [&]() {  // the row's plane and column from its place in the tile
            const uint32_t row = fdiv(L, g.dnz), mi = row / (uint32_t)(T.bj + 2);
            const uint32_t jr = row - mi * (uint32_t)(T.bj + 2);
            return ((uint32_t)(i0 + (int)mi) * (uint32_t)g.ny + (uint32_t)(j0 + (int)jr - 1)) * (uint32_t)nz + (L - row * (uint32_t)nz);
          });
          lp[L] = rg[m] * dv + be * lp[L];
        }
      __syncthreads();
      // ---- q_k = A p_k; q of the edge rows published ----
#pragma unroll
      for (int m = 0; m < M; ++m) {
        if (m < ni) {  // uniform
          const uint32_t nb = nb_own(m);
          const int L = (int)fresh((uint32_t)Lb) + m * SM;
          const V pc = p[m];
          const V n0 = (m + 1 < M) ? (m + 1 < ni ? p[m + 1 < M ? m + 1 : m] : ph) : ph;
          const V n3 = (m > 0) ? p[m > 0 ? m - 1 : 0] : pl;
          const V n1 = lp[L + nz], n4 = lp[L - nz], n2 = lp[L + 1], n5 = lp[L - 1];
          V s = V(0);
          s = (nb & 1) ? s + (n0 - pc) : s;
          s = (nb & 2) ? s + (n1 - pc) : s;
          s = (nb & 4) ? s + (n2 - pc) : s;
          s = (nb & 8) ? s + (n3 - pc) : s;
          s = (nb & 16) ? s + (n4 - pc) : s;
          s = (nb & 32) ? s + (n5 - pc) : s;
          V qv = (nb & NB_UNKNOWN) ? s * qc : V(0);
          if ((nb & (NB_UNKNOWN | NB_SLOW)) == (NB_UNKNOWN | NB_SLOW)) {
            const uint32_t idx = fresh(gidx) + (uint32_t)m * sx;
            s = V(0);
            const V pn[6] = {n0, n1, n2, n3, n4, n5};
#pragma unroll
            for (int f0 = 0; f0 < 6; f0 += NBF) {
              V bf[NBF];  // read together (a closed face's weight is not used)
#pragma unroll
              for (int f = 0; f < NBF; ++f) bf[f] = ra.beta[f0 + f][idx];
              if (NBF < 6) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int f = 0; f < NBF; ++f) s = (nb & (1u << (f0 + f))) ? s + bf[f] * (pn[f0 + f] - pc) : s;
              if (NBF < 6) __builtin_amdgcn_sched_barrier(0);
            }
            qv = s / ((V)g.h * (V)g.h);
          }
          q[m] = qv;
          if (!resid && act && (m == 0 || m == ni - 1 || jedge)) put_q(fresh(hb) + (uint32_t)m * cols, qv);
          const V dv = d_own(m, nb);
          const V z = r[m] * dv;
          v[0] = acc(v[0], r[m], z);
          v[1] = acc(v[1], r[m], r[m]);
          v[2] = acc(v[2], pc, qv);
          v[3] = acc(v[3], qv, z);
          v[4] = acc(v[4], qv, dv * qv);
          v[5] = acc(v[5], qv, r[m]);
          v[6] = acc(v[6], qv, qv);
          if (M > 4) __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    // ---- MIXED: x64 += x, x = 0; r = b - A x64 in FP64, stored in FP32; r
    // of the edge rows left in hr for the ring ----
    if (resid) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        if (act && m < ni) {
          const int L = (int)fresh((uint32_t)Lb) + m * SM;
          const double xn = lx[L] + (double)(XL ? xs_[m * RT] : x[XL ? 0 : m]);
          lx[L] = xn;
          if (m == 0 || m == ni - 1 || jedge) st_dev(ra.hx + (fresh(hb) + (uint32_t)m * cols), xn);
        }
        if constexpr (XL) xs_[m * RT] = V(0);
        else x[m] = V(0);
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): the values have reached memory
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      const double none[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if (!grid_meet(none, seq, ra.rec, ra.quit, T.nblk, &sh.lost, []() {}, []() { return true; },
                     [](const double (&)[8]) {}))
        return;
      ++seq;
      const double xl = has_lo ? ld_dev(ra.hx + fresh(ho_lo)) : 0.0, xh = has_hi ? ld_dev(ra.hx + fresh(ho_hi)) : 0.0;
#pragma unroll
      for (int m = 0; m < MJ; ++m)
        if (ho[m] != RES_NONE) lx[fresh(Lg[m]) & 0xffffffu] = ld_dev(ra.hx + fresh(ho[m]));
      __syncthreads();
      const double ih2 = 1.0 / ((double)g.h * (double)g.h);
      v[0] = v[1] = v[3] = v[5] = 0.0;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const uint32_t nb = nb_own(m);
        if (nb & NB_UNKNOWN) {
          const int L = (int)fresh((uint32_t)Lb) + m * SM;
          const uint32_t idx = fresh(gidx) + (uint32_t)m * sx;
          const double xc = lx[L];
          const double n0 = (m + 1 < ni) ? lx[L + SM] : xh;
          const double n3 = (m > 0) ? lx[L - SM] : xl;
          const double xn[6] = {n0, lx[L + nz], lx[L + 1], n3, lx[L - nz], lx[L - 1]};
          double s = 0.0, ax;
          if (!(nb & NB_SLOW)) {
#pragma unroll
            for (int f = 0; f < 6; ++f)
              if (nb & (1u << f)) s += xn[f] - xc;
            ax = (ra.bc * s) * ih2;
          } else {
            const int8_t mk = o.mark[idx];
#pragma unroll
            for (int f = 0; f < 6; ++f)
              if (nb & (1u << f)) {
                const int64_t n = (int64_t)idx + face_step(f);
                // a neighbour off the unknowns holds pressure 0
                const double xf = is_unknown(OP_VARDENS, o.mark[n]) ? xn[f] : 0.0;
                s += face_beta<double>(o, idx, n, mk, o.mark[n]) * (xf - xc);
              }
            ax = s / ((double)g.h * (double)g.h);
          }
          const double rv = (double)b[idx] - ax;
          const V rf = (V)rv;
          r[m] = rf;
          const V z = rf * d_own(m, nb);
          v[0] = acc(v[0], rf, z);
          v[1] += rv * rv;
          v[3] = acc(v[3], q[m], z);
          v[5] = acc(v[5], q[m], rf);
        }
        if (act && m < ni && (m == 0 || m == ni - 1 || jedge)) {
          const uint32_t at = fresh(hb) + (uint32_t)m * cols;
          st_dev(ra.hr + at, r[m]);
          if (!check) put_q(at, q[m]);  // with the number of the meeting that follows
        }
      }
      __builtin_amdgcn_s_waitcnt(0x0f70);
      __atomic_signal_fence(__ATOMIC_SEQ_CST);
      ++refinements;
      new_r = true;
    }
    // ---- the meeting, and the scalars that follow from it ----
    // the ring words that this thread waits for, as bits (opaque: see grid_meet)
    uint32_t want = (has_lo ? 1u : 0u) | (has_hi ? 2u : 0u);
#pragma unroll
    for (int m = 0; m < MJ; ++m) want |= ho[m] != RES_NONE ? 4u << m : 0u;
    want = fresh(check ? 0u : want);
    QW wl = {0, 0}, wh = {0, 0}, wg[MJ];
#pragma unroll
    for (int m = 0; m < MJ; ++m) wg[m] = QW{0, 0};
    auto load_ring = [&]() {
      const uint64_t* const h = ra.hq[seq & 1];
      if (want & 1u) get_q(h, ho_lo, wl);
      if (want & 2u) get_q(h, ho_hi, wh);
#pragma unroll
      for (int m = 0; m < MJ; ++m)
        if (want & (4u << m)) get_q(h, ho[m], wg[m]);
    };
    auto ring_here = [&]() -> bool {
      bool ok = true;
      ok = (q_here(wl, hl) | !(want & 1u)) & ok;
      ok = (q_here(wh, hh) | !(want & 2u)) & ok;
#pragma unroll
      for (int m = 0; m < MJ; ++m) ok = (q_here(wg[m], hg[m]) | !(want & (4u << m))) & ok;
      return ok;
    };
    auto scalars = [&](const double (&s)[8]) {
      auto below = [&](double rr2) -> bool { return ra.eps_abs >= 0.0 ? rr2 < ra.eps_abs : rr2 <= sh.stop2; };
      int nx = 0;
      if (!check) {  // s: the sums of iteration k; what iteration k + 1 needs
        const bool zero_pq = s[2] == 0.0, bad_pq = bad(s[2]);
        const double a = zero_pq || bad_pq ? 0.0 : s[0] / s[2];
        const double rzn = (s[0] - (2.0 * a) * s[3]) + (a * a) * s[4];
        const double rrn = (s[1] - (2.0 * a) * s[5]) + (a * a) * s[6];
        // the expansion has lost its digits (see cg_scalars)
        const bool spent = !(rzn * s[0] > 0.0) || (o.precond && !zero_pq && !(a > 0.0)) || rrn > 1e12 * sh.bb;
        const bool met = zero_pq || spent || below(rrn > 0.0 ? rrn : 0.0);
        sh.al = a;
        sh.be = rzn / s[0];
        sh.rz = rzn;
        sh.rr = rrn;
        sh.rz_prev = s[0];
        sh.it_done = k + 1;
        if (bad(rzn) || bad(rrn) || bad_pq) {
          sh.nonfin = 1;
          nx = N_END;
        } else if (!MIX && zero_pq) {  // the launch form records the iteration that met it
          sh.conv = 1;
          sh.it_done = k;
          nx = N_END;
        } else if (met || (!MIX && k + 1 >= cap)) {
          nx = N_CHECK | (zero_pq ? 0 : N_STEP);
        } else {
          nx = N_STEP | (k + 1 >= cap ? N_END : 0);
        }
      } else {  // r.z and r.r as they are
        const bool nf = bad(s[0]) || bad(s[1]);
        sh.al = sh.be = 0.0;
        sh.rz = s[0];
        sh.rr = s[1];
        sh.nonfin = nf;
        if (start) {
          sh.bb = s[1];
          sh.stop2 = (tol * tol) * s[1];
        }
        if (MIX && !start) {  // the FP64 true residual decides; the iteration restarts from it
          const bool cv = s[1] <= sh.stop2;
          const bool stagnant = sh.prev_true >= 0.0 && s[1] > 0.25 * sh.prev_true;
          sh.prev_true = s[1];
          sh.conv = cv;
          if (!cv && (k >= cap || ++sh.restarts > MAX_RESTARTS || stagnant || nf)) sh.missed = 1;
          if (cv || sh.missed) nx = N_END;
        } else {
          const bool cv = below(s[1]);
          sh.conv = cv;
          if (cv || nf || k >= cap) nx = N_END;
          else if (!start) sh.be = s[0] / sh.rz_prev;
        }
      }
      sh.next = nx;
    };
    if (!grid_meet(v, seq, ra.rec, ra.quit, T.nblk, &sh.lost, load_ring, ring_here, scalars)) return;
    ++seq;
    const int next = __builtin_amdgcn_readfirstlane(sh.next);
    al = uniform_reg((V)sh.al);
    be = uniform_reg((V)sh.be);
    if (!check) ++k;
    if (next & N_END) {
      if (next & N_STEP)  // x takes its last step
#pragma unroll
        for (int m = 0; m < M; ++m) {
          if constexpr (XL) xs_[m * RT] = xs_[m * RT] + al * p[m];
          else x[m] = x[m] + al * p[m];
        }
      break;
    }
    step = (next & N_STEP) != 0;
    check = (next & N_CHECK) != 0;
    start = false;
  }
#pragma unroll
  for (int m = 0; m < M; ++m) {
    if (!(act && m < ni)) continue;
    const uint32_t idx = gidx + (uint32_t)m * sx;
    const V xv = XL ? xs_[m * RT] : x[XL ? 0 : m];
    if (MIX) x64out[idx] = lx[Lb + m * SM] + (double)xv;
    else xout[idx] = xv;
  }
  if (blk == 0 && t == 0) {
    sc->iter = sh.it_done;
    sc->converged = (sh.conv && !sh.nonfin) || sh.missed;  // as the launch form: the host lowers it when missed
    sc->nonfinite = sh.nonfin && !sh.missed;
    // x = 0 may meet the criterion: then r = b is its true residual
    sc->refinements = refinements + ((MIX && start && sh.conv) ? 1 : 0);
    sc->rr = sh.rr;
    sc->rz = sh.rz;
    sc->bb = sh.bb;
    sc->res_missed = sh.missed;
    sc->res_restarts = sh.restarts;
    sc->res_seq = seq;
    sc->done = 1;
  }
}

__global__ void k_res_clear(uint32_t* quit, uint32_t raised, SolveScalars* sc) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *quit = raised;
    sc->done = 0;
  }
}
__global__ void k_res_words(uint64_t* w, int64_t n) {  // no word carries a meeting's number
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (int64_t)gridDim.x * blockDim.x) w[q] = 0;
}

// Compiled sizes: cells and j ring cells per thread.  1024 threads a CU have
// 128 vector registers each.  r, q, p and, in FP32 and MIXED, 1/diag are in
// registers, x too where it is not in LDS (res_xl); what does not fit goes
// through scratch memory in every iteration.  The compiler spills, at 3, 4, 6,
// 8, 10 and 12 cells, 0, 0, 9, 28, 174 and 234 registers (FP32; up to 204
// bytes a lane), 4, 8, 65, 72, 199 and 278 (MIXED; up to 332 bytes) and 4, 18,
// 80 and 141 (FP64; up to 224 bytes): part of the step from 12.0 to 19.3 us
// between 128^3 and 130^3 in the MIXED form (8 and 10 cells).
constexpr int RES_NM = 8;
constexpr int RES_M[RES_NM] = {1, 2, 3, 4, 6, 8, 10, 12}, RES_MJ[RES_NM] = {1, 1, 2, 2, 3, 3, 4, 4};
constexpr int RES_NM64 = 6;

// Tile of a resident solve on at most `most` blocks: fewest cells per thread,
// then the smallest ring, then the fewest blocks.  False: the grid does not
// fit (registers, LDS or threads) and the launch-per-iteration kernels run.
inline bool resident_tile(const Grid& g, int most, int esize, bool mix, ResTile& out) {
  const int mmax = (esize == 8) ? RES_NM64 : RES_NM;
  int64_t best = -1;
  if (g.nz > RT) return false;
  for (int ntj = 1; ntj <= most && ntj <= g.ny; ++ntj) {
    const int bj = (g.ny + ntj - 1) / ntj;
    if ((int64_t)bj * g.nz > RT || (g.ny + bj - 1) / bj != ntj) continue;
    for (int nti = most / ntj; nti >= 1; --nti) {
      const int bi = (g.nx + nti - 1) / nti;
      if ((g.nx + bi - 1) / bi != nti) continue;
      if (bi > RES_M[mmax - 1]) break;
      const int64_t tile = (int64_t)bi * (bj + 2) * g.nz;
      int mi = 0;
      while (mi < mmax && (RES_M[mi] < bi || (int64_t)RES_MJ[mi] * RT < (int64_t)2 * bi * g.nz)) ++mi;
      if (mi >= mmax) continue;
      // x64 (MIXED), p, and x of the larger columns
      const int64_t lds = tile * (esize + (mix ? 8 : 0)) +
                          (res_xl(RES_M[mi], esize == 8, mix) ? (int64_t)RES_M[mi] * RT * esize : 0);
      if (tile >= (1 << 24) || lds > RES_LDS_MAX) continue;
      const int64_t ring = (int64_t)2 * (bi + bj) * g.nz;
      const int64_t cost = ((int64_t)mi * (1 << 20) + ring) * 1024 + nti * ntj;
      if (best >= 0 && cost >= best) continue;
      best = cost;
      out.bi = bi; out.bj = bj; out.nti = nti; out.ntj = ntj;
      out.nblk = nti * ntj;
      out.cols = bj * g.nz;
      out.cells = bi * bj * g.nz;
      out.m = RES_M[mi]; out.mj = RES_MJ[mi];
      out.dl = out.dr = 0;
      int64_t more = lds;
      if (esize == 8 && out.m <= 6 && more + (int64_t)out.m * RT * 8 <= RES_LDS_MAX) {
        out.dl = 1;
        more += (int64_t)out.m * RT * 8;
      }
      if (esize == 8 && out.m <= 4 && more + (int64_t)(2 + out.mj) * RT * 8 <= RES_LDS_MAX) {
        out.dr = 1;
        more += (int64_t)(2 + out.mj) * RT * 8;
      }
      out.lds = (size_t)more;
    }
  }
  if (best < 0) return false;
  out.dbi = make_fastdiv((uint32_t)(out.bi * g.nz));
  return true;
}

template <class V, bool MIX>
using ResKernel = void (*)(OpArgs, ResArgs<V>, const V*, V*, double*, SolveScalars*, double, int, int);
template <class V, bool MIX>
ResKernel<V, MIX> resident_kernel(int m) {
  switch (m) {
    case 1: return k_cg_resident<V, MIX, 1, 1>;
    case 2: return k_cg_resident<V, MIX, 2, 1>;
    case 3: return k_cg_resident<V, MIX, 3, 2>;
    case 4: return k_cg_resident<V, MIX, 4, 2>;
    case 6: return k_cg_resident<V, MIX, 6, 3>;
    case 8: return k_cg_resident<V, MIX, 8, 3>;
    default: break;
  }
  if constexpr (sizeof(V) == 4) return m == 10 ? k_cg_resident<V, MIX, 10, 4> : k_cg_resident<V, MIX, 12, 4>;
  return nullptr;
}

inline uint32_t* resident_quit(Ctx& c) { return (uint32_t*)(c.res_buf + 2 * RG * RWORDS); }

// Queues a resident solve (after the masks).  False when it cannot run: the
// grid does not fit, the device cannot hold all blocks at once, or an earlier
// one of this context was left by a block that waited too long.
template <class V, bool MIX>
bool resident_launch(Ctx& c, const OpArgs& o, const V* b, V* x, double* x64, double eps_abs, double tol, int cap, int R,
                     double bc) {
  ResArgs<V> a;
  if (!c.res_buf || c.res_off || !resident_tile(c.g, c.res_blocks, (int)sizeof(V), MIX, a.t)) return false;
  const int64_t n = (int64_t)a.t.nblk * a.t.cells;
  if (n > c.res_cells) return false;
  // records, quit word, then q halos (two buffers of two planes), r and x64 halos
  const int64_t words = 2 * RG * RWORDS + 16 + 4 * c.res_cells;
  uint64_t* base = (uint64_t*)c.res_buf;
  a.rec = base;
  a.quit = resident_quit(c);
  uint64_t* h = base + 2 * RG * RWORDS + 16;
  a.plane = (uint64_t)c.res_cells;
  a.hq[0] = h;
  a.hq[1] = h + 2 * c.res_cells;
  a.hr = (V*)(h + 4 * c.res_cells);
  a.hx = (double*)(h + 5 * c.res_cells);
  void* spare[6] = {c.vp, c.vq, c.vp2, c.vr2, c.vq2, c.vp3};  // the launch form's vectors
  for (int f = 0; f < 6; ++f) a.beta[f] = (V*)spare[f];
  a.eps_abs = eps_abs;
  a.bc = bc;
  auto kern = resident_kernel<V, MIX>(a.t.m);
  if (!kern) return false;
  if (hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)a.t.lds) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  // meeting numbers are not used twice while a word may still carry them
  if (c.res_seq == 0 || c.res_seq > 0x7fffffffu) {
    launch(c, "pcg_res_words", dim3(256), dim3(256), 0, k_res_words, base, words);
    c.res_seq = 1;
  }
  a.seq0 = c.res_seq;
  launch(c, "pcg_res_clear", dim3(1), dim3(64), 0, k_res_clear, a.quit, c.res_raise_quit ? 1u : 0u, c.scal);
  c.res_raise_quit = false;
  OpArgs oc = o;
  SolveScalars* sc = c.scal;
  void* args[] = {(void*)&oc, (void*)&a, (void*)&b, (void*)&x, (void*)&x64, (void*)&sc, (void*)&tol, (void*)&cap,
                  (void*)&R};
  PendingEvent pe;
  const bool timed = launch_begin(c, "pcg_resident", pe);
  const hipError_t e = hipLaunchCooperativeKernel((const void*)kern, dim3(a.t.nblk), dim3(RT), args,
                                                  (unsigned)a.t.lds, c.stream);
  if (e != hipSuccess) (void)hipGetLastError();
  launch_end(c, pe, timed);
  return e == hipSuccess;
}
