// How a solver launch covers the grid (host arithmetic): (j, k) column tiles,
// their planes split along i into runs, one block each (pcg.hip).
#pragma once
#include <algorithm>
#include <cstdint>

namespace mpf {

constexpr int MAX_BLK = 1024;  // blocks per solver launch (k_cgf on large grids: more, tiling_region_blocks)
// Column tiles of TCELLS / TK rows of TK cells, TK = 128 or 64 by the grid
// (make_tiling), with a one-cell ring in LDS.
constexpr int TCELLS = 1024;  // cells of a tile's plane
constexpr int TK_WIDE = 128, TK_NARROW = 64;

struct Tiling {
  int ntj, ntk, seg, nblk;
  int tk;   // cells of a tile along k (TK)
  int ns5;  // single-kernel iteration: blocks of slow-row partials after the nblk tile blocks
};

// Planes are split so the launch has about `blocks` blocks: one resident round
// on 256 CUs, i.e. as many 512-thread blocks as fit a CU at the kernel's
// register use (three for FP32 vectors without slow rows, two otherwise).
// by_offset: the kernel reaches the planes of a run by 32-bit byte offsets
// (k_cgf), so a run has no more of them than these reach as FP64 values.
inline Tiling make_tiling(int nx, int ny, int nz, int blocks, int tk, bool by_offset) {
  Tiling t;
  t.tk = tk;
  t.ns5 = 0;
  const int tj = TCELLS / tk;
  t.ntj = (ny + tj - 1) / tj;
  t.ntk = (nz + tk - 1) / tk;
  const int tiles = t.ntj * t.ntk;
  int nseg = blocks / tiles;
  if (nseg < 1) nseg = 1;
  if (nseg > nx) nseg = nx;
  if (by_offset) {
    const int64_t most = std::max<int64_t>(1, 0xfffffff0ll / (8 * (int64_t)ny * nz) - 6);
    if (nseg < (nx + most - 1) / most) nseg = (int)((nx + most - 1) / most);
  }
  t.seg = (nx + nseg - 1) / nseg;
  nseg = (nx + t.seg - 1) / t.seg;
  t.nblk = tiles * nseg;
  return t;
}

// Wide tiles read whole 512-byte rows and fewer ring cells per plane; narrow
// ones pad less where nz ends early in the last wide tile.  A launch costs
// about (seg + 3) plane steps (three fill the pipeline), a narrow step up to
// 8/7 of a wide one (105 us a narrow launch against 94 at 256^3, where both
// run 32 planes; 56 against 64 at 192^3, 14 planes against 20, before the
// plane loop lost its branches).
inline Tiling make_tiling(int nx, int ny, int nz, int blocks, bool by_offset) {
  const Tiling w = make_tiling(nx, ny, nz, blocks, TK_WIDE, by_offset);
  const Tiling n = make_tiling(nx, ny, nz, blocks, TK_NARROW, by_offset);
  return 8 * (n.seg + 3) < 7 * (w.seg + 3) ? n : w;
}

constexpr int FUSED_BLOCKS = 512;  // blocks k_cgf asks for

// Blocks that a region of the partial sums has room for.  Any tiling has at
// most MAX_BLK if the wide tiles number no more (a larger grid is refused),
// except k_cgf's, whose offsets ask for shorter runs from about 5.4e8 cells
// on: 811^3 has 714 tiles and two runs.
inline int tiling_region_blocks(int nx, int ny, int nz) {
  const Tiling one = make_tiling(nx, ny, nz, 1, TK_WIDE, false);
  if (one.nblk > MAX_BLK) return MAX_BLK;
  return std::max(MAX_BLK, make_tiling(nx, ny, nz, FUSED_BLOCKS, true).nblk);
}

}  // namespace mpf
