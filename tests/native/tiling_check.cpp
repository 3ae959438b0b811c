// Checks the solver launches' tiling (csrc/tiling.h) over all grids a context
// accepts: a grid is solved exactly if its wide tiles number at most MAX_BLK,
// every launch's blocks have room in the partial sums, the runs cover the
// planes, and the planes of k_cgf's runs stay within 32-bit byte offsets.
#include "../../2017multiphase_amd/csrc/tiling.h"

#include <cmath>
#include <cstdio>
#include <random>

using namespace mpf;

static int bad = 0;
static void check(int nx, int ny, int nz) {
  const int64_t tiles = (int64_t)((ny + 7) / 8) * ((nz + 127) / 128);
  const int room = tiling_region_blocks(nx, ny, nz);
  const Tiling all[] = {make_tiling(nx, ny, nz, 768, false), make_tiling(nx, ny, nz, 512, false),
                        make_tiling(nx, ny, nz, 256, TK_WIDE, false), make_tiling(nx, ny, nz, 512, TK_WIDE, false),
                        make_tiling(nx, ny, nz, FUSED_BLOCKS, true)};
  for (int q = 0; q < 5; ++q) {
    const Tiling& t = all[q];
    const int nseg = t.nblk / (t.ntj * t.ntk);
    bool ok = room >= MAX_BLK && (int64_t)nseg * t.seg >= nx && (int64_t)(nseg - 1) * t.seg < nx &&
              (tiles > MAX_BLK || t.nblk <= room) &&
              (int64_t)t.ntj * (TCELLS / t.tk) >= ny && (int64_t)t.ntk * t.tk >= nz;
    // k_cgf: from one plane below a run to four past it
    if (q == 4 && tiles <= MAX_BLK) ok = ok && (uint64_t)(t.seg + 6) * 8ull * ny * nz <= 0xfffffff0ull;
    if (!ok) {
      std::printf("%d x %d x %d, launch %d: tiles %lld room %d tk %d seg %d blocks %d\n", nx, ny, nz, q,
                  (long long)tiles, room, t.tk, t.seg, t.nblk);
      ++bad;
    }
  }
}

int main() {
  const int64_t most = 0xffffffffll / 3;  // cells of a context
  const int edge[][3] = {{4, 4, 4}, {256, 256, 256}, {811, 811, 811}, {860, 860, 860}, {900, 900, 900}, {1024, 1024, 1024},
                         {1398, 1000, 1024}, {1430, 1000, 1000}, {5000000, 16, 16}, {4, 8, 131072}, {4, 8, 131073}};
  for (const auto& e : edge) check(e[0], e[1], e[2]);
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  for (int q = 0; q < 400000; ++q) {
    // sides log-uniform, most of them as large as a context takes
    const double a = 4 * std::pow(2000.0, u(rng)), b = 4 * std::pow(2000.0, u(rng));
    const double c = std::min(std::pow(10.0, 4 + 5.2 * std::sqrt(u(rng))) / (a * b), 1e7);
    const int nx = (int)c, ny = (int)a, nz = (int)b;
    if (nx < 4 || (int64_t)nx * ny * nz > most) continue;
    check(nx, ny, nz);
  }
  std::printf("%d bad\n", bad);
  return bad != 0;
}
