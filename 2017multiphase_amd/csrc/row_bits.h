// The phases of the cells as bits, row by row along k, in words of 64: cell
// (i, j, k) at bit k + 2 of row (i + 2, j + 2), with empty rows and bits around
// the grid, so that every row of a window of up to five cells is a few bits of
// one unaligned read (run_row_bits, grid.hip).
#pragma once
#include <cstdint>

namespace mpf {

struct RowBits {
  const uint64_t* f;  // liquid or solid
  const uint64_t* a;  // air (also single air particles)
  int nw;             // words a row
  int ny4;            // rows a plane
  uint32_t* odd;      // set by run_air_regular: some air particle is not finite or off the grid
};

// Cells k-2 .. k+2 (bits 0 .. 4) of row (i, j), both counted with the border.
__device__ __forceinline__ uint32_t row_window(const uint64_t* __restrict__ rows, const RowBits& rb, int i, int j, int k) {
  uint16_t v;
  __builtin_memcpy(&v, (const uint8_t*)(rows + ((int64_t)i * rb.ny4 + j) * rb.nw) + (k >> 3), 2);
  return ((uint32_t)v >> (k & 7)) & 31u;
}

// The air window of a face of axis A (four cells along A, five across) as rows
// of NK bits in two words.  Across the face the outer cells lie 1.5 cells or
// more from its centre, beyond the kernel's 1.4: their weights are 0, and
// with finite particles inside their cells 0 is all they add.  near[] keeps
// the 36 cells that can weigh.
template <int A>
struct AirWindow {
  static constexpr int NI = A == 0 ? 4 : 5, NJ = A == 1 ? 4 : 5, NK = A == 2 ? 4 : 5, RW = 64 / NK;
  static constexpr uint32_t ROW = (1u << NK) - 1u;
  static_assert(NI * NJ <= 2 * RW, "two words");
  static constexpr bool row_near(int r) {
    const int di = r / NJ, dj = r % NJ;
    return (A == 0 || (di >= 1 && di <= 3)) && (A == 1 || (dj >= 1 && dj <= 3));
  }
  static constexpr uint32_t bits_near = A == 2 ? 15u : 14u;
  static constexpr uint64_t near_word(int word) {
    uint64_t m = 0;
    for (int r = word * RW; r < NI * NJ && r < (word + 1) * RW; ++r)
      if (row_near(r)) m |= (uint64_t)bits_near << (NK * (r % RW));
    return m;
  }
};

}  // namespace mpf
