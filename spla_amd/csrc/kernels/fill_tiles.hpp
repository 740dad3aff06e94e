// The tiles of a matrix that a fill mode needs, counted and enumerated column by column
// without a loop over the columns. Host and device code.
//
// A tile of rows x cols elements at (r, c) with nr x nc elements inside the matrix is
// active if (SPLA's block_is_active, src/block_generation/block.hpp:58-66)
//   upper: c + nc + colOff > r + rowOff,   lower: r + nr + rowOff > c + colOff.
// So the active tiles of a tile column are those in front of, or behind, a row that moves
// by cols from one column to the next: a sum of floors of an arithmetic sequence, which
// has a closed form as rows and cols are powers of two.
//
// Why not walk the columns: every workgroup looks its tile up, and with hundreds of tile
// columns the walk outlasts a short product. Measured, walk / closed form: real
// 40000 x 40000 x 64, upper, 22.6 / 3.3 ms, complex 100 x 4e6 x 40, upper, 2005 /
// 4.5 ms.
#pragma once

#include <cstdint>

#include "kernels/gemm_desc.hpp"

namespace spla_amd {

struct FillTiles {
  int mode;        // TileFill, not FillFull
  int64_t off;     // colOff - rowOff
  int64_t m, n;    // elements
  int rows, cols;  // of a tile, powers of two
  int64_t tilesM, tilesN;

  static constexpr int64_t low(int64_t a, int64_t b) { return a < b ? a : b; }
  static constexpr int64_t high(int64_t a, int64_t b) { return a > b ? a : b; }
  // a / d and the same rounded up (0 for a <= 0) by a power of two; a shift also where the
  // kernel does not know d beforehand
  static constexpr int64_t div(int64_t a, int64_t d) { return a >> __builtin_ctzll(d); }
  static constexpr int64_t up(int64_t a, int64_t d) { return a > 0 ? div(a + d - 1, d) : 0; }

  // active tile rows [first_row, end_row) of tile column tn
  constexpr int64_t first_row(int64_t tn) const {
    const int64_t c = tn * cols + off;
    return mode != FillLower || c <= 0 ? 0 : (c >= m ? tilesM : div(c, rows));
  }
  constexpr int64_t end_row(int64_t tn) const {
    return mode != FillUpper ? tilesM : low(tilesM, up(low((tn + 1) * cols, n) + off, rows));
  }
  constexpr int64_t column(int64_t tn) const { return high(0, end_row(tn) - first_row(tn)); }

  // sum of floor((u cols + b) / rows) over u < x, b >= 0
  constexpr int64_t floors(int64_t x, int64_t b) const {
    if (cols >= rows) return x * (x - 1) / 2 * div(cols, rows) + x * div(b, rows);
    const int64_t r = div(rows, cols);
    return quotients(div(b, cols) + x, r) - quotients(div(b, cols), r);
  }
  // sum of floor(v / r) over v < y
  static constexpr int64_t quotients(int64_t y, int64_t r) {
    const int64_t a = div(y, r);
    return a * (a - 1) / 2 * r + a * (y - a * r);
  }

  // active tiles of the tile columns in front of tn < tilesN (whole columns)
  constexpr int64_t before(int64_t tn) const {
    if (mode == FillUpper) {
      // column u ends at tile row floor((u cols + b) / rows) between 0 and tilesM
      const int64_t b = cols + off + rows - 1;
      const int64_t zero = low(tn, up(rows - b, cols));         // columns without a tile
      const int64_t full = low(tn, up(tilesM * rows - b, cols));  // from here on: all rows
      return floors(full - zero, zero * cols + b) + (tn - full) * tilesM;
    }
    // column u begins at tile row floor((u cols + off) / rows) up to its last tile
    const int64_t some = low(tn, up(m - off, cols));  // columns with a tile
    const int64_t all = low(some, up(rows - off, cols));  // columns with all of them
    return some * tilesM - floors(some - all, all * cols + off);
  }
  constexpr int64_t total() const { return before(tilesN - 1) + column(tilesN - 1); }

  // tile t, counted down the columns, 0 <= t < total()
  constexpr void locate(int64_t t, int& tm, int& tn) const {
    int64_t a = 0, e = tilesN;  // before(a) <= t, before(e) > t or e == tilesN
    while (e - a > 1) {
      const int64_t mid = a + (e - a) / 2;
      if (before(mid) <= t)
        a = mid;
      else
        e = mid;
    }
    tn = static_cast<int>(a);
    tm = static_cast<int>(first_row(a) + t - before(a));
  }
};

}  // namespace spla_amd
