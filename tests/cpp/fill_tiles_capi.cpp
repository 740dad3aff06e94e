// C entry points over kernels/fill_tiles.hpp for the host tests
// (tests/test_fill_tiles_host.py).
#include "kernels/fill_tiles.hpp"

namespace {
spla_amd::FillTiles make(const long long* p) {
  const long long m = p[0], n = p[1];
  const int rows = static_cast<int>(p[2]), cols = static_cast<int>(p[3]);
  return {static_cast<int>(p[4]), p[5], m, n, rows, cols, (m + rows - 1) / rows,
          (n + cols - 1) / cols};
}
}  // namespace

extern "C" {

long long fill_total(const long long* p) { return make(p).total(); }

void fill_locate(const long long* p, long long t, int* out) { make(p).locate(t, out[0], out[1]); }
}
