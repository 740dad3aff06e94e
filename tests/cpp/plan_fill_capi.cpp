// C entry points over the whole-device planner with fill modes and single
// precision, for the host tests (tests/test_plan_fill_host.py).
#include "runtime/tuner.hpp"

extern "C" {

long long plan_active_tiles_c(long long m, long long n, int rows, int cols, int mode,
                              long long rowOff, long long colOff) {
  return spla_amd::plan_active_tiles(m, n, rows, cols, spla_amd::PlanFill{mode, rowOff, colOff});
}

// out: [cfg, splits, kSplit, tilesM, tilesN]
void plan_fill_c(int complex, long long m, long long n, long long k, int scalarBytes, int mode,
                 long long rowOff, long long colOff, long long* out) {
  const double eff[3] = {spla_amd::Tuner::efficiency(0), spla_amd::Tuner::efficiency(1),
                         spla_amd::Tuner::efficiency(2)};
  spla_amd::GemmPlan p =
      spla_amd::plan_gemm(complex != 0, m, n, k, 256, -1, 0, eff, true, scalarBytes,
                          spla_amd::PlanFill{mode, rowOff, colOff});
  out[0] = p.cfg;
  out[1] = p.splits;
  out[2] = p.kSplit;
  out[3] = p.tilesM;
  out[4] = p.tilesN;
}
}
