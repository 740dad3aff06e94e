// C entry point over the whole-device planner and the coarse plan it starts from, for
// the host tests (tests/test_plan_sums_host.py).
#include "runtime/tuner.hpp"

extern "C" {

// out: [splits, kSplit] of the plan, [splits, kSplit] of the coarse plan, small, kSum
void plan_sums_c(int complex, long long m, long long n, long long k, int scalarBytes, int mode,
                 long long* out) {
  const double eff[3] = {spla_amd::Tuner::efficiency(0), spla_amd::Tuner::efficiency(1),
                         spla_amd::Tuner::efficiency(2)};
  const spla_amd::GemmPlan p = spla_amd::plan_gemm(complex != 0, m, n, k, 256, -1, 0, eff, true,
                                                   scalarBytes, spla_amd::PlanFill{mode, 0, 0});
  const spla_amd::GemmPlan c = spla_amd::plan_coarse(complex != 0, m, n, k, 256, -1, 0, true);
  out[0] = p.splits;
  out[1] = p.kSplit;
  out[2] = c.splits;
  out[3] = c.kSplit;
  out[4] = p.small;
  out[5] = p.kSum;
}
}
