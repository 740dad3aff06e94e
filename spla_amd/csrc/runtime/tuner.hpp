// Tile-shape and split-K planner of the FP64 MFMA GEMM.
//
// A plan is picked by a cost model of the launch: for every tile shape and
// split factor the model counts the workgroups of the active tiles over the CUs,
// their time at the shape's sustained MFMA rate, tile padding waste, and the
// HBM time of the split-K reduction; the cheapest plan wins whose sums are no longer
// than the coarse plan's. Plans are cached per problem key and depend only on the
// shape, and so do the kernels' sums, however the operands are aligned: repeated
// calls of one product return bitwise identical results (the batch API's plans, by
// contrast, can be timed: see batched.hpp).
// Environment overrides (for tuning sweeps): SPLA_AMD_TILE=L|M|XL,
// SPLA_AMD_SPLITS=<n>.
#pragma once

#include <cstdint>
#include <map>
#include <mutex>
#include <tuple>

namespace spla_amd {

struct GemmPlan {
  int cfg = 0;          // GemmTileConfig
  int splits = 1;       // split-K factor
  int64_t kSplit = 0;   // embedded reduction length per split
  int64_t kSum = 0;     // embedded length of the sums a split adds up (0: one sum)
  int tilesM = 0, tilesN = 0;
  int activeTiles = 0;  // of these, the tiles that the fill mode needs
  double estSeconds = 0.0;
  bool small = false;   // one launch of small.hip instead of the tiles above
};

// Part of C that a product needs (the kernels' TileFill and offsets).
struct PlanFill {
  int mode = 0;
  int64_t rowOff = 0, colOff = 0;
};

class Tuner {
public:
  // complex: complex operands; m, n, k in elements; numCUs of the device.
  // wholeChip: the product has the device to itself (a single call); false for the
  // block products of a batch, which run side by side on several streams.
  // scalarBytes: 8 or 4 (single precision). fill: whole-device plans count the tiles
  // it leaves.
  GemmPlan plan(bool complex, int layoutA, int layoutB, int64_t m, int64_t n, int64_t k,
                int numCUs, bool wholeChip = true, int scalarBytes = 8,
                const PlanFill& fill = PlanFill());

  // Sustained fraction of the per-CU FP64 matrix rate assumed for a tile config.
  static double efficiency(int cfg);

private:
  using Key = std::tuple<bool, int, int, int64_t, int64_t, int64_t, int, bool, int, int, int64_t>;
  std::mutex lock_;
  std::map<Key, GemmPlan> cache_;
};

// Tiles of rows x cols elements that the fill mode leaves active (the kernels'
// tile_active over all tiles of an m x n matrix).
int64_t plan_active_tiles(int64_t m, int64_t n, int rows, int cols, const PlanFill& fill);

// Plan and time of a coarse model that the forced plans, the block products of a
// batch and the automatic mode's choice of arithmetic are made with: waves of
// workgroups over the resident slots, no fill mode. Its split count also says which
// products the allocation-free entry point takes.
GemmPlan plan_coarse(bool complex, int64_t m, int64_t n, int64_t k, int numCUs, int forceCfg,
                     int forceSplits, bool wholeChip);

// Pure cost model (no state), exposed for tests.
GemmPlan plan_gemm(bool complex, int64_t m, int64_t n, int64_t k, int numCUs, int forceCfg,
                   int forceSplits, const double* effByCfg, bool wholeChip = true,
                   int scalarBytes = 8, const PlanFill& fill = PlanFill());

}  // namespace spla_amd
