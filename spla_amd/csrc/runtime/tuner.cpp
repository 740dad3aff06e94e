#include "runtime/tuner.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "kernels/fill_tiles.hpp"
#include "kernels/gemm_desc.hpp"

namespace spla_amd {
namespace {

// Per-CU FP64 matrix rate of gfx950: 128 flop / clock / CU at 2.4 GHz.
constexpr double kPeakPerCU = 128.0 * 2.4e9;
constexpr double kHbmBytesPerSecond = 5.0e12;  // sustained, for the split-K reduction
constexpr double kLaunchSeconds = 4.0e-6;

int blocks_per_cu(int cfg) {
  switch (cfg) {
    case TileM:
      return 4;
    default:
      return 2;
  }
}

int env_int(const char* name, int dflt) {
  const char* v = std::getenv(name);
  if (!v || !*v) return dflt;
  return std::atoi(v);
}

int env_tile() {
  const char* v = std::getenv("SPLA_AMD_TILE");
  if (!v) return -1;
  if (!std::strcmp(v, "L")) return TileL;
  if (!std::strcmp(v, "M")) return TileM;
  if (!std::strcmp(v, "XL")) return TileXL;
  return -1;
}

}  // namespace

GemmPlan plan_coarse(bool complex, int64_t m, int64_t n, int64_t k, int numCUs, int forceCfg,
                     int forceSplits, bool wholeChip) {
  const int64_t Mp = complex ? 2 * m : m;
  const int64_t Kp = complex ? 2 * k : k;
  constexpr int cands[] = {TileL, TileM, TileXL};
  constexpr double rate[] = {0.8, 0.55, 0.85};  // L, M, XL
  GemmPlan best;
  best.estSeconds = 1e300;
  for (int cfg : cands) {
    if (forceCfg >= 0 && cfg != forceCfg) continue;
    if (forceCfg < 0 && cfg == TileXL) continue;  // opt-in only
    const TileShape ts = tile_shape(cfg);
    const int64_t tilesM = (Mp + ts.bm - 1) / ts.bm;
    const int64_t tilesN = (n + ts.bn - 1) / ts.bn;
    const int64_t tiles = tilesM * tilesN;
    const int64_t kBlocks = std::max<int64_t>(1, (Kp + ts.bk - 1) / ts.bk);
    const int bpc = blocks_per_cu(cfg);
    const int64_t slots = static_cast<int64_t>(numCUs) * bpc;
    const double eff = rate[cfg];
    // split factors: every split keeps at least 8 k-blocks; up to 64, or, for a
    // product that has the device to itself, as many as fill the resident workgroup
    // slots when there are few tiles (small m, n and a long reduction: HBM-bound,
    // every CU must stream its share of A and B). Batch blocks share the device
    // with the blocks on the other streams and keep the cap of 64.
    const int64_t fillSplits = wholeChip ? slots / std::max<int64_t>(1, tiles) : 0;
    const int64_t maxSplits = std::max<int64_t>(
        1, std::min<int64_t>(kBlocks / 8, std::max<int64_t>(64, fillSplits)));
    // A and B are read once whatever the split; with fewer workgroups than resident
    // slots only that share of the HBM bandwidth is drawn
    const double bytes = static_cast<double>(m + n) * static_cast<double>(k) * (complex ? 16.0 : 8.0);
    // candidates 1, 2, 3, 4, 6, 9, ... up to maxSplits and the count that fills every
    // resident slot once, or exactly the forced count
    const int64_t forced = forceSplits > 0 ? std::min<int64_t>(forceSplits, maxSplits) : 0;
    std::vector<int64_t> cand;
    if (forced > 0) {
      cand.push_back(forced);
    } else {
      for (int64_t s = 1; s <= maxSplits; s = (s < 4 ? s + 1 : s * 3 / 2)) cand.push_back(s);
      if (fillSplits > 0 && fillSplits <= maxSplits) cand.push_back(fillSplits);
    }
    for (const int64_t s : cand) {
      const int64_t kbPerSplit = (kBlocks + s - 1) / s;
      const int64_t splits = (kBlocks + kbPerSplit - 1) / kbPerSplit;  // no empty split
      const int64_t blocks = tiles * splits;
      if (blocks > (int64_t(1) << 31) - 1) continue;
      const int64_t waves = (blocks + slots - 1) / slots;
      const double blockFlops = 2.0 * ts.bm * ts.bn * kbPerSplit * ts.bk;
      const double waveSeconds = blockFlops * bpc / (kPeakPerCU * eff);
      // HBM throughput grows with the resident workgroups (their loads in flight)
      const double active = std::min(1.0, static_cast<double>(blocks) / slots);
      const double tMem = wholeChip ? bytes / (kHbmBytesPerSecond * active) : 0.0;
      double t = std::max(waves * waveSeconds, tMem) + kLaunchSeconds;
      if (splits > 1)
        t += (splits + 2) * 8.0 * Mp * n / kHbmBytesPerSecond + kLaunchSeconds;
      if (t < best.estSeconds * 0.999) {
        best.cfg = cfg;
        best.splits = static_cast<int>(splits);
        best.kSplit = kbPerSplit * ts.bk;
        best.tilesM = static_cast<int>(tilesM);
        best.tilesN = static_cast<int>(tilesN);
        best.estSeconds = t;
      }
    }
  }
  if (best.kSplit <= 0) {
    // no candidate passed (e.g. a forced tile whose grid would not fit): one split
    best.cfg = forceCfg >= 0 ? forceCfg : TileL;
    const TileShape ts = tile_shape(best.cfg);
    best.splits = 1;
    best.kSplit = std::max<int64_t>(1, (Kp + ts.bk - 1) / ts.bk) * ts.bk;
    best.tilesM = static_cast<int>((Mp + ts.bm - 1) / ts.bm);
    best.tilesN = static_cast<int>((n + ts.bn - 1) / ts.bn);
  }
  return best;
}

namespace {

// Bytes of partial sums. The allocation-free entry point (complex doubles) holds
// 64 MiB: a product whose coarse plan fits, with one split too, keeps within it.
constexpr double kSmallWorkspace = 64.0 * (1 << 20);
constexpr double kLargestWorkspace = 256.0 * (1 << 20);

// Products that one launch of 16 x 16 tiles (small.hip) does in less time than the tile
// kernels. Its waves hold 512 reduction indices in flight, and every tile reads its rows
// of A and B anew. Measured, us a call, tile kernels / small (launch and wait alone are
// 15.6): d 13 x 32 x 263 24.4 / 17.2, 256 x 256 x 1024 27.1 / 22.4, 512 x 512 x 263 29.3 /
// 21.4, but 13 x 32 x 2048 27.3 / 26.9 (A^T B 26.8 / 28.7) and 512 x 512 x 512 A^T B 28.1 /
// 31.3; z 256 x 256 x 512 31.0 / 25.9, 1024 x 1024 x 32 A^H B 27.0 / 28.5; s 64 x 64 x 2048
// 26.4 / 22.2, 1024 x 1024 x 32 20.4 / 21.3.
bool small_product(int64_t m, int64_t n, int64_t Kp, int scalarBytes) {
  constexpr int64_t kRows = 16, kMostTiles = 2048, kMostWork = int64_t(1) << 18;
  const int64_t tilesM = (m + kRows - 1) / kRows, tilesN = (n + kRows - 1) / kRows;
  if (tilesM > kMostTiles || tilesN > kMostTiles || tilesM * tilesN > kMostTiles) return false;
  return Kp <= 8192 / scalarBytes && tilesM * tilesN * Kp <= kMostWork;
}

}  // namespace

int64_t plan_active_tiles(int64_t m, int64_t n, int rows, int cols, const PlanFill& fill) {
  const int64_t tilesM = (m + rows - 1) / rows, tilesN = (n + cols - 1) / cols;
  if (fill.mode == FillFull) return tilesM * tilesN;
  if (tilesM <= 0 || tilesN <= 0) return 0;
  return FillTiles{fill.mode, fill.colOff - fill.rowOff, m, n, rows, cols, tilesM, tilesN}.total();
}

// Whole-device plans. Every workgroup of a launch computes one tile over one
// split. With one round of resident workgroups a CU has q of them side by side;
// a single one keeps its matrix cores busy to 0.88 (M) or 0.85 (L) of what a full
// CU reaches (700 x 700 x 30011 complex on M tiles: 242 workgroups 1.82 ms, 726
// 1.72 ms). Past that the dispatcher hands workgroups out as slots free up, and a
// last, partial round can land more than once on the same CU (1210 workgroups:
// 2.07 ms), which many short rounds avoid (5808: 1.68 ms; its lower triangle: 924
// workgroups 1.00 ms, 4092 0.95 ms). Workgroups that start together do not end
// together either (1000 x 1000 x 1e5 real on L tiles: 512 workgroups 3.00 ms, 1024
// 2.94 ms). Splitting the reduction costs the write and read of the partial sums and
// a launch.
static GemmPlan plan_tiles(bool complex, int64_t m, int64_t n, int64_t k, int numCUs, int forceCfg,
                           int forceSplits, const double* effByCfg, bool wholeChip,
                           int scalarBytes, const PlanFill& fill) {
  const GemmPlan coarse =
      plan_coarse(complex, m, n, k, numCUs, forceCfg, forceSplits, wholeChip);
  if (!wholeChip || forceCfg >= 0 || forceSplits > 0) return coarse;
  constexpr double kBlockSeconds = 0.6e-6;  // shortest k-block of one workgroup (latency)
  constexpr double kLastRound = 0.03;  // of the last round: workgroups that finish apart
  constexpr double kReduceLaunchSeconds = 4.0e-6;
  const int64_t Mp = complex ? 2 * m : m;
  const int64_t Kp = complex ? 2 * k : k;
  const double sums = static_cast<double>(Mp) * n * scalarBytes;  // bytes of one split
  const bool small = complex && scalarBytes == 8 && fill.mode == FillFull &&
                     (coarse.splits == 1 || coarse.splits * sums <= kSmallWorkspace);
  const double limit = small ? kSmallWorkspace
                       : scalarBytes == 4
                           ? std::max(kLargestWorkspace, coarse.splits * sums + 1)
                           : kLargestWorkspace;
  const double bytes = static_cast<double>(m + n) * k * scalarBytes * (complex ? 2 : 1);
  GemmPlan best = coarse;
  best.small = small_product(m, n, Kp, scalarBytes);
  double bestSeconds = 1e300, fullSeconds = 1e300;
  for (int cfg : {TileL, TileM}) {
    const TileShape ts = tile_shape(cfg);
    const int rows = complex ? ts.bm / 2 : ts.bm;
    const int64_t bk = ts.bk * (scalarBytes == 4 ? 2 : 1);  // a k-block is 128 bytes of a row
    const int64_t tilesM = (m + rows - 1) / rows, tilesN = (n + ts.bn - 1) / ts.bn;
    const int64_t allTiles = tilesM * tilesN;
    const int64_t tiles = std::max<int64_t>(1, plan_active_tiles(m, n, rows, ts.bn, fill));
    // half tiles at the right edge and along the diagonal of a fill mode cost half
    const double share = std::min(
        1.0, 0.5 * plan_active_tiles(m, n, rows, ts.bn / 2, fill) / static_cast<double>(tiles));
    const double needed = static_cast<double>(tiles) / allTiles;  // of C
    const int64_t kBlocks = std::max<int64_t>(1, (Kp + bk - 1) / bk);
    const double peak = kPeakPerCU * (8.0 / scalarBytes) * effByCfg[cfg];
    const double lone = cfg == TileL ? 0.85 : 0.88;
    // address set-up, first loads, epilogue (complex 60000 x 128 x 128: 142 us on M tiles,
    // 164 us on L tiles, which the same time for both preferred)
    const double workgroupSeconds = cfg == TileL ? 10e-6 : 2.5e-6;
    const int64_t maxSplits = std::max<int64_t>(
        1, std::min<int64_t>(kBlocks / scalarBytes,
                             std::max<int64_t>(64, 4 * numCUs * blocks_per_cu(cfg) / tiles)));
    int64_t lastSplits = 0;
    for (int64_t s = 1; s <= maxSplits; s += std::max<int64_t>(1, s / 32)) {
      const int64_t kb = (kBlocks + s - 1) / s;
      const int64_t splits = (kBlocks + kb - 1) / kb;  // no empty split
      if (splits == lastSplits || allTiles * splits > (int64_t(1) << 31) - 1) continue;
      lastSplits = splits;
      if (splits > 1 && splits * sums > limit) break;
      // No longer sums than the coarse plan's, since their rounding errors grow with the
      // length (s 4 x 10 x 309: 1.9e-7 of the result in 2 splits, 2.9e-7 in 1; z 1238 x
      // 1207 x 4119 2.6e-14 root mean square in 28 splits, 1.3e-13 in 1). Double precision
      // has M tiles that add up sums of that length.
      const bool longer = kb * bk >= coarse.kSplit + (scalarBytes == 4 ? bk : 1);
      if (longer && (scalarBytes == 4 || cfg != TileM)) continue;
      const int perCU = longer && !complex ? 3 : blocks_per_cu(cfg);  // gemm_f64_stretch_kernel
      const int64_t slots = static_cast<int64_t>(numCUs) * perCU;
      const double work = 2.0 * ts.bm * ts.bn * bk * kb / peak;  // one workgroup on a full CU
      auto seconds = [&](int64_t groups) {
        const int64_t rounds = groups / slots, rest = groups % slots;
        double t = rounds * perCU * work * share + (rounds > 0 ? (0.7 + 0.3 * rounds) : 0.0) *
                                               workgroupSeconds;
        if (rest > 0) {
          const int64_t spread = (rest + numCUs - 1) / numCUs;
          const int64_t q = rounds > 0 ? std::min<int64_t>(perCU, spread + 1) : spread;
          t += std::max(q * work / (q == 1 ? lone : 1.0), kb * kBlockSeconds) + workgroupSeconds;
        }
        t += kLastRound * work * std::min<double>(perCU, groups / static_cast<double>(numCUs));
        const double inFlight = std::min(1.0, groups / (2.0 * numCUs));
        t = std::max(t, bytes / (kHbmBytesPerSecond * inFlight)) + kLaunchSeconds;
        if (splits > 1)
          t += (1.2 * splits + 2) * sums * needed / kHbmBytesPerSecond + kReduceLaunchSeconds;
        return t;
      };
      const double t = seconds(tiles * splits);
      fullSeconds = std::min(fullSeconds, seconds(allTiles * splits));
      if (t < bestSeconds * 0.999) {
        bestSeconds = t;
        best.cfg = cfg;
        best.splits = static_cast<int>(splits);
        best.kSplit = kb * bk;
        best.kSum = longer ? coarse.kSplit / (2 * bk) * (2 * bk) : 0;
        best.tilesM = static_cast<int>(tilesM);
        best.tilesN = static_cast<int>(tilesN);
      }
    }
  }
  // what the automatic mode compares the split form with: its margin (0.8) was
  // drawn for the coarse model's rates, 0.84 of those reached now
  best.estSeconds = std::min(coarse.estSeconds, fullSeconds / 0.84);
  return best;
}

GemmPlan plan_gemm(bool complex, int64_t m, int64_t n, int64_t k, int numCUs, int forceCfg,
                   int forceSplits, const double* effByCfg, bool wholeChip, int scalarBytes,
                   const PlanFill& fill) {
  GemmPlan p = plan_tiles(complex, m, n, k, numCUs, forceCfg, forceSplits, effByCfg, wholeChip,
                          scalarBytes, fill);
  const TileShape ts = tile_shape(p.cfg);
  p.activeTiles =
      static_cast<int>(plan_active_tiles(m, n, complex ? ts.bm / 2 : ts.bm, ts.bn, fill));
  return p;
}

// Measured on long reductions: 2048 x 2048 x 2e4, complex and real, 74.2-75.6
// TFLOP/s on L tiles and 71.7-72.4 on M tiles.
double Tuner::efficiency(int cfg) { return cfg == TileM ? 0.91 : 0.95; }

GemmPlan Tuner::plan(bool complex, int layoutA, int layoutB, int64_t m, int64_t n, int64_t k,
                     int numCUs, bool wholeChip, int scalarBytes, const PlanFill& fill) {
  const int forceCfg = env_tile();
  const int forceSplits = env_int("SPLA_AMD_SPLITS", 0);
  const Key key{complex, layoutA, layoutB, m, n, k, numCUs, wholeChip, scalarBytes, fill.mode,
                fill.mode == FillFull ? 0 : fill.colOff - fill.rowOff};
  std::lock_guard<std::mutex> guard(lock_);
  if (forceCfg < 0 && forceSplits <= 0) {
    auto it = cache_.find(key);
    if (it != cache_.end()) return it->second;
  }
  double eff[NumTileConfigs];
  for (int c = 0; c < NumTileConfigs; ++c) eff[c] = efficiency(c);
  GemmPlan p = plan_gemm(complex, m, n, k, numCUs, forceCfg, forceSplits, eff, wholeChip, scalarBytes,
                         fill);
  if (forceCfg < 0 && forceSplits <= 0) cache_[key] = p;
  return p;
}

}  // namespace spla_amd
