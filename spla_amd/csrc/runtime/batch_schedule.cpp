#include "runtime/batch_schedule.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

#include "kernels/gemm_desc.hpp"
#include "spla/types.h"

namespace spla_amd {
namespace {

constexpr double kPeakPerCU = 128.0 * 2.4e9;  // FP64 matrix flop / s per CU
constexpr double kItemOverhead = 2.0e-6;      // prologue + epilogue per workgroup
constexpr double kLaunchOverhead = 8.0e-6;    // per launch in the graph
constexpr double kReduceBytesPerSecond = 4.0e12;
// A thread of the reduction adds the partial sums of its elements one after the other, with
// eight loads in flight (20 real blocks up to 512 x 512 x 65536 on small tiles: 0.49, 0.53,
// 0.62 and 0.74 ms with up to 64, 128, 256 and 256 splits, of which the products take 0.3
// ms; 0.68, 0.94, 1.45 and 1.90 ms with one load after the other).
constexpr double kReduceLoadSeconds = 0.07e-6;
constexpr int kReduceThreads = 256;
constexpr int kMinKBlocksPerSplit = 16;

int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

}  // namespace

int batch_blocks_per_cu(int cfg) { return cfg == TileM ? 4 : 2; }

int batch_slots(int cfg, int numCUs, std::size_t items) {
  const std::size_t slots = static_cast<std::size_t>(std::max(1, numCUs)) * batch_blocks_per_cu(cfg);
  return static_cast<int>(std::max<std::size_t>(1, std::min(slots, items)));
}

bool batch_tile_active(int fillMode, int64_t rowOff, int64_t colOff, int64_t r, int64_t c,
                       int64_t nr, int64_t nc) {
  if (fillMode == SPLA_FILL_MODE_UPPER) return c + nc + colOff > r + rowOff;
  if (fillMode == SPLA_FILL_MODE_LOWER) return r + nr + rowOff > c + colOff;
  return true;
}

BatchSchedule plan_batch_schedule(const std::vector<BatchShape>& shapes, bool complex,
                                  bool alphaZero, int cfg, double splitScale, int numCUs,
                                  double efficiency) {
  BatchSchedule out;
  out.cfg = cfg;
  out.splitScale = splitScale;
  const TileShape ts = tile_shape(cfg);
  const int comps = complex ? 2 : 1;
  const int ar = ts.bm / comps;  // element rows per tile
  const int perCU = batch_blocks_per_cu(cfg);
  const int slots = std::max(1, numCUs) * perCU;
  const double slotRate = kPeakPerCU * efficiency / perCU;

  struct Tile {
    int block, tm, tn;
    double share;  // of the tile's cost: a half for the half tiles of batched.hip
  };
  std::vector<Tile> tiles;
  std::vector<double> tileCost(shapes.size(), 0.0);
  double total = 0.0;
  for (std::size_t b = 0; b < shapes.size(); ++b) {
    const BatchShape& s = shapes[b];
    if (s.m <= 0 || s.n <= 0) continue;
    const int64_t Kp = alphaZero ? 0 : s.k * comps;
    tileCost[b] = 2.0 * ts.bm * ts.bn * static_cast<double>(std::max<int64_t>(Kp, ts.bk)) /
                  slotRate;
    const int64_t tilesM = ceil_div(s.m, ar), tilesN = ceil_div(s.n, ts.bn);
    for (int64_t tn = 0; tn < tilesN; ++tn)
      for (int64_t tm = 0; tm < tilesM; ++tm) {
        const int64_t r = tm * ar, c = tn * ts.bn;
        if (!batch_tile_active(s.fillMode, s.rowOff, s.colOff, r, c, std::min<int64_t>(ar, s.m - r),
                               std::min<int64_t>(ts.bn, s.n - c)))
          continue;
        const double share = s.n - c <= ts.bn / 2 ? 0.5 : 1.0;
        tiles.push_back({static_cast<int>(b), static_cast<int>(tm), static_cast<int>(tn), share});
        total += share * tileCost[b];
      }
  }
  const double target = std::max(total / (3.0 * slots), 20e-6);

  out.blocks.resize(shapes.size());
  for (std::size_t b = 0; b < shapes.size(); ++b) {
    const BatchShape& s = shapes[b];
    BatchBlock& bb = out.blocks[b];
    std::memset(&bb, 0, sizeof(bb));
    if (s.m <= 0 || s.n <= 0) continue;
    const int64_t Kp = alphaZero ? 0 : s.k * comps;
    const int64_t kBlocks = ceil_div(Kp, ts.bk);
    int64_t sp = static_cast<int64_t>(std::ceil(tileCost[b] * splitScale / target - 1e-6));
    sp = std::max<int64_t>(1, std::min<int64_t>(sp, std::max<int64_t>(1, kBlocks /
                                                                       kMinKBlocksPerSplit)));
    const int64_t kbPer = kBlocks > 0 ? ceil_div(kBlocks, sp) : 1;
    sp = kBlocks > 0 ? ceil_div(kBlocks, kbPer) : 1;  // no empty split
    bb.m = static_cast<int>(s.m);
    bb.n = static_cast<int>(s.n);
    bb.Kp = Kp;
    bb.Mp = static_cast<int>(s.m * comps);
    bb.splits = static_cast<int>(sp);
    bb.kSplit = kbPer * ts.bk;
    if (sp > 1) {
      bb.workOffset = out.workDoubles;
      out.workDoubles += sp * s.n * bb.Mp;
    }
  }

  // items in decreasing cost order: the splits of a tile cost the same, so the tiles are
  // ordered and their splits follow each other
  struct Costed {
    BatchItem item;
    double cost;
  };
  std::vector<std::pair<double, int>> order(tiles.size());  // (cost of a split, tile)
  std::size_t count = 0;
  double reduceSeconds = 0.0;
  int mostSplits = 0;
  for (std::size_t i = 0; i < tiles.size(); ++i) {
    const Tile& t = tiles[i];
    const BatchBlock& bb = out.blocks[t.block];
    order[i] = {t.share * tileCost[t.block] / bb.splits + kItemOverhead, static_cast<int>(i)};
    count += bb.splits;
    if (bb.splits > 1) {
      out.reduce.push_back({t.block, t.tm, t.tn});
      mostSplits = std::max(mostSplits, bb.splits);
      reduceSeconds +=
          (bb.splits + 2.0) * ar * ts.bn * 8.0 * comps / kReduceBytesPerSecond;
    }
  }
  std::stable_sort(order.begin(), order.end(),
                   [](const auto& a, const auto& b) { return a.first > b.first; });
  std::vector<Costed> items;
  items.reserve(count);
  for (const auto& o : order) {
    const Tile& t = tiles[o.second];
    for (int q = 0; q < out.blocks[t.block].splits; ++q)
      items.push_back({{t.block, t.tm, t.tn, q}, o.first});
  }
  out.items.reserve(items.size());
  // longest processing time first: each item goes to the slot that frees up
  // first (ties: the lowest slot), which is also the persistent launch's schedule
  const int nSlots = batch_slots(cfg, numCUs, items.size());
  using Slot = std::pair<double, int>;  // (load, slot)
  std::vector<Slot> load(nSlots);  // a heap, the least load first
  for (int i = 0; i < nSlots; ++i) load[i] = {0.0, i};
  std::vector<int> slotOf(items.size());
  out.slotStart.assign(nSlots + 1, 0);
  double makespan = 0.0;
  for (std::size_t i = 0; i < items.size(); ++i) {
    out.items.push_back(items[i].item);
    Slot sl = load[0];
    sl.first += items[i].cost;
    makespan = std::max(makespan, sl.first);
    slotOf[i] = sl.second;
    ++out.slotStart[sl.second + 1];
    int at = 0;  // the slot sinks to its new place
    for (int child = 1; child < nSlots; child = 2 * at + 1) {
      if (child + 1 < nSlots && load[child + 1] < load[child]) ++child;
      if (!(load[child] < sl)) break;
      load[at] = load[child];
      at = child;
    }
    load[at] = sl;
  }
  for (int w = 0; w < nSlots; ++w) out.slotStart[w + 1] += out.slotStart[w];
  out.slotItems.resize(items.size());
  std::vector<int> next(out.slotStart.begin(), out.slotStart.end() - 1);
  for (std::size_t i = 0; i < items.size(); ++i)
    out.slotItems[next[slotOf[i]]++] = static_cast<int>(i);
  reduceSeconds = std::max(reduceSeconds, static_cast<double>(mostSplits) *
                                              (ar * ts.bn / kReduceThreads) * kReduceLoadSeconds);
  out.modelSeconds = makespan + reduceSeconds + kLaunchOverhead * (out.reduce.empty() ? 1 : 2);
  return out;
}

}  // namespace spla_amd
