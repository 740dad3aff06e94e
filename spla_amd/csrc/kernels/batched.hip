// Batched FP64 / complex-FP64 block products of one ring step: one GEMM launch
// over the (block, tile, split) items of every block, then one reduction launch
// over the tiles whose reduction is split, which adds the partial sums in split
// order (bitwise reproducible) and applies alpha / beta. The GEMM launch is
// grouped (one workgroup per item, in decreasing cost order: the dispatcher
// hands them to the CUs as these free up) or persistent (one workgroup per
// resident slot, each working through the static list the host's
// longest-processing-time schedule gave it). Both launches read only
// descriptors and operands; the partial sums are written before they are read
// in every launch, so the pair can be replayed from a hipGraph without clearing
// anything.
//
// ssb blocks (SPLA src/pgemm_ssb/ring_ssb_gpu.cpp:193-197): C_b <- alpha op(A_b) B_b
// + beta C_b with op(A) = A^T / A^H, A k x m (K-major). sbs blocks
// (src/pgemm_sbs/ring_sbs_gpu.cpp:57-88): op(A) = A, A m x k (MN-major).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels/batched_desc.hpp"
#include "kernels/launch.hpp"
#include "kernels/tile_mma.hpp"

namespace spla_amd {
namespace {

using namespace tile;

template <bool CPLX>
__device__ __forceinline__ void update_c(const BatchDesc& d, const BatchBlock& b, int i, int j,
                                         double re, double im) {
  if (CPLX) {
    double* c = b.C + (static_cast<int64_t>(j) * b.ldc + i) * 2;
    double outRe = d.alphaRe * re - d.alphaIm * im;
    double outIm = d.alphaRe * im + d.alphaIm * re;
    if (!d.betaZero) {
      const double cr = c[0], ci = c[1];
      outRe += d.betaRe * cr - d.betaIm * ci;
      outIm += d.betaRe * ci + d.betaIm * cr;
    }
    c[0] = outRe;
    c[1] = outIm;
  } else {
    double* c = b.C + static_cast<int64_t>(j) * b.ldc + i;
    double out = d.alphaRe * re;
    if (!d.betaZero) out += d.betaRe * c[0];
    c[0] = out;
  }
}

// Wave tiles of a configuration (see gemm_f64.hip): R = fragments per 32 embedded rows.
// HALF: half of the columns (tiles of which no more exist, see gemm_tile).
template <bool CPLX, bool CONJ, int LA, int CFG, bool HALF = false, bool WIDE = false>
using BatchMma = TileMma<double, CPLX, CONJ, LA, KMajor, (CPLX ? 1 : 2) * (CFG == TileM ? 1 : 2),
                         (CFG == TileM ? 2 : 4) / (HALF ? 2 : 1), WIDE>;

// One (block, tile, split) item, or tile `part` of the REP x REP tiles of T that cover it; on
// return every thread has passed the tile routine's last barrier, so the LDS
// buffers may be reused at once.
template <typename T, typename H, bool CPLX, int REP = 1>
__device__ __forceinline__ void batched_item(const BatchDesc& d, const BatchItem& it, int part,
                                             void* lds) {
  static_assert(2 * H::BN == T::BN && H::AR == T::AR, "half of the columns");
  const BatchBlock& b = d.blocks[uniform(it.block)];
  const int m = uniform(b.m), n = uniform(b.n), Mp = uniform(b.Mp), s = uniform(it.s);
  const int64_t kSplit = uniform(b.kSplit);
  const int64_t kBegin = s * kSplit;
  const int64_t kEnd = min(uniform(b.Kp), kBegin + kSplit);
  const TileOperands<double> op{uniform(b.A), uniform(b.B), uniform(b.lda), uniform(b.ldb), m, n};
  BatchBlock c;  // what update_c reads
  c.C = uniform(b.C);
  c.ldc = uniform(b.ldc);
  const bool flip = T::flip_result(d.conjA, d.conjB);
  const bool whole = uniform(b.splits) == 1;
  double* w = d.work + uniform(b.workOffset) + static_cast<int64_t>(s) * n * Mp;
  auto run = [&](auto tile, int row, int col) {
    using U = typename decltype(tile)::type;
    typename U::Acc acc;
    U::run(op, row, col, kBegin, kEnd, *static_cast<typename U::Smem*>(lds), acc);
    if (whole) {
      U::for_each(row, col, m, n, flip, acc,
                  [&](int i, int j, double re, double im) { update_c<CPLX>(d, c, i, j, re, im); });
    } else {
      U::for_each(row, col, m, n, flip, acc, [&](int i, int j, double re, double im) {
        store_work<double, CPLX>(w, Mp, i, j, re, im);
      });
    }
  };
  const int row = (uniform(it.tm) * REP + part % REP) * T::AR;
  const int col = (uniform(it.tn) * REP + part / REP) * T::BN;
  if (row >= m || col >= n) return;
  if (n - col <= H::BN)
    run(Type<H>(), row, col);
  else
    run(Type<T>(), row, col);
}

// Grouped launch: workgroup = item (gridDim.x = number of items). LDS for as many workgroups
// per CU as the schedule counts: small complex tiles leave registers for a fifth, which
// starts out of turn on a CU that others should take (128 ragged complex blocks 13.15 ->
// 13.0 ms).
constexpr int kLdsPerCU = 160 << 10;

template <bool CPLX, bool CONJ, int LA, int CFG>
__global__ void __launch_bounds__(kThreads, CFG == TileM ? 4 : 2) batched_gemm_kernel(BatchDesc d) {
  using T = BatchMma<CPLX, CONJ, LA, CFG>;
  using H = BatchMma<CPLX, CONJ, LA, CFG, true>;
  __shared__ union {
    typename T::Smem sm;
    unsigned char room[kLdsPerCU / (CFG == TileM ? 4 : 2)];
  } lds;
  batched_item<T, H, CPLX>(d, d.items[blockIdx.x], 0, &lds);
}

// The grouped launch for blocks with wide rows (tile_wide): every tile as M tiles, a
// workgroup each (BatchKernels::perItem).
constexpr int batch_wide_rep(int cfg) { return cfg == TileM ? 1 : 2; }

template <bool CPLX, bool CONJ, int LA, int CFG>
__global__ void __launch_bounds__(kThreads, 3) batched_gemm_wide_kernel(BatchDesc d) {
  using T = BatchMma<CPLX, CONJ, LA, TileM, false, true>;
  using H = BatchMma<CPLX, CONJ, LA, TileM, true, true>;
  __shared__ typename T::Smem sm;
  constexpr int REP = batch_wide_rep(CFG);
  batched_item<T, H, CPLX, REP>(d, d.items[blockIdx.x / (REP * REP)], blockIdx.x % (REP * REP), &sm);
}

// The persistent launch for blocks with wide rows.
template <bool CPLX, bool CONJ, int LA, int CFG>
__global__ void __launch_bounds__(kThreads, 3) batched_gemm_wide_persistent_kernel(BatchDesc d) {
  using T = BatchMma<CPLX, CONJ, LA, TileM, false, true>;
  using H = BatchMma<CPLX, CONJ, LA, TileM, true, true>;
  __shared__ typename T::Smem sm;
  constexpr int REP = batch_wide_rep(CFG);
  const int end = d.slotStart[blockIdx.x + 1];
  for (int i = d.slotStart[blockIdx.x]; i < end; ++i)
#pragma unroll 1
    for (int part = 0; part < REP * REP; ++part)
      batched_item<T, H, CPLX, REP>(d, d.items[uniform(d.slotItems[i])], part, &sm);
}

// Persistent launch: one workgroup per slot works through its static list of
// items (gridDim.x = number of slots); no workgroup waits for another.
template <bool CPLX, bool CONJ, int LA, int CFG>
__global__ void __launch_bounds__(kThreads, CFG == TileM ? 4 : 2)
    batched_gemm_persistent_kernel(BatchDesc d) {
  using T = BatchMma<CPLX, CONJ, LA, CFG>;
  using H = BatchMma<CPLX, CONJ, LA, CFG, true>;
  __shared__ typename T::Smem sm;
  const int end = d.slotStart[blockIdx.x + 1];
  for (int i = d.slotStart[blockIdx.x]; i < end; ++i)
    batched_item<T, H, CPLX>(d, d.items[uniform(d.slotItems[i])], 0, &sm);
}

// AR x BN: element rows and columns of a tile of the GEMM launch.
template <bool CPLX, int AR, int BN>
__global__ void __launch_bounds__(kThreads) batched_reduce_kernel(BatchDesc d) {
  const BatchReduceTile t = d.reduce[blockIdx.x];
  const BatchBlock b = d.blocks[t.block];
  const int i0 = t.tm * AR;
  const int j0 = t.tn * BN;
  const int rows = min(AR, b.m - i0);
  const int cols = min(BN, b.n - j0);
  const int64_t stride = static_cast<int64_t>(b.n) * b.Mp;
  const double* w0 = d.work + b.workOffset;
  for (int e = threadIdx.x; e < rows * cols; e += kThreads) {
    const int i = i0 + e % rows;
    const int j = j0 + e / rows;
    const double* p = w0 + static_cast<int64_t>(j) * b.Mp + (CPLX ? 2 * i : i);
    double re = 0.0, im = 0.0;
    // bound by the latency of these loads: eight in flight, added in order (20 real blocks
    // with up to 256 splits 1.45 -> 0.62 ms, a batch's products and sums)
#pragma unroll 8
    for (int s = 0; s < b.splits; ++s) {
      re += p[s * stride];
      if (CPLX) im += p[s * stride + 1];
    }
    update_c<CPLX>(d, b, i, j, re, im);
  }
}

template <bool CPLX, bool CONJ, int LA, int CFG>
const void* gemm_kernel_of(BatchDispatch dispatch) {
  switch (dispatch) {
    case BatchPersistent:
      return reinterpret_cast<const void*>(&batched_gemm_persistent_kernel<CPLX, CONJ, LA, CFG>);
    case BatchWide:
      return reinterpret_cast<const void*>(&batched_gemm_wide_kernel<CPLX, CONJ, LA, CFG>);
    case BatchWidePersistent:
      return reinterpret_cast<const void*>(
          &batched_gemm_wide_persistent_kernel<CPLX, CONJ, LA, CFG>);
    default:
      return reinterpret_cast<const void*>(&batched_gemm_kernel<CPLX, CONJ, LA, CFG>);
  }
}

template <bool CPLX, bool CONJ, int LA>
const void* gemm_kernel_for(int cfg, BatchDispatch dispatch) {
  return cfg == TileM ? gemm_kernel_of<CPLX, CONJ, LA, TileM>(dispatch)
                      : gemm_kernel_of<CPLX, CONJ, LA, TileL>(dispatch);
}

}  // namespace

BatchKernels batched_kernels(bool complex, bool conjA, int layoutA, int cfg,
                             BatchDispatch dispatch) {
  BatchKernels k;
  if (complex) {
    k.gemm = layoutA == MNMajor ? gemm_kernel_for<true, false, MNMajor>(cfg, dispatch)
             : conjA            ? gemm_kernel_for<true, true, KMajor>(cfg, dispatch)
                                : gemm_kernel_for<true, false, KMajor>(cfg, dispatch);
    k.reduce = cfg == TileM ? reinterpret_cast<const void*>(&batched_reduce_kernel<true, 32, 64>)
                            : reinterpret_cast<const void*>(&batched_reduce_kernel<true, 64, 128>);
  } else {
    k.gemm = layoutA == MNMajor ? gemm_kernel_for<false, false, MNMajor>(cfg, dispatch)
                                : gemm_kernel_for<false, false, KMajor>(cfg, dispatch);
    k.reduce = cfg == TileM ? reinterpret_cast<const void*>(&batched_reduce_kernel<false, 64, 64>)
                            : reinterpret_cast<const void*>(&batched_reduce_kernel<false, 128, 128>);
  }
  k.threads = kThreads;
  k.perItem = dispatch == BatchWide ? batch_wide_rep(cfg) * batch_wide_rep(cfg) : 1;
  return k;
}

}  // namespace spla_amd
