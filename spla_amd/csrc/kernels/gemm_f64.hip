// FP64 / complex-FP64 GEMM on the gfx950 FP64 matrix cores (v_mfma_f64_16x16x4_f64),
// and the same kernels in FP32 / complex-FP32 on the FP32 matrix cores
// (v_mfma_f32_16x16x4_f32, FP32 accumulation as in a single-precision BLAS).
//
// Replaces the vendor ?gemm call of SPLA's local engine
// (src/gpu_util/multiply_gpu.cpp:40-76 -> rocblas_{d,z}gemm) for the
// operations the engine issues: opA in {N, T, C}, opB in {N, T, C}.
//
// Structure of one workgroup (256 threads = 4 wave64):
//   * a tile of the output (sizes in embedded rows, see gemm_desc.hpp), split
//     over a 2 x 2 grid of waves; the k loop is that of tile_mma.hpp;
//   * split-K: a split writes its raw partial sums to a workspace; the
//     reduction kernel adds the splits in a fixed order (bitwise
//     reproducible) and applies alpha / beta. With one split the epilogue is
//     fused.
//   * workgroup -> tile mapping is XCD aware: consecutive workgroups are
//     dispatched round-robin over the 8 XCDs, so the index is remapped such
//     that each XCD works on a compact group of tiles that share A and B
//     panels in its L2.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels/fill_tiles.hpp"
#include "kernels/gemm_desc.hpp"
#include "kernels/gemm_epilogue.hpp"
#include "kernels/launch.hpp"
#include "kernels/tile_mma.hpp"

namespace spla_amd {
namespace {

using namespace tile;

// Maps workgroup `bid` of G to (split, tile row, tile column) over the active tiles of
// rows x cols. Only these are launched: workgroups that leave at once let the
// dispatcher pile others onto their CUs (700 x 700 x 30011 complex, lower triangle, 924
// workgroups, 3.6 per CU: 1.00 ms, with 770 empty ones among them 1.02 to 1.25 ms).
// `parts` workgroups share a tile, `part` is this one's.
__device__ __forceinline__ void map_block(const GemmDesc& d, int bid, int G, int rows, int cols,
                                          int parts, int& s, int& tm, int& tn, int& part) {
  int lin = bid;
  if ((G & 7) == 0) lin = (bid & 7) * (G >> 3) + (bid >> 3);
  part = lin % parts;
  lin /= parts;
  s = lin / d.activeTiles;
  const int t = lin - s * d.activeTiles;
  if (d.fillMode != FillFull) {  // tile by tile down the columns
    const FillTiles tiles{d.fillMode, d.fillColOff - d.fillRowOff, d.m, d.n, rows, cols,
                          d.tilesM, d.tilesN};
    tiles.locate(t, tm, tn);
    return;
  }
  constexpr int kGroup = 8;
  const int group = t / (kGroup * d.tilesN);
  const int firstM = group * kGroup;
  const int gsize = min(d.tilesM - firstM, kGroup);
  const int inGroup = t - group * kGroup * d.tilesN;
  tm = firstM + inGroup % gsize;
  tn = inGroup / gsize;
}

// Body of one workgroup (shared by the FP64 and FP32 kernels). A tile of the grid is one
// of T (Whole), or repM x repN of them, one after the other (Loop) or a workgroup each
// (Part). A tile of which at most half the columns exist, or (Whole) lie in active half
// tiles of a fill mode, runs as the half tile H: the matrix cores are what bounds the kernel, so the other half is not
// computed (real 100003 x 260 x 260 341 -> 326 us, a batch of 128 ragged complex blocks 14.1
// -> 13.7 ms).
// STRETCHES: see TileMma::run.
enum TileWork : int { Whole, Loop, Part };
template <typename T, typename H, typename S, bool CPLX, TileWork WORK, bool STRETCHES = false>
__device__ __forceinline__ void gemm_tile(const GemmDesc& d, int repM, int repN, void* lds) {
  static_assert(2 * H::BN == T::BN && H::AR == T::AR, "half of the columns");
  if (WORK == Whole) repM = repN = 1;
  const int bid = WORK == Part ? blockIdx.y * gridDim.x + blockIdx.x : blockIdx.x;
  const int G = WORK == Part ? gridDim.x * gridDim.y : gridDim.x;
  int s, tm, tn, part;
  map_block(d, bid, G, T::AR * repM, T::BN * repN, WORK == Part ? repM * repN : 1, s, tm, tn, part);
  s = uniform(s);
  tm = uniform(tm);
  tn = uniform(tn);
  part = uniform(part);
  const int first = tm * T::AR * repM;
  const int col0 = tn * T::BN * repN;
  bool left = true, right = true;  // half tiles that are needed
  if (d.fillMode != FillFull) {
    const int64_t nr = min(T::AR * repM, d.m - first);
    const int64_t nc = min(T::BN * repN, d.n - col0);
    if (WORK == Whole && nc > H::BN) {
      left = tile_active(d, first, col0, nr, H::BN);
      right = tile_active(d, first, col0 + H::BN, nr, nc - H::BN);
    }
  }
  const int64_t kBegin = static_cast<int64_t>(s) * d.kSplit;
  const int64_t kEnd = min(d.Kp, kBegin + d.kSplit);
  const TileOperands<S> op{uniform(static_cast<const S*>(d.A)), uniform(static_cast<const S*>(d.B)),
                           uniform(d.lda), uniform(d.ldb), uniform(d.m), uniform(d.n)};
  const bool flip = T::flip_result(d.conjA, d.conjB);
  S* w = static_cast<S*>(d.work) + static_cast<int64_t>(s) * d.n * d.Mp;
  constexpr int kBlock = kBlockBytes / sizeof(S);  // embedded
  const int stretch = d.kSum > 0 ? static_cast<int>(d.kSum / kBlock) : 1 << 30;
  auto run = [&](auto tile, int row, int col) {
    using U = typename decltype(tile)::type;
    typename U::Acc acc;
    U::template run<STRETCHES>(op, row, col, kBegin, kEnd, *static_cast<typename U::Smem*>(lds),
                               acc, stretch);
    if (d.splits > 1) {
      U::for_each(row, col, d.m, d.n, flip, acc,
                  [&](int i, int j, S re, S im) { store_work<S, CPLX>(w, d.Mp, i, j, re, im); });
    } else if (d.betaZero) {
      U::for_each(row, col, d.m, d.n, flip, acc, [&](int i, int j, S re, S im) {
        store_update<S, CPLX>(d, i, j, re, im, S(0), S(0));
      });
    } else {
      U::for_each_update(row, col, d.m, d.n, flip, acc, static_cast<const S*>(d.C), d.ldc,
                         [&](int i, int j, S re, S im, S cr, S ci) {
                           store_update<S, CPLX>(d, i, j, re, im, cr, ci);
                         });
    }
  };
  auto one = [&](int row, int col) {
    row = uniform(row);
    col = uniform(left ? col : col + H::BN);
    if (uniform(static_cast<int>(!(left && right) || d.n - col <= H::BN)))
      run(Type<H>(), row, col);
    else
      run(Type<T>(), row, col);
  };
  if constexpr (WORK == Whole) {
    one(first, col0);
  } else {
#pragma unroll 1
    for (int t = part; t < (WORK == Part ? part + 1 : repM * repN); ++t) {
      const int row = first + (t % repM) * T::AR, col = col0 + (t / repM) * T::BN;
      if (row < d.m && col < d.n) one(row, col);
    }
  }
}

template <bool CPLX, bool CONJ, int LA, int LB, int FM, int FN, int MINBLOCKS>
__global__ void __launch_bounds__(kThreads, MINBLOCKS) gemm_f64_kernel(GemmDesc d) {
  using T = TileMma<double, CPLX, CONJ, LA, LB, FM, FN>;
  using H = TileMma<double, CPLX, CONJ, LA, LB, FM, FN / 2>;
  __shared__ typename T::Smem sm;
  gemm_tile<T, H, double, CPLX, Whole>(d, 1, 1, &sm);
}

// M tiles that add their sums up in stretches (GemmDesc::kSum), so that a product needs
// neither longer sums nor the memory traffic of more splits: complex 1238 x 1207 x 4119
// 0.73 ms and 2.6e-14 root mean square error in one split; one long sum has 0.72 ms and
// 1.3e-13, 28 splits on L tiles 1.09 ms and 2.6e-14. The totals fit beside the four
// workgroups per CU of complex tiles; real ones have registers for three (1601 x 1190 x
// 20905 1.28 ms either way).
template <bool CPLX, bool CONJ, int LA, int LB, int FM, int FN>
__global__ void __launch_bounds__(kThreads, CPLX ? 4 : 3) gemm_f64_stretch_kernel(GemmDesc d) {
  using T = TileMma<double, CPLX, CONJ, LA, LB, FM, FN>;
  using H = TileMma<double, CPLX, CONJ, LA, LB, FM, FN / 2>;
  __shared__ typename T::Smem sm;
  gemm_tile<T, H, double, CPLX, Whole, true>(d, 1, 1, &sm);
}

// Tiles of repM x repN of the kernel's own (see launch_layout).
template <bool CPLX, bool CONJ, int LA, int LB, int FM, int FN>
__global__ void __launch_bounds__(kThreads, 2) gemm_f64_multi_kernel(GemmDesc d, int repM, int repN) {
  using T = TileMma<double, CPLX, CONJ, LA, LB, FM, FN>;
  using H = TileMma<double, CPLX, CONJ, LA, LB, FM, FN / 2>;
  __shared__ typename T::Smem sm;
  gemm_tile<T, H, double, CPLX, Loop>(d, repM, repN, &sm);
}

// The same with a workgroup for each of them, operands with wide rows (tile_wide).
template <bool CPLX, bool CONJ, int LA, int LB, int FM, int FN>
__global__ void __launch_bounds__(kThreads, 3) gemm_f64_wide_kernel(GemmDesc d, int repM, int repN) {
  using T = TileMma<double, CPLX, CONJ, LA, LB, FM, FN, true>;
  using H = TileMma<double, CPLX, CONJ, LA, LB, FM, FN / 2, true>;
  __shared__ typename T::Smem sm;
  gemm_tile<T, H, double, CPLX, Part, true>(d, repM, repN, &sm);
}

template <bool CPLX, bool CONJ, int LA, int LB, int FM, int FN, int MINBLOCKS>
__global__ void __launch_bounds__(kThreads, MINBLOCKS) gemm_f32_kernel(GemmDesc d) {
  using T = TileMma<float, CPLX, CONJ, LA, LB, FM, FN>;
  using H = TileMma<float, CPLX, CONJ, LA, LB, FM, FN / 2>;
  __shared__ typename T::Smem sm;
  gemm_tile<T, H, float, CPLX, Whole>(d, 1, 1, &sm);
}

// Tiles of repM x repN of the kernel's own (see launch_layout).
template <bool CPLX, bool CONJ, int LA, int LB, int FM, int FN>
__global__ void __launch_bounds__(kThreads, 2) gemm_f32_multi_kernel(GemmDesc d, int repM, int repN) {
  using T = TileMma<float, CPLX, CONJ, LA, LB, FM, FN>;
  using H = TileMma<float, CPLX, CONJ, LA, LB, FM, FN / 2>;
  __shared__ typename T::Smem sm;
  gemm_tile<T, H, float, CPLX, Loop>(d, repM, repN, &sm);
}

// The same with a workgroup for each of them, operands with wide rows (tile_wide).
template <bool CPLX, bool CONJ, int LA, int LB, int FM, int FN>
__global__ void __launch_bounds__(kThreads, 3) gemm_f32_wide_kernel(GemmDesc d, int repM, int repN) {
  using T = TileMma<float, CPLX, CONJ, LA, LB, FM, FN, true>;
  using H = TileMma<float, CPLX, CONJ, LA, LB, FM, FN / 2, true>;
  __shared__ typename T::Smem sm;
  gemm_tile<T, H, float, CPLX, Part>(d, repM, repN, &sm);
}

// Adds the split-K partial sums in split order and applies alpha / beta.
template <typename S, bool CPLX>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(GemmDesc d, int tileRows,
                                                            int tileCols) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t total = static_cast<int64_t>(d.m) * d.n;
  if (idx >= total) return;
  const int i = static_cast<int>(idx % d.m);
  const int j = static_cast<int>(idx / d.m);
  if (d.fillMode != FillFull) {
    const int64_t r0 = (i / tileRows) * static_cast<int64_t>(tileRows);
    const int64_t c0 = (j / tileCols) * static_cast<int64_t>(tileCols);
    const int64_t nr = min<int64_t>(tileRows, d.m - r0);
    const int64_t nc = min<int64_t>(tileCols, d.n - c0);
    if (!tile_active(d, r0, c0, nr, nc)) return;
  }
  S re = S(0), im = S(0);
  const int64_t stride = static_cast<int64_t>(d.n) * d.Mp;
  if (CPLX) {
    const S* w = static_cast<const S*>(d.work) + static_cast<int64_t>(j) * d.Mp + 2 * i;
    for (int s = 0; s < d.splits; ++s) {
      re += w[s * stride];
      im += w[s * stride + 1];
    }
  } else {
    const S* w = static_cast<const S*>(d.work) + static_cast<int64_t>(j) * d.Mp + i;
    for (int s = 0; s < d.splits; ++s) re += w[s * stride];
  }
  store_result<S, CPLX>(d, i, j, re, im);
}

// Many splits over few elements (small m, n, long reduction): ELEMS elements per
// block, 256 / ELEMS split groups per element. Group g sums splits g, g + groups,
// ... in order and the group sums are added pairwise, so the result is bitwise
// reproducible. Bound by latency: with 16 elements per block the 256 sums of a 16 x
// 16 product over 1024 splits ran in 16 blocks of 64 loads after each other (30
// us); four take 64 blocks of 8 loads over its 512 splits now (4.4 us).
template <typename S, bool CPLX, int ELEMS>
__global__ void __launch_bounds__(256) splitk_reduce_wide_kernel(GemmDesc d, int tileRows,
                                                                 int tileCols) {
  constexpr int kGroups = 256 / ELEMS;
  __shared__ S part[kGroups][ELEMS][2];
  const int e = threadIdx.x % ELEMS;
  const int g = threadIdx.x / ELEMS;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * ELEMS + e;
  const int64_t total = static_cast<int64_t>(d.m) * d.n;
  bool live = idx < total;
  const int i = live ? static_cast<int>(idx % d.m) : 0;
  const int j = live ? static_cast<int>(idx / d.m) : 0;
  if (live && d.fillMode != FillFull) {
    const int64_t r0 = (i / tileRows) * static_cast<int64_t>(tileRows);
    const int64_t c0 = (j / tileCols) * static_cast<int64_t>(tileCols);
    const int64_t nr = min<int64_t>(tileRows, d.m - r0);
    const int64_t nc = min<int64_t>(tileCols, d.n - c0);
    live = tile_active(d, r0, c0, nr, nc);
  }
  S re = S(0), im = S(0);
  if (live) {
    const int64_t stride = static_cast<int64_t>(d.n) * d.Mp;
    const S* w = static_cast<const S*>(d.work) + static_cast<int64_t>(j) * d.Mp + (CPLX ? 2 * i : i);
#pragma unroll 8
    for (int sp = g; sp < d.splits; sp += kGroups) {
      re += w[sp * stride];
      if (CPLX) im += w[sp * stride + 1];
    }
  }
  part[g][e][0] = re;
  part[g][e][1] = im;
  for (int half = kGroups / 2; half > 0; half /= 2) {
    __syncthreads();
    if (g < half) {
      part[g][e][0] += part[g + half][e][0];
      if (CPLX) part[g][e][1] += part[g + half][e][1];
    }
  }
  if (g == 0 && live) store_result<S, CPLX>(d, i, j, part[0][e][0], part[0][e][1]);
}

// C <- beta * C (k == 0 or alpha == 0); beta == 0 writes zeros without reading C.
template <typename S, bool CPLX>
__global__ void __launch_bounds__(256) scale_kernel(GemmDesc d) {
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t total = static_cast<int64_t>(d.m) * d.n;
  if (idx >= total) return;
  const int i = static_cast<int>(idx % d.m);
  const int j = static_cast<int>(idx / d.m);
  const S bRe = static_cast<S>(d.betaRe), bIm = static_cast<S>(d.betaIm);
  if (CPLX) {
    S* c = static_cast<S*>(d.C) + (static_cast<int64_t>(j) * d.ldc + i) * 2;
    if (d.betaZero) {
      c[0] = S(0);
      c[1] = S(0);
    } else {
      const S cr = c[0], ci = c[1];
      c[0] = bRe * cr - bIm * ci;
      c[1] = bRe * ci + bIm * cr;
    }
  } else {
    S* c = static_cast<S*>(d.C) + static_cast<int64_t>(j) * d.ldc + i;
    c[0] = d.betaZero ? S(0) : bRe * c[0];
  }
}

// Wave tiles: L 64 x 64 embedded rows and columns (two workgroups per CU), M
// 32 x 32 (four); XL is two L tiles one after the other (128 x 64 wave tiles, one
// wave per SIMD, keep the compiler moving accumulators between register files).
// Operands with wide rows (tile_wide) run every shape as M tiles, a workgroup each.
template <bool F32, bool CPLX, bool CONJ, int LA, int LB>
hipError_t launch_layout(const GemmDesc& d, int cfg, hipStream_t stream) {
  constexpr int R = CPLX ? 1 : 2;  // fragments per 32 embedded rows
  const dim3 block(kThreads);
  const dim3 grid(static_cast<unsigned>(d.activeTiles * d.splits));
  const int elem = (F32 ? 4 : 8) * (CPLX ? 2 : 1);
  if (tile_wide(d.lda, elem) || tile_wide(d.ldb, elem)) {
    const TileShape ts = tile_shape(cfg), tm = tile_shape(TileM);
    const int repM = ts.bm / tm.bm, repN = ts.bn / tm.bn;
    const dim3 wide(grid.x, repM * repN);  // two counts: threads along x fit 32 bits
    if constexpr (F32)
      hipLaunchKernelGGL((gemm_f32_wide_kernel<CPLX, CONJ, LA, LB, R, 2>), wide, block, 0, stream,
                         d, repM, repN);
    else
      hipLaunchKernelGGL((gemm_f64_wide_kernel<CPLX, CONJ, LA, LB, R, 2>), wide, block, 0, stream,
                         d, repM, repN);
    return hipGetLastError();
  }
  if constexpr (F32) {
    switch (cfg) {
      case TileM:
        hipLaunchKernelGGL((gemm_f32_kernel<CPLX, CONJ, LA, LB, R, 2, 4>), grid, block, 0, stream,
                           d);
        break;
      case TileXL:
        hipLaunchKernelGGL((gemm_f32_multi_kernel<CPLX, CONJ, LA, LB, 2 * R, 4>), grid,
                           block, 0, stream, d, 2, 1);
        break;
      default:
        hipLaunchKernelGGL((gemm_f32_kernel<CPLX, CONJ, LA, LB, 2 * R, 4, 2>), grid, block, 0,
                           stream, d);
        break;
    }
  } else {
    switch (cfg) {
      case TileM:
        if (d.kSum > 0)
          hipLaunchKernelGGL((gemm_f64_stretch_kernel<CPLX, CONJ, LA, LB, R, 2>), grid, block, 0,
                             stream, d);
        else
          hipLaunchKernelGGL((gemm_f64_kernel<CPLX, CONJ, LA, LB, R, 2, 4>), grid, block, 0,
                             stream, d);
        break;
      case TileXL:
        hipLaunchKernelGGL((gemm_f64_multi_kernel<CPLX, CONJ, LA, LB, 2 * R, 4>), grid,
                           block, 0, stream, d, 2, 1);
        break;
      default:
        hipLaunchKernelGGL((gemm_f64_kernel<CPLX, CONJ, LA, LB, 2 * R, 4, 2>), grid, block, 0,
                           stream, d);
        break;
    }
  }
  return hipGetLastError();
}

// A is conjugated only as A^H (K-major), B only as B^H (MN-major): MN-major A
// times K-major B is never conjugated.
template <bool F32, bool CPLX, int LA, int LB>
hipError_t launch_conj(const GemmDesc& d, int cfg, hipStream_t stream) {
  if constexpr (CPLX && !(LA == MNMajor && LB == KMajor)) {
    if ((d.conjA != 0) != (d.conjB != 0))
      return launch_layout<F32, CPLX, true, LA, LB>(d, cfg, stream);
  } else {
    if (d.conjA || d.conjB) return hipErrorInvalidValue;
  }
  return launch_layout<F32, CPLX, false, LA, LB>(d, cfg, stream);
}

template <bool F32, bool CPLX>
hipError_t launch_typed(const GemmDesc& d, int la, int lb, int cfg, hipStream_t stream) {
  if (la == KMajor && lb == KMajor) return launch_conj<F32, CPLX, KMajor, KMajor>(d, cfg, stream);
  if (la == KMajor && lb == MNMajor)
    return launch_conj<F32, CPLX, KMajor, MNMajor>(d, cfg, stream);
  if (la == MNMajor && lb == KMajor)
    return launch_conj<F32, CPLX, MNMajor, KMajor>(d, cfg, stream);
  return launch_conj<F32, CPLX, MNMajor, MNMajor>(d, cfg, stream);
}

}  // namespace

hipError_t launch_gemm_f64(const GemmDesc& d, bool complex, int layoutA, int layoutB, int cfg,
                           hipStream_t stream) {
  return complex ? launch_typed<false, true>(d, layoutA, layoutB, cfg, stream)
                 : launch_typed<false, false>(d, layoutA, layoutB, cfg, stream);
}

hipError_t launch_gemm_f32(const GemmDesc& d, bool complex, int layoutA, int layoutB, int cfg,
                           hipStream_t stream) {
  return complex ? launch_typed<true, true>(d, layoutA, layoutB, cfg, stream)
                 : launch_typed<true, false>(d, layoutA, layoutB, cfg, stream);
}

template <typename S>
hipError_t launch_splitk_reduce_s(const GemmDesc& d, bool complex, int cfg, hipStream_t stream) {
  // fill modes are decided per half tile (gemm_tile)
  const TileShape ts = tile_shape(cfg);
  const int tileRows = complex ? ts.bm / 2 : ts.bm, tileCols = ts.bn / 2;
  const int64_t total = static_cast<int64_t>(d.m) * d.n;
  // One element per thread fills the chip from 16384 elements on; below, up to
  // 16 splits after each other still cost less than the group sums.
  if (d.splits > 64 || (d.splits > 16 && total < 16384)) {
    const bool few = total <= 4096;
    const int elems = few ? 4 : 16;
    const dim3 wide(static_cast<unsigned>((total + elems - 1) / elems));
    auto* kernel = complex ? (few ? splitk_reduce_wide_kernel<S, true, 4>
                                  : splitk_reduce_wide_kernel<S, true, 16>)
                           : (few ? splitk_reduce_wide_kernel<S, false, 4>
                                  : splitk_reduce_wide_kernel<S, false, 16>);
    hipLaunchKernelGGL(kernel, wide, dim3(256), 0, stream, d, tileRows, tileCols);
    return hipGetLastError();
  }
  const dim3 grid(static_cast<unsigned>((total + 255) / 256));
  if (complex)
    hipLaunchKernelGGL((splitk_reduce_kernel<S, true>), grid, dim3(256), 0, stream, d, tileRows,
                       tileCols);
  else
    hipLaunchKernelGGL((splitk_reduce_kernel<S, false>), grid, dim3(256), 0, stream, d, tileRows,
                       tileCols);
  return hipGetLastError();
}

hipError_t launch_splitk_reduce(const GemmDesc& d, bool complex, int cfg, hipStream_t stream,
                                bool f32) {
  return f32 ? launch_splitk_reduce_s<float>(d, complex, cfg, stream)
             : launch_splitk_reduce_s<double>(d, complex, cfg, stream);
}

hipError_t launch_scale(const GemmDesc& d, bool complex, hipStream_t stream, bool f32) {
  const int64_t total = static_cast<int64_t>(d.m) * d.n;
  if (total == 0) return hipSuccess;
  const dim3 grid(static_cast<unsigned>((total + 255) / 256));
  if (f32) {
    if (complex)
      hipLaunchKernelGGL((scale_kernel<float, true>), grid, dim3(256), 0, stream, d);
    else
      hipLaunchKernelGGL((scale_kernel<float, false>), grid, dim3(256), 0, stream, d);
  } else {
    if (complex)
      hipLaunchKernelGGL((scale_kernel<double, true>), grid, dim3(256), 0, stream, d);
    else
      hipLaunchKernelGGL((scale_kernel<double, false>), grid, dim3(256), 0, stream, d);
  }
  return hipGetLastError();
}

}  // namespace spla_amd
