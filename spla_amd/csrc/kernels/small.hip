// Products too small for the tile kernels (gemm_f64.hip), FP64 and FP32, real and
// complex, every operand layout: one launch, no workspace.
//
// What bounds them: latency. A tile of the tile kernels walks the reduction one
// k-block after the other, and splitting it costs a second launch (d 13 x 32 x 263:
// 9.8 us for 2 splits of 9 k-blocks, 4.1 us for their sum). Here a workgroup owns 16 x
// 16 elements of C and its waves share the reduction: every wave has all loads of
// 32 reduction indices in flight, straight from memory into the operand registers, and
// the waves' sums are added in wave order in LDS. d 13 x 32 x 263: 24.6 -> 17.2 us a
// call, of which launching and waiting for any kernel take 15.6.
//
// Operands: a 16-byte piece per lane and step. K-major: E neighbouring reduction
// indices of row l16 (E = 16 bytes / element); MN-major: E single elements. Step s of
// a wave covers reduction indices 4 E s + E kk + e. Rows past the operand's last one
// read that one and feed outputs that are not stored; reduction indices past the end
// read the last one and are zeroed in both operands. MFMA operand order and
// accumulator layout as in tile_mma.hpp.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels/gemm_desc.hpp"
#include "kernels/gemm_epilogue.hpp"
#include "kernels/launch.hpp"
#include "kernels/tile_mma.hpp"

namespace spla_amd {
namespace {

using namespace tile;

constexpr int kTile = 16;
constexpr int kGroup = 32;  // reduction indices whose loads a wave has in flight together
constexpr int kMaxWaves = 16;

// One operand's rows of a tile as a lane sees them.
template <typename S, bool CPLX, int LAYOUT>
struct SmallOperand {
  static constexpr int kComps = CPLX ? 2 : 1;
  static constexpr int kElem = sizeof(S) * kComps;
  static constexpr int E = 16 / kElem;
  static constexpr int kStep = 4 * E;  // reduction indices of a step
  using Piece = S[E][kComps];

  const char* base;  // the lane's row, its first reduction index
  int64_t kBytes;    // from one reduction index to the next
  S sign;            // of the imaginary part

  __device__ __forceinline__ void init(const void* X, int64_t ld, int row, int last, bool conj) {
    const int lane = threadIdx.x & 63;
    const int64_t r = min(row + (lane & 15), last);
    kBytes = LAYOUT == KMajor ? kElem : ld * kElem;
    base = static_cast<const char*>(X) + r * (LAYOUT == KMajor ? ld * kElem : kElem) +
           (lane >> 4) * E * kBytes;
    sign = conj ? S(-1) : S(1);
  }
  __device__ __forceinline__ void element(S (&v)[kComps], const char* p) const {
    using V = typename VecOf<S, kComps>::loose;
    const V x = *reinterpret_cast<const V*>(p);
    if constexpr (CPLX) {
      v[0] = x[0];
      v[1] = x[1];
    } else {
      v[0] = x;
    }
  }
  // step at reduction index k, all of it inside the reduction
  __device__ __forceinline__ void load(Piece& v, int64_t k) const {
    const char* p = base + k * kBytes;
    if constexpr (LAYOUT == KMajor) {
      using V = typename VecOf<S, 16 / sizeof(S)>::loose;
      const V x = *reinterpret_cast<const V*>(p);
#pragma unroll
      for (int e = 0; e < E; ++e)
#pragma unroll
        for (int c = 0; c < kComps; ++c) v[e][c] = x[e * kComps + c];
    } else {
#pragma unroll
      for (int e = 0; e < E; ++e) element(v[e], p + e * kBytes);
    }
  }
  // the same with reduction indices from kEnd on as zeros
  __device__ __forceinline__ void load_checked(Piece& v, int64_t k, int64_t kEnd) const {
    const int64_t first = k + ((threadIdx.x & 63) >> 4) * E;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int64_t past = first + e - (kEnd - 1);  // > 0: read the last one instead
      element(v[e], base + (k + e - (past > 0 ? past : 0)) * kBytes);
#pragma unroll
      for (int c = 0; c < kComps; ++c) v[e][c] = past > 0 ? S(0) : v[e][c];
    }
  }
};

template <typename S, bool CPLX, int LA, int LB>
__global__ void __launch_bounds__(64 * kMaxWaves) small_gemm_kernel(GemmDesc d) {
  using OpA = SmallOperand<S, CPLX, LA>;
  using OpB = SmallOperand<S, CPLX, LB>;
  using V4 = typename VecOf<S, 4>::type;
  constexpr int kComps = CPLX ? 2 : 1;
  constexpr int E = OpA::E, kStep = OpA::kStep, kSteps = kGroup / kStep;
  extern __shared__ __attribute__((aligned(16))) unsigned char shared[];
  S(*sums)[kComps][kTile][kTile + 1] = reinterpret_cast<S(*)[kComps][kTile][kTile + 1]>(shared);

  const int row = static_cast<int>(blockIdx.x) % d.tilesM * kTile;
  const int col = static_cast<int>(blockIdx.x) / d.tilesM * kTile;
  if (d.fillMode != FillFull && !tile_active(d, row, col, min(kTile, d.m - row), min(kTile, d.n - col)))
    return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6;
  const int l16 = lane & 15, kk = lane >> 4;
  OpA a;
  OpB b;
  a.init(d.A, d.lda, row, d.m - 1, CPLX && d.conjA);
  b.init(d.B, d.ldb, col, d.n - 1, CPLX && d.conjB);

  V4 re = {S(0), S(0), S(0), S(0)}, im = re;
  auto mma = [&](const typename OpA::Piece& x, const typename OpB::Piece& y) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      re = mfma16x16x4<false>(y[e][0], x[e][0], re);
      if constexpr (CPLX) {
        const S ai = x[e][1] * a.sign, bi = y[e][1] * b.sign;
        im = mfma16x16x4<false>(y[e][0], ai, im);
        re = mfma16x16x4<false>(bi, -ai, re);
        im = mfma16x16x4<false>(bi, x[e][0], im);
      }
    }
  };
  // d.kSplit (whole steps) reduction indices per wave
  int64_t k = wave * d.kSplit;
  const int64_t kEnd = min(d.k, k + d.kSplit);
  typename OpA::Piece x[kSteps];
  typename OpB::Piece y[kSteps];
  for (; k + kGroup <= kEnd; k += kGroup) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      a.load(x[s], k + s * kStep);
      b.load(y[s], k + s * kStep);
    }
#pragma unroll
    for (int s = 0; s < kSteps; ++s) mma(x[s], y[s]);
  }
  if (k < kEnd) {
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if (k + s * kStep >= kEnd) break;  // the same for the whole wave
      a.load_checked(x[s], k + s * kStep, kEnd);
      b.load_checked(y[s], k + s * kStep, kEnd);
    }
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
      if (k + s * kStep >= kEnd) break;
      mma(x[s], y[s]);
    }
  }

#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int j = sizeof(S) == 8 ? kk + 4 * r : 4 * kk + r;
    sums[wave][0][j][l16] = re[r];
    if (CPLX) sums[wave][kComps - 1][j][l16] = im[r];
  }
  __syncthreads();
  for (int e = threadIdx.x; e < kTile * kTile; e += blockDim.x) {
    const int i = e % kTile, j = e / kTile;
    if (row + i >= d.m || col + j >= d.n) continue;
    S sr = sums[0][0][j][i], si = sums[0][kComps - 1][j][i];
    for (int w = 1; w < waves; ++w) {
      sr += sums[w][0][j][i];
      if (CPLX) si += sums[w][kComps - 1][j][i];
    }
    store_result<S, CPLX>(d, row + i, col + j, sr, si);
  }
}

template <typename S, bool CPLX>
hipError_t launch_typed(const GemmDesc& desc, int layoutA, int layoutB, hipStream_t stream) {
  constexpr int kStep = SmallOperand<S, CPLX, KMajor>::kStep;
  GemmDesc d = desc;
  d.tilesM = (d.m + kTile - 1) / kTile;
  d.tilesN = (d.n + kTile - 1) / kTile;
  const int64_t steps = (d.k + kStep - 1) / kStep;
  int64_t waves = (d.k + kGroup - 1) / kGroup;
  waves = waves < kMaxWaves ? waves : kMaxWaves;
  d.kSplit = (steps + waves - 1) / waves * kStep;
  waves = (steps * kStep + d.kSplit - 1) / d.kSplit;  // no empty wave
  const std::size_t shared = waves * kTile * (kTile + 1) * sizeof(S) * (CPLX ? 2 : 1);
  const dim3 grid(static_cast<unsigned>(d.tilesM) * d.tilesN), block(static_cast<unsigned>(64 * waves));
  auto* kernel = layoutA == KMajor
                     ? (layoutB == KMajor ? small_gemm_kernel<S, CPLX, KMajor, KMajor>
                                          : small_gemm_kernel<S, CPLX, KMajor, MNMajor>)
                     : (layoutB == KMajor ? small_gemm_kernel<S, CPLX, MNMajor, KMajor>
                                          : small_gemm_kernel<S, CPLX, MNMajor, MNMajor>);
  hipLaunchKernelGGL(kernel, grid, block, shared, stream, d);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_small_gemm(const GemmDesc& d, bool complex, int layoutA, int layoutB,
                             hipStream_t stream, bool f32) {
  if (f32)
    return complex ? launch_typed<float, true>(d, layoutA, layoutB, stream)
                   : launch_typed<float, false>(d, layoutA, layoutB, stream);
  return complex ? launch_typed<double, true>(d, layoutA, layoutB, stream)
                 : launch_typed<double, false>(d, layoutA, layoutB, stream);
}

}  // namespace spla_amd
