// Streaming FP64 / complex-FP64 A^T B and A^H B for small m, n and long
// reductions (both operands K-major: the ssb local product with opA = T or C,
// opB = N). Such products are bound by HBM bandwidth: a complex product moves
// 16 (m + n) bytes per reduction index for 8 m n flops, i.e. m n / (2 (m + n))
// flop per byte, below the FP64 matrix ridge (78.6 TFLOP/s / 8 TB/s = 9.8) for
// m = n <= 39.
//
// Each wave owns the whole m x n output in FM x FN MFMA fragments of 16 x 16
// elements. It streams chunks of 128 bytes of every row, eight rows per load
// instruction, through registers and a part of LDS of its own into the layout of
// the MFMA operands: no barrier in the loop, the loads of the next chunk in flight
// during the MFMAs of this one. The waves of all workgroups take the chunks in
// turn, so that the chip reads one moving window of every row.
//
// Why through LDS: a fragment read straight into registers takes 64 bytes of 16
// rows per load instruction, half a cache line. Measured (one card, kernel alone,
// same accumulation): complex m = n = 16, k = 8e6 745 -> 580 us (5.5 -> 7.1 TB/s),
// m = n = 32, k = 4e6 1037 -> 606 us (3.9 -> 6.8 TB/s); 256-byte chunks, two
// chunks in flight and four workgroups per CU instead of two are 1 to 5 % slower,
// loads without the non-temporal hint 10 to 13 %.
//
// Small outputs (GROUPS > 1): m, n <= 16 / GROUPS. A fragment holds GROUPS
// stretches of 128 bytes of its 16 / GROUPS rows; the products of equal stretches
// lie in the diagonal blocks of the accumulator and are added at the end. With one
// stretch the matrix cores would spend 16 x 16 outputs on m x n and bound the
// product (m = n = 1: 1.2 TB/s).
//
// Arithmetic as in tile_mma.hpp: complex operands are not expanded (four MFMAs per
// pair of fragments, the MFMA's own negation), B is the first MFMA operand, lane
// (kk, l16) holds rows kk + 4 r of D (columns of C) and column l16 (row of C).
// Two accumulators per output (complex: the two products of each component, real:
// the two elements of a chunk's 16-byte pieces) halve the length of the sums, where
// there are registers for them.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels/gemm_desc.hpp"
#include "kernels/launch.hpp"
#include "kernels/tile_mma.hpp"

namespace spla_amd {
namespace {

using namespace tile;

constexpr int kWaves = 4;
constexpr int kChunkRowBytes = 128;  // of one row and stretch

// Accumulators per output: two where there are registers for them (launch bounds: 256). Real
// m > 32 with n > 16 is the one shape with one (with two, 254 registers and 8 spilled).
constexpr int sums_per_output(int fm, int fn, int comps, int lines) {
  return 16 * fm * fn * comps + 6 * 2 * (fm + fn) * lines < 200 ? 2 : 1;
}

// LINES: 128-byte stretches of a row that follow each other in a chunk; TURN: stretches that
// a wave takes at its turn, in TURN / LINES chunks. The turns decide which sums an element
// goes to, so they are the same however the operands lie in memory. ALIGNED: every row
// starts on a cache line (see rows_aligned).
template <bool CPLX, bool CONJ, int FM, int FN, int GROUPS, int LINES, int TURN, bool ALIGNED>
__global__ void __launch_bounds__(kWaves * 64, 2) skinny_gemm_kernel(GemmDesc d) {
  static_assert(GROUPS == 1 || (FM == 1 && FN == 1), "stretches share one fragment");
  static_assert(GROUPS == 1 || TURN == 1, "one or the other");
  static_assert(TURN % LINES == 0, "whole chunks");
  constexpr int kComps = CPLX ? 2 : 1;
  constexpr int kElem = 8 * kComps;
  constexpr int kRows = 16 / GROUPS;  // rows of A or columns of B in a fragment
  constexpr int kChunk = kChunkRowBytes * GROUPS * LINES;  // bytes of a row in one chunk
  constexpr int kParts = TURN / LINES;  // chunks of a turn
  constexpr int kTurn = kChunk * kParts;
  constexpr int kTurnElems = kTurn / kElem;
  constexpr int kPerRow = kChunk / 16;      // 16-byte pieces of a row
  constexpr int kLoadsA = 2 * FM * LINES, kLoads = 2 * (FM + FN) * LINES;  // per lane and chunk
  constexpr int kLineBytes = 16 * (FM + FN) * kRowBytes;
  constexpr int kStageBytes = LINES * kLineBytes;
  constexpr int kSumBytes = FM * FN * kComps * 16 * 17 * 8;
  constexpr int kWaveBytes = kStageBytes > kSumBytes ? kStageBytes : kSumBytes;
  constexpr int kSums = sums_per_output(FM, FN, kComps, LINES);
  __shared__ __attribute__((aligned(16))) unsigned char lds[kWaves][kWaveBytes];
  typedef double loose2 __attribute__((ext_vector_type(2), aligned(8)));

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int kk = lane >> 4;
  // turns of this wave: id, id + waves, id + 2 waves, ...; the partial one at the
  // end of the reduction goes to the wave that is next
  const int64_t turns = d.k / kTurnElems;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * kWaves;
  const int64_t id = static_cast<int64_t>(blockIdx.x) * kWaves + wave;
  const int64_t mine = turns > id ? (turns - id + waves - 1) / waves : 0;
  const bool tail = d.k % kTurnElems != 0 && turns % waves == id;

  // Piece u of a lane: row and 16-byte piece of A or B, and where it lies in LDS.
  // Rows past the operand's last one read that one: they feed outputs that are
  // not stored.
  constexpr int kLoadRows = GROUPS == 1 ? 64 / kPerRow : 1;  // of one load instruction
  auto piece_row = [&](int u) {
    const int v = u < kLoadsA ? u : u - kLoadsA;
    return GROUPS == 1 ? v * kLoadRows + lane / kPerRow : (v * 64 + lane) / kPerRow;
  };
  auto piece_col = [&](int u) {
    const int v = u < kLoadsA ? u : u - kLoadsA;
    return GROUPS == 1 ? lane % kPerRow : (v * 64 + lane) % kPerRow;
  };
  auto slot = [&](int u) {
    const int row = piece_row(u), col = piece_col(u), first = u < kLoadsA ? 0 : 16 * FM;
    return (GROUPS == 1 ? col / 8 * kLineBytes + (first + row) * kRowBytes
                        : (first + col / 8 * kRows + row) * kRowBytes) +
           16 * (col % 8);
  };
  const char* p[kLoads];
#pragma unroll
  for (int u = 0; u < kLoads; ++u) {
    const int row = piece_row(u);
    p[u] = u < kLoadsA ? static_cast<const char*>(d.A) + min(row, d.m - 1) * d.lda * kElem
                       : static_cast<const char*>(d.B) + min(row, d.n - 1) * d.ldb * kElem;
    p[u] += 16 * piece_col(u);
  }
  unsigned char* const own = lds[wave];
  const unsigned char* const operand = own + l16 * kRowBytes + 16 * kk;

  dbl4 re[kSums][FM][FN], im[kSums][CPLX ? FM : 1][CPLX ? FN : 1];
#pragma unroll
  for (int h = 0; h < kSums; ++h)
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int g = 0; g < FN; ++g) {
        re[h][f][g] = dbl4{0.0, 0.0, 0.0, 0.0};
        if constexpr (CPLX) im[h][f][g] = dbl4{0.0, 0.0, 0.0, 0.0};
      }
  // one chunk, from its registers through LDS; `next` runs once the registers are free
  auto compute = [&](const dbl2 (&x)[kLoads], auto next) {
#pragma unroll
    for (int u = 0; u < kLoads; ++u) *reinterpret_cast<dbl2*>(own + slot(u)) = x[u];
    __builtin_amdgcn_sched_barrier(0);
    next();
    // LDS serves a wave's own accesses in order: only the compiler must keep it
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s = 0; s < 2 * LINES; ++s) {
      const unsigned char* const from = operand + s / 2 * kLineBytes + 64 * (s % 2);
      dbl2 a[FM], b[FN];
#pragma unroll
      for (int f = 0; f < FM; ++f)
        a[f] = *reinterpret_cast<const dbl2*>(from + f * 16 * kRowBytes);
#pragma unroll
      for (int g = 0; g < FN; ++g)
        b[g] = *reinterpret_cast<const dbl2*>(from + (FM + g) * 16 * kRowBytes);
#pragma unroll
      for (int q = 0; q < 2 * kComps; ++q)
#pragma unroll
        for (int f = 0; f < FM; ++f)
#pragma unroll
          for (int g = 0; g < FN; ++g) {
            constexpr int h = kSums - 1;  // the second sum
            if constexpr (!CPLX) {
              re[q * h][f][g] = mfma16x16x4<false>(b[g][q], a[f][q], re[q * h][f][g]);
            } else {
              if (q == 0) re[0][f][g] = mfma16x16x4<false>(b[g][0], a[f][0], re[0][f][g]);
              if (q == 1) im[0][f][g] = mfma16x16x4<CONJ>(b[g][0], a[f][1], im[0][f][g]);
              if (q == 2) re[h][f][g] = mfma16x16x4<!CONJ>(b[g][1], a[f][1], re[h][f][g]);
              if (q == 3) im[h][f][g] = mfma16x16x4<false>(b[g][1], a[f][0], im[h][f][g]);
            }
          }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

#pragma unroll
  for (int u = 0; u < kLoads; ++u) p[u] += id * kTurn;
  if (mine > 0) {
    dbl2 x[kLoads];
    auto load = [&]() {
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const loose2* q = reinterpret_cast<const loose2*>(p[u]);
        x[u] = ALIGNED ? __builtin_nontemporal_load(q) : *q;
      }
    };
    load();
    // from the last chunk of a turn to the first of the next
    const int64_t step = waves * kTurn - (kParts - 1) * kChunk;
    for (int64_t c = 1; c < mine * kParts; ++c) {
      const int64_t by = c % kParts == 0 ? step : kChunk;
#pragma unroll
      for (int u = 0; u < kLoads; ++u) p[u] += by;
      compute(x, load);
    }
    compute(x, [] {});
#pragma unroll
    for (int u = 0; u < kLoads; ++u) p[u] += step;
  }
  if (tail) {  // p is at the partial turn: elements past the reduction are zero
    const int rest = static_cast<int>(d.k % kTurnElems) * kComps;  // doubles
#pragma unroll
    for (int part = 0; part < kParts; ++part) {
      const int left = rest - part * (kChunk / 8);
      if (left <= 0) break;
      dbl2 x[kLoads];
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const int at = 2 * piece_col(u);
        const double* q = reinterpret_cast<const double*>(p[u] + part * kChunk);
        x[u] = dbl2{0.0, 0.0};
        if (at < left) x[u][0] = q[0];
        if (at + 1 < left) x[u][1] = q[1];
      }
      compute(x, [] {});
    }
  }

  // The sums of the four waves and of the stretches, in this order, through LDS.
  __syncthreads();
  double* sums = reinterpret_cast<double*>(own);
#pragma unroll
  for (int f = 0; f < FM; ++f)
#pragma unroll
    for (int g = 0; g < FN; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        double* s = sums + ((f * FN + g) * kComps * 16 + kk + 4 * r) * 17 + l16;
        s[0] = kSums == 2 ? re[0][f][g][r] + re[kSums - 1][f][g][r] : re[0][f][g][r];
        if constexpr (CPLX)
          s[16 * 17] = kSums == 2 ? im[0][f][g][r] + im[kSums - 1][f][g][r] : im[0][f][g][r];
      }
  __syncthreads();
  const bool flip = CPLX && (CONJ ? !d.conjA : (d.conjA && d.conjB));  // see TileMma::flip_result
  double* work = static_cast<double*>(d.work) + static_cast<int64_t>(blockIdx.x) * d.n * d.Mp;
  for (int e = threadIdx.x; e < d.n * d.Mp; e += kWaves * 64) {
    const int j = e / d.Mp;
    const int i = (e % d.Mp) / kComps, c = (e % d.Mp) % kComps;
    const int at = ((i / 16 * FN + j / 16) * kComps + c) * 16 * 17 + (j % 16) * 17 + i % 16;
    double sum = 0.0;
    for (int w = 0; w < kWaves; ++w)
#pragma unroll
      for (int s = 0; s < GROUPS; ++s)
        sum += reinterpret_cast<const double*>(lds[w])[at + s * kRows * 18];
    work[e] = flip && c ? -sum : sum;
  }
}

// Rows that do not start on cache lines: every 128-byte stretch lies in two lines,
// which the waves of its neighbours read as well, so the loads leave the lines in
// the caches (complex m = n = 32, k = 4000001 1013 -> 812 us; 26 x 12, 6576433 791 ->
// 687 us), and one fragment per operand takes two stretches at a time, three lines
// for two (m = n = 16, k = 8000001 803 -> 678 us; more fragments have no registers
// for it). Rows on cache lines load one stretch at a time, the two of a turn one after the
// other (m = n = 16, k = 8e6, whole call: complex 614 us, real 321 us; turns of one
// stretch 635 and 335).
bool rows_aligned(const GemmDesc& d, int elemBytes) {
  const uint64_t bits = reinterpret_cast<uintptr_t>(d.A) | reinterpret_cast<uintptr_t>(d.B) |
                        (d.m > 1 ? static_cast<uint64_t>(d.lda) * elemBytes : 0) |
                        (d.n > 1 ? static_cast<uint64_t>(d.ldb) * elemBytes : 0);
  return bits % kChunkRowBytes == 0;
}

template <bool CPLX, bool CONJ, int FM, int FN, int GROUPS = 1>
hipError_t launch(const GemmDesc& d, hipStream_t stream) {
  constexpr int kLines = GROUPS == 1 && FM == 1 && FN == 1 ? 2 : 1;
  if (rows_aligned(d, CPLX ? 16 : 8))
    hipLaunchKernelGGL((skinny_gemm_kernel<CPLX, CONJ, FM, FN, GROUPS, 1, kLines, true>),
                       dim3(d.splits), dim3(kWaves * 64), 0, stream, d);
  else
    hipLaunchKernelGGL((skinny_gemm_kernel<CPLX, CONJ, FM, FN, GROUPS, kLines, kLines, false>),
                       dim3(d.splits), dim3(kWaves * 64), 0, stream, d);
  return hipGetLastError();
}

template <bool CPLX, bool CONJ>
hipError_t launch_typed(const GemmDesc& d, hipStream_t stream) {
  const bool wide = d.n > 16;
  if (d.m > 32) {
    if constexpr (!CPLX)
      return wide ? launch<CPLX, CONJ, 4, 2>(d, stream) : launch<CPLX, CONJ, 4, 1>(d, stream);
    return hipErrorInvalidValue;
  }
  if (d.m > 16)
    return wide ? launch<CPLX, CONJ, 2, 2>(d, stream) : launch<CPLX, CONJ, 2, 1>(d, stream);
  if (wide) return launch<CPLX, CONJ, 1, 2>(d, stream);
  switch (skinny_groups(d.m, d.n)) {
    case 16:
      return launch<CPLX, CONJ, 1, 1, 16>(d, stream);
    case 8:
      return launch<CPLX, CONJ, 1, 1, 8>(d, stream);
    case 4:
      return launch<CPLX, CONJ, 1, 1, 4>(d, stream);
    case 2:
      return launch<CPLX, CONJ, 1, 1, 2>(d, stream);
    default:
      return launch<CPLX, CONJ, 1, 1>(d, stream);
  }
}

}  // namespace

int skinny_groups(int64_t m, int64_t n) {
  const int64_t rows = m > n ? m : n;
  return rows > 8 ? 1 : (rows > 4 ? 2 : (rows > 2 ? 4 : (rows > 1 ? 8 : 16)));
}

int skinny_sums(bool complex, int64_t m, int64_t n) {
  const int fm = m > 32 ? 4 : (m > 16 ? 2 : 1), fn = n > 16 ? 2 : 1;
  return sums_per_output(fm, fn, complex ? 2 : 1, 1);
}

bool skinny_supported(bool complex, int layoutA, int layoutB, int64_t m, int64_t n) {
  return layoutA == KMajor && layoutB == KMajor && m >= 1 && n >= 1 && m <= (complex ? 32 : 64) &&
         n <= 32;
}

hipError_t launch_skinny_gemm(const GemmDesc& d, bool complex, hipStream_t stream) {
  if (!complex) return launch_typed<false, false>(d, stream);
  return d.conjA != d.conjB ? launch_typed<true, true>(d, stream)
                            : launch_typed<true, false>(d, stream);
}

}  // namespace spla_amd
