// Host/device shared descriptors of the FP64 and FP32 MFMA GEMM kernels.
//
// The kernels compute C <- alpha * opA(A) * opB(B) + beta * C for column-major
// real or interleaved complex operands of one scalar type (double or float;
// the FP32 kernels accumulate in FP32, as a single-precision BLAS does). A
// complex product is four real products per pair of elements, exactly 8*m*n*k
// flops, with no operand expanded in memory. Its sizes are given as those of
// one real GEMM of size (2m) x n x (2k), the "embedded" sizes Mp and Kp:
// q = 2*l + c runs over the real (c = 0) and imaginary (c = 1) parts. Split-K partial
// sums are stored as interleaved (re, im) pairs, i.e. in C's own column-major complex
// layout.
#pragma once

#include <cstdint>

namespace spla_amd {

// Storage order of an operand as seen by the product.
//   KMajor : the reduction index is contiguous (A^T/A^H read of A, B read of B).
//   MNMajor: the output index is contiguous (A read of A, B^T/B^H read of B).
enum OperandLayout : int { KMajor = 0, MNMajor = 1 };

// Fill predicate of a rectangular tile of C, following SPLA's block_is_active
// (src/block_generation/block.hpp:58-66). Coordinates are in elements of the
// (sub-)matrix C; rowOff / colOff locate it in the global matrix.
enum TileFill : int { FillFull = 0, FillUpper = 1, FillLower = 2 };

struct GemmDesc {
  const void* A;  // first element of A (scalars of the kernel's type)
  const void* B;
  void* C;
  void* work;  // split-K partial sums: [splits][N][Mp], raw (unscaled) sums

  int64_t lda, ldb, ldc;  // leading dimensions in elements (complex or real)

  int m, n;   // output rows / columns in elements
  int64_t k;  // reduction length in elements

  int Mp;         // embedded output rows: m (real) or 2m (complex)
  int64_t Kp;     // embedded reduction length: k (real) or 2k (complex)
  int64_t kSplit; // embedded reduction length handled by one split (multiple of the k-block)
  int64_t kSum;   // 0, or the embedded length summed at a time (two k-blocks or a multiple):
                  // the sums of a split are added up (TileM, double precision)
  int splits;
  int tilesM, tilesN;
  int activeTiles;  // tiles that the fill mode needs (all of them without one)

  double alphaRe, alphaIm, betaRe, betaIm;
  int betaZero;  // beta == 0: C is written without being read

  int conjA, conjB;  // complex conjugation of the operand (complex only)

  int fillMode;  // TileFill
  int64_t fillRowOff, fillColOff;
};

// Tile configurations of the FP64 MFMA kernel. Rows are embedded rows.
enum GemmTileConfig : int {
  TileL = 0,   // 128 x 128 block, 4 waves of 64 x 64, 2 blocks per CU
  TileM = 1,   // 64 x 64 block, 4 waves of 32 x 32, 4 blocks per CU
  TileXL = 2,  // 256 x 128 block: two L tiles in turn, 2 blocks per CU (opt-in)
  NumTileConfigs = 3
};

struct TileShape {
  int bm, bn, bk;
};

inline TileShape tile_shape(int cfg) {
  switch (cfg) {
    case TileM:
      return {64, 64, 16};
    case TileXL:
      return {256, 128, 16};
    default:
      return {128, 128, 16};
  }
}

// The tile kernels address a wave's share of a tile with 32-bit lane offsets: 32
// rows of a K-major operand or 32 reduction indices of an MN-major one. Operands
// whose leading dimension spreads these over 4 GiB (complex doubles: from 8.1e6
// elements) take kernels with 64-bit lane addresses, M tiles of which a workgroup each
// covers the planned tile (there are registers for the addresses; one or two vector
// instructions per load): complex 64 x 64 x 8.2e6 A^H B 5.0 ms, real 100 x 100 x
// 16.5e6 10.1 ms (with every element's address and bounds made in the loop 6.5 and 13.8).
inline bool tile_wide(int64_t ld, int elemBytes) {
  return 33 * ld * elemBytes >= (int64_t(1) << 32);
}

}  // namespace spla_amd
