// Epilogue of the single-product kernels (gemm_f64.hip, small.hip): fill predicate and
// the alpha / beta update of C. Device code only.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels/gemm_desc.hpp"

namespace spla_amd {

__device__ __forceinline__ bool tile_active(const GemmDesc& d, int64_t r, int64_t c, int64_t nr,
                                            int64_t nc) {
  // SPLA block_is_active (src/block_generation/block.hpp:58-66) on a tile.
  if (d.fillMode == FillUpper) return c + nc + d.fillColOff > r + d.fillRowOff;
  if (d.fillMode == FillLower) return r + nr + d.fillRowOff > c + d.fillColOff;
  return true;
}

// C <- alpha * (re, im) + beta * C in the scalar type S (beta == 0: C not read).
template <typename S, bool CPLX>
__device__ __forceinline__ void store_result(const GemmDesc& d, int i, int j, S re, S im) {
  const S aRe = static_cast<S>(d.alphaRe), aIm = static_cast<S>(d.alphaIm);
  const S bRe = static_cast<S>(d.betaRe), bIm = static_cast<S>(d.betaIm);
  if (CPLX) {
    S* c = static_cast<S*>(d.C) + (static_cast<int64_t>(j) * d.ldc + i) * 2;
    S outRe = aRe * re - aIm * im;
    S outIm = aRe * im + aIm * re;
    if (!d.betaZero) {
      const S cr = c[0], ci = c[1];
      outRe += bRe * cr - bIm * ci;
      outIm += bRe * ci + bIm * cr;
    }
    c[0] = outRe;
    c[1] = outIm;
  } else {
    S* c = static_cast<S*>(d.C) + static_cast<int64_t>(j) * d.ldc + i;
    S out = aRe * re;
    if (!d.betaZero) out += bRe * c[0];
    c[0] = out;
  }
}

}  // namespace spla_amd
