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

// C <- alpha * (re, im) + beta * (cr, ci) in the scalar type S; (cr, ci): C before, not
// used when beta == 0.
template <typename S, bool CPLX>
__device__ __forceinline__ void store_update(const GemmDesc& d, int i, int j, S re, S im, S cr,
                                             S ci) {
  const S aRe = static_cast<S>(d.alphaRe), aIm = static_cast<S>(d.alphaIm);
  const S bRe = static_cast<S>(d.betaRe), bIm = static_cast<S>(d.betaIm);
  if (CPLX) {
    S* c = static_cast<S*>(d.C) + (static_cast<int64_t>(j) * d.ldc + i) * 2;
    S outRe = aRe * re - aIm * im;
    S outIm = aRe * im + aIm * re;
    if (!d.betaZero) {
      outRe += bRe * cr - bIm * ci;
      outIm += bRe * ci + bIm * cr;
    }
    c[0] = outRe;
    c[1] = outIm;
  } else {
    S* c = static_cast<S*>(d.C) + static_cast<int64_t>(j) * d.ldc + i;
    // written out: which product the compiler rounds first differs with its surroundings
    const S out = aRe * re;
    c[0] = d.betaZero ? out : static_cast<S>(fma(bRe, cr, out));
  }
}

// The same, reading C (beta == 0: C not read).
template <typename S, bool CPLX>
__device__ __forceinline__ void store_result(const GemmDesc& d, int i, int j, S re, S im) {
  S cr = S(0), ci = S(0);
  if (!d.betaZero) {
    const S* c = static_cast<const S*>(d.C) + (static_cast<int64_t>(j) * d.ldc + i) * (CPLX ? 2 : 1);
    cr = c[0];
    if (CPLX) ci = c[1];
  }
  store_update<S, CPLX>(d, i, j, re, im, cr, ci);
}

}  // namespace spla_amd
