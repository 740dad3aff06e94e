// MFMA tile routine shared by the single-product kernels (gemm_f64.hip: FP64
// and FP32, real and complex) and the batched kernels (batched.hip).
// Device code only; include from HIP translation units.
//
// What bounds it: the matrix cores, and the vector ALU next to them. On gfx950
// a VALU instruction does not run beside an FP64 or FP32 MFMA of its SIMD: in
// register-only loops (two waves per SIMD) one v_xor_b32 per MFMA takes
// v_mfma_f64_16x16x4_f64 from 77.7 to 71.0 TFLOP/s, two to 68.9, four to 65.4
// (v_mfma_f32_16x16x4_f32: 155, 134, 120, 105), while scalar instructions and
// one ds_read_b128 per MFMA cost nothing. The k loop is therefore written
// without vector arithmetic:
//   * complex operands are not expanded. A fragment holds 16 complex rows (or
//     columns); a lane's 16-byte chunk gives the real and the imaginary operand
//     as they lie in memory, and four MFMAs (re re, im im, im re, re im) make
//     the real and the imaginary accumulators of the same lane. Signs: the FP64
//     MFMA negates its operand itself; FP32 flips the imaginary part of A, one
//     VALU instruction for 2 FN MFMAs. A conjugated result is the product of
//     the other operand's conjugate, so one template bit covers all four
//     conj(A), conj(B) forms (flip_result negates the imaginary part once, in
//     the epilogue).
//   * global addresses are a wave-uniform 64-bit base (scalar unit) plus a
//     32-bit lane offset that stays the same for the whole reduction.
//   * rows past the operand's edge are clamped to its last row when the
//     offsets are made: they only feed outputs that are not stored, so ragged
//     tiles run the same loop (with per-element checks in the loop the edge
//     tiles of a 1000 x 1000 x 1e5 product held it at 39 TFLOP/s).
//   * LDS addresses are one base per operand plus immediate offsets (the two
//     buffers are unrolled).
//   * the last, partial k-block takes a separate checked load.
//
// Measured against the same tiles with the embedding's swaps and signs, 64-bit
// addresses and row checks in the loop (one card): complex doubles 2048 x 2048 x
// 2e5 A^H B 102.3 -> 92.2 ms (72.8 TFLOP/s), 100000 x 4096 x 4096 A B 201.8 ->
// 176.4 ms (76.1 of the 77.7 a register-only loop reaches), complex floats 2048 x
// 2048 x 2e5 58.9 -> 45.3 ms (148 of 155), real doubles 1000 x 1000 x 1e5 A^T B
// (ragged) 5.53 -> 3.59 ms.
//
// Layouts. A k-block is 128 bytes of a K-major row (8 complex or 16 real
// doubles, 16 complex or 32 real floats) in two sub-blocks of four 16-byte
// chunks; lane group kk = lane / 16 reads chunk kk of its row. MN-major
// operands lie in LDS as they lie in memory, [reduction index][row]: a 16-byte
// read there holds VR neighbouring rows of one reduction index, which become
// the same lane's operands of VR fragments (fragment p covers rows
// VR * (lane % 16) + p), so nothing is transposed. Both layouts take the
// reduction index in the same order inside a sub-block (element s of chunk kk).
//
// The MFMAs take B as their first operand: D rows are columns of C and a
// lane's D column is a row of C, so 16 lanes store 16 neighbouring rows of a
// column of C (128 bytes of doubles, 256 of complex doubles).
// Accumulators of lane (kk, l16), column l16 of D: D rows kk + 4 r (FP64) or
// 4 kk + r (FP32), r = 0..3.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "kernels/gemm_desc.hpp"

namespace spla_amd {
namespace tile {

typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef double dbl2 __attribute__((ext_vector_type(2)));
typedef float flt4 __attribute__((ext_vector_type(4)));

template <typename S, int N>
struct VecOf {
  typedef S type __attribute__((ext_vector_type(N)));
  // as it lies in a caller's matrix: aligned like one scalar
  typedef S loose __attribute__((ext_vector_type(N), aligned(sizeof(S))));
};
template <typename S>
struct VecOf<S, 1> {
  typedef S type;
  typedef S loose;
};

// Load of one register piece (4, 8 or 16 bytes) at a 32-bit lane offset.
template <typename P>
__device__ __forceinline__ P buffer_load(__amdgpu_buffer_rsrc_t rsrc, uint32_t off,
                                         uint32_t scalarOff) {
  static_assert(sizeof(P) == 4 || sizeof(P) == 8 || sizeof(P) == 16, "piece of 4, 8 or 16 bytes");
  if constexpr (sizeof(P) == 16)
    return __builtin_bit_cast(P, __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, scalarOff, 0));
  else if constexpr (sizeof(P) == 8)
    return __builtin_bit_cast(P, __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, scalarOff, 0));
  else
    return __builtin_bit_cast(P, __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, scalarOff, 0));
}

template <int N>
struct Index {
  static constexpr int value = N;
};

template <typename T>
struct Type {
  using type = T;
};

// The same value in a scalar register: loads through pointers that the kernel's
// own stores might alias leave wave-uniform values in vector registers.
template <typename V>
__device__ __forceinline__ V uniform(V v) {
  static_assert(sizeof(V) == 4 || sizeof(V) == 8, "one or two registers");
  if constexpr (sizeof(V) == 4) {
    return __builtin_bit_cast(
        V, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(uint32_t, v)));
  } else {
    const uint64_t b = __builtin_bit_cast(uint64_t, v);
    const uint64_t lo =
        static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b)));
    const uint64_t hi =
        static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b >> 32)));
    return __builtin_bit_cast(V, hi << 32 | lo);
  }
}

constexpr int kThreads = 256;
constexpr int kChunk = 16;      // bytes of one lane's fragment read
constexpr int kBlockBytes = 128;  // bytes of a K-major row in one k-block
// Row stride of K-major tiles in LDS, measured with the bank-conflict counter on
// the fragment reads (ds_read_b128: 16 rows x 4 chunks per wave): 160-byte rows
// read conflict-free, 144-, 176- and 208-byte rows cost 4 conflict cycles.
constexpr int kRowBytes = 160;

// D = B-operand x A-operand + D; NEG negates the A operand.
template <bool NEG>
__device__ __forceinline__ dbl4 mfma16x16x4(double b, double a, dbl4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(b, a, c, 0, 0, NEG ? 2 : 0);
}
template <bool NEG>
__device__ __forceinline__ flt4 mfma16x16x4(float b, float a, flt4 c) {
  static_assert(!NEG, "the FP32 MFMA has no operand negation");
  return __builtin_amdgcn_mfma_f32_16x16x4f32(b, a, c, 0, 0, 0);
}

// One operand of one tile product: element (row, l) at X + row * ld + l
// (K-major) or X + l * ld + row (MN-major).
template <typename S>
struct TileOperands {
  const S* A;
  const S* B;
  int64_t lda, ldb;  // elements
  int m, n;          // element rows / columns of C
};

// Moves ROWS rows x one k-block of an operand from global memory through
// registers to LDS.
// WIDE: rows (K-major) or reduction indices (MN-major) so far apart that 32-bit
// lane offsets do not reach over a wave's pieces (tile_wide of gemm_desc.hpp): 64-bit lane
// addresses, one per piece (K-major) or one of the first (MN-major), to which a wave-uniform
// distance is added for every load.
template <typename S, bool CPLX, int LAYOUT, int ROWS, bool WIDE>
struct TileStage {
  static constexpr int kComps = CPLX ? 2 : 1;
  static constexpr int kElem = sizeof(S) * kComps;          // bytes of an element
  static constexpr int kPerChunk = kChunk / kElem;          // elements of a chunk
  static constexpr int kBK = kBlockBytes / kElem;           // elements of a k-block
  static constexpr int kBytes = ROWS * (LAYOUT == KMajor ? kRowBytes : kBlockBytes);
  // K-major: 16-byte chunks, eight lanes per row; MN-major: single elements,
  // neighbouring lanes on neighbouring rows
  static constexpr int kScalars = LAYOUT == KMajor ? kChunk / sizeof(S) : (CPLX ? 2 : 1);
  static constexpr int kPieceBytes = kScalars * sizeof(S);
  static constexpr int kPieces = ROWS * kBlockBytes / (kThreads * kPieceBytes);
  static_assert(kPieces >= 1, "tile smaller than one piece per thread");
  using Piece = typename VecOf<S, kScalars>::type;
  struct Regs {
    Piece p[kPieces];
  };

  // One wave-uniform base per wave and 32-bit lane offsets. K-major: wave w moves
  // rows w ROWS / 4 .. (w + 1) ROWS / 4 - 1, piece u its rows 8 u .. 8 u + 7 (an
  // offset per piece); MN-major: the same rows in every piece, piece u
  // u * pieceStep bytes further on.
  static constexpr int kWaveRows = ROWS / 4;
  static constexpr int kOffs = LAYOUT == KMajor ? kPieces : 1;
  const char* origin;   // the tile's first row, first reduction index
  const char* base;     // the wave's first row or reduction index (WIDE: the tile's)
  int last;             // last row that exists, relative to the tile
  int64_t rowBytes;
  int64_t blockStep;    // bytes from one k-block to the next
  uint32_t pieceStep;
  uint32_t off[kOffs];
  const char* address[WIDE ? kOffs : 1];  // WIDE: in place of the offsets
  int64_t kEnd;         // reduction range in elements, relative to k-block 0
  int fast;             // k-blocks 0 .. fast - 1 are whole

  // Row (relative to the tile) of the thread's piece u.
  __device__ __forceinline__ static int tile_row(int tid, int u) {
    return LAYOUT == KMajor ? (tid >> 6) * kWaveRows + 8 * u + ((tid & 63) >> 3) : tid % ROWS;
  }
  // rows [rowBase, limit) of the operand at X exist (at least one); reduction
  // elements [k0, k1).
  __device__ __forceinline__ void init(const S* X, int64_t ld, int rowBase, int limit, int64_t k0,
                                       int64_t k1) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    last = limit - 1 - rowBase;
    const int64_t ldBytes = ld * kElem;
    const uint32_t ld32 = static_cast<uint32_t>(ldBytes);
    const char* x = reinterpret_cast<const char*>(X) + static_cast<int64_t>(rowBase) *
                                                           (LAYOUT == KMajor ? ldBytes : kElem);
    kEnd = k1 - k0;
    rowBytes = LAYOUT == KMajor ? ldBytes : kElem;
    origin = x + k0 * (LAYOUT == KMajor ? kElem : ldBytes);
    fast = static_cast<int>(kEnd / kBK);
    if constexpr (WIDE) {
      base = origin;
      blockStep = LAYOUT == KMajor ? kBlockBytes : kBK * ldBytes;
#pragma unroll
      for (int u = 0; u < kOffs; ++u) {
        const int64_t row = min(tile_row(threadIdx.x, u), last);
        address[u] = LAYOUT == KMajor
                         ? origin + row * ldBytes + kChunk * (lane & 7)
                         : origin + (threadIdx.x / ROWS) * ldBytes + row * kElem;
      }
    } else if (LAYOUT == KMajor) {
      const int first = min(wave * kWaveRows, last);
      base = origin + first * ldBytes;
      blockStep = kBlockBytes;
      pieceStep = 0;
#pragma unroll
      for (int u = 0; u < kPieces; ++u)
        off[u % kOffs] = static_cast<uint32_t>(min(tile_row(threadIdx.x, u), last) - first) * ld32 +
                         kChunk * (lane & 7);
    } else {
      constexpr int kPerWave = ROWS < 64 ? 64 / ROWS : 1;  // reduction indices of a wave's piece
      const int first = ROWS < 64 ? wave * kPerWave : wave * 64 / ROWS;
      base = origin + first * ldBytes;
      blockStep = kBK * ldBytes;
      pieceStep = (kThreads / ROWS) * ld32;
      off[0] = static_cast<uint32_t>(min(tile_row(threadIdx.x, 0), last)) * kElem;
      if (ROWS < 64) off[0] += static_cast<uint32_t>(lane / ROWS) * ld32;
    }
  }

  // readfirstlane: wave-uniform already, but kept in scalar registers for certain
  __device__ __forceinline__ static __amdgpu_buffer_rsrc_t resource(const char* p) {
    const uint64_t b = reinterpret_cast<uint64_t>(p);
    const uint64_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b));
    const uint64_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(b >> 32));
    return __builtin_amdgcn_make_buffer_rsrc(
        reinterpret_cast<void*>(hi << 32 | (lo & 0xffffffffu)), 0, 0xffffffff, 0x00020000);
  }

  // k-block kb < fast. Buffer loads: the base is four scalar registers, the lane
  // offset one vector register that never changes.
  __device__ __forceinline__ void load_fast(Regs& r, int kb) const {
    if constexpr (WIDE) {
      using Loose = typename VecOf<S, kScalars>::loose;
#pragma unroll
      for (int u = 0; u < kPieces; ++u)
        r.p[u] = *reinterpret_cast<const Loose*>(
            LAYOUT == KMajor ? address[u] + kb * blockStep
                             : address[0] + (kb * kBK + u * (kThreads / ROWS)) * (blockStep / kBK));
      return;
    }
    const __amdgpu_buffer_rsrc_t rsrc = resource(base + kb * blockStep);
#pragma unroll
    for (int u = 0; u < kPieces; ++u)
      r.p[u] = buffer_load<Piece>(
          rsrc, off[u % kOffs],
          LAYOUT == KMajor ? 0 : __builtin_amdgcn_readfirstlane(u * pieceStep));
  }

  // k-block kb, whole or not. Reduction indices past the range are zero in both
  // operands; they are read from the range's last element, so that every load is
  // issued without a branch. A k-block past the range leaves r as it is.
  __device__ __forceinline__ void load(Regs& r, int kb) const {
    if (kb < fast) return load_fast(r, kb);
    const int64_t left = kEnd - static_cast<int64_t>(kb) * kBK;
    if (left <= 0) return;
    const int rem = static_cast<int>(min(left, static_cast<int64_t>(kBK)));
    // The thread index passes through an empty statement so that these offsets
    // are made here, once, and not kept in registers through the loop.
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    using Elem = typename VecOf<S, CPLX ? 2 : 1>::type;
    constexpr int kElems = kPieceBytes / kElem;  // of one piece, along the reduction index
    const int64_t ldBytes = blockStep / kBK;     // MN-major
    const char* b = LAYOUT == KMajor ? base + kb * blockStep : origin + kb * blockStep;
    const __amdgpu_buffer_rsrc_t rsrc = resource(b);
    bool in[kPieces][kElems];
#pragma unroll
    for (int u = 0; u < kPieces; ++u)
#pragma unroll
      for (int e = 0; e < kElems; ++e) {
        const int first = LAYOUT == KMajor ? kPerChunk * (tid & 7) : (tid + kThreads * u) / ROWS;
        in[u][e] = first + e < rem;
        const int l = min(first + e, rem - 1);
        Elem v;
        if constexpr (WIDE) {
          using Loose = typename VecOf<S, CPLX ? 2 : 1>::loose;
          const int64_t row = min(tile_row(tid, u), last);
          v = *reinterpret_cast<const Loose*>(
              LAYOUT == KMajor ? origin + row * rowBytes + kb * blockStep + l * kElem
                               : b + l * ldBytes + row * kElem);
        } else if constexpr (LAYOUT == KMajor) {
          v = buffer_load<Elem>(rsrc, off[u] + (l - first) * kElem, 0);
        } else {
          v = buffer_load<Elem>(rsrc,
                                min(tile_row(tid, u), last) * kElem +
                                    static_cast<uint32_t>(l) * static_cast<uint32_t>(ldBytes),
                                0);
        }
        if constexpr (kScalars == 1) {
          r.p[u] = v;
        } else if constexpr (CPLX) {
          r.p[u][2 * e] = v[0];
          r.p[u][2 * e + 1] = v[1];
        } else {
          r.p[u][e] = v;
        }
      }
    if (rem == kBK) return;
#pragma unroll
    for (int u = 0; u < kPieces; ++u)
#pragma unroll
      for (int e = 0; e < kElems; ++e) {
        if constexpr (kScalars == 1) {
          r.p[u] = in[u][e] ? r.p[u] : S(0);
        } else {
#pragma unroll
          for (int c = 0; c < kComps; ++c)
            r.p[u][kComps * e + c] = in[u][e] ? r.p[u][kComps * e + c] : S(0);
        }
      }
  }

  __device__ __forceinline__ static void store(const Regs& r, unsigned char* lds) {
    unsigned char* p = LAYOUT == KMajor
                           ? lds + tile_row(threadIdx.x, 0) * kRowBytes + kChunk * (threadIdx.x & 7)
                           : lds + threadIdx.x * kElem;
    constexpr int kStep = LAYOUT == KMajor ? 8 * kRowBytes : kThreads * kElem;
#pragma unroll
    for (int u = 0; u < kPieces; ++u) *reinterpret_cast<Piece*>(p + u * kStep) = r.p[u];
  }
};

// Fragments of one operand for one sub-block: F fragments of 16 rows.
template <typename S, bool CPLX, int LAYOUT, int ROWS, int F>
struct TileFrags {
  using Stage = TileStage<S, CPLX, LAYOUT, ROWS, false>;
  static constexpr int kSteps = Stage::kPerChunk;  // MFMA steps of a sub-block
  // MN-major: neighbouring rows of one read, each a fragment of its own
  static constexpr int VR = LAYOUT == KMajor ? 1 : (kSteps < F ? kSteps : F);
  static_assert(F % VR == 0, "fragments come in groups of VR");
  S re[kSteps][F];
  S im[CPLX ? kSteps : 1][F];

  // row (relative to the wave) of entry i of fragment f
  __device__ __forceinline__ static int row(int f, int i) {
    return 16 * VR * (f / VR) + VR * i + f % VR;
  }

  __device__ __forceinline__ void read(const unsigned char* lds, int waveRow, int sub) {
    const int l16 = threadIdx.x & 15;
    const int kk = (threadIdx.x & 63) >> 4;
    if constexpr (LAYOUT == KMajor) {
      constexpr int kN = kChunk / sizeof(S);
      using V = typename VecOf<S, kN>::type;
      const unsigned char* p = lds + (waveRow + l16) * kRowBytes + kChunk * kk;
#pragma unroll
      for (int f = 0; f < F; ++f) {
        const V v = *reinterpret_cast<const V*>(p + f * 16 * kRowBytes + sub * 4 * kChunk);
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
          re[s][f] = v[CPLX ? 2 * s : s];
          if (CPLX) im[s % (CPLX ? kSteps : 1)][f] = v[(CPLX ? 2 * s + 1 : s)];
        }
      }
    } else {
      constexpr int kN = VR * (CPLX ? 2 : 1);
      using V = typename VecOf<S, kN>::type;
      const unsigned char* p =
          lds + (kSteps * kk * ROWS + waveRow + VR * l16) * Stage::kElem;
#pragma unroll
      for (int s = 0; s < kSteps; ++s)
#pragma unroll
        for (int q = 0; q < F / VR; ++q) {
          const V v = *reinterpret_cast<const V*>(
              p + ((sub * (Stage::kBK / 2) + s) * ROWS + 16 * VR * q) * Stage::kElem);
          if constexpr (kN == 1) {
            re[s][q] = v;
          } else {
#pragma unroll
            for (int w = 0; w < VR; ++w) {
              re[s][VR * q + w] = v[CPLX ? 2 * w : w];
              if (CPLX) im[s % (CPLX ? kSteps : 1)][VR * q + w] = v[CPLX ? 2 * w + 1 : w];
            }
          }
        }
    }
  }
};

// Tile of AR x BN elements of C (four waves in a 2 x 2 grid, each FM x FN
// fragments of 16 x 16 elements) over the embedded reduction range
// [kBegin, kEnd), accumulated in registers. WIDE: see TileStage. CONJ: one of A and B is conjugated
// (see flip_result). On return every thread has passed the final barrier, so the
// LDS buffers may be reused at once (reads issued after that barrier only fill
// registers that are discarded).
template <typename S, bool CPLX, bool CONJ, int LA, int LB, int FM, int FN, bool WIDE = false>
struct TileMma {
  static constexpr int WAVES_M = 2, WAVES_N = 2;
  static constexpr int AR = 16 * FM * WAVES_M;  // element rows
  static constexpr int BN = 16 * FN * WAVES_N;
  static constexpr bool kF64 = sizeof(S) == 8;
  static constexpr int kComps = CPLX ? 2 : 1;
  using V4 = typename VecOf<S, 4>::type;
  using StageA = TileStage<S, CPLX, LA, AR, WIDE>;
  using StageB = TileStage<S, CPLX, LB, BN, WIDE>;
  using FragsA = TileFrags<S, CPLX, LA, AR, FM>;
  using FragsB = TileFrags<S, CPLX, LB, BN, FN>;
  static constexpr int kSteps = FragsA::kSteps;
  static constexpr int kPasses = kSteps * (CPLX ? 4 : 1);  // of FM x FN MFMAs per sub-block

  struct Smem {
    alignas(16) unsigned char a[2][StageA::kBytes];
    alignas(16) unsigned char b[2][StageB::kBytes];
  };
  struct Acc {
    V4 re[FM][FN];
    V4 im[CPLX ? FM : 1][CPLX ? FN : 1];
  };

  // The imaginary part of the sum is to be negated: the kernel computes A B, or
  // conj(A) B for CONJ, and conj(A) conj(B) = conj(A B), A conj(B) = conj(conj(A) B).
  __device__ __forceinline__ static bool flip_result(int conjA, int conjB) {
    return CPLX && (CONJ ? !conjA : (conjA && conjB));
  }

  // pass p of a sub-block: FM x FN MFMAs
  __device__ __forceinline__ static void mfma_pass(Acc& acc, const FragsA& a, const FragsB& b,
                                                   int p) {
    if constexpr (!CPLX) {
#pragma unroll
      for (int f = 0; f < FM; ++f)
#pragma unroll
        for (int g = 0; g < FN; ++g)
          acc.re[f][g] = mfma16x16x4<false>(b.re[p][g], a.re[p][f], acc.re[f][g]);
    } else {
      const int s = p / 4;
#pragma unroll
      for (int f = 0; f < FM; ++f) {
        const S ar = a.re[s][f], ai = a.im[s][f];
        // re += ar br -+ ai bi; im += +-ai br + ar bi
        const S minus = kF64 ? ai : -ai;
#pragma unroll
        for (int g = 0; g < FN; ++g) {
          if (p % 4 == 0)
            acc.re[f][g] = mfma16x16x4<false>(b.re[s][g], ar, acc.re[f][g]);
          else if (p % 4 == 1)
            acc.re[f][g] =
                CONJ ? mfma16x16x4<false>(b.im[s][g], ai, acc.re[f][g])
                     : mfma16x16x4<kF64>(b.im[s][g], minus, acc.re[f][g]);
          else if (p % 4 == 2)
            acc.im[f][g] =
                CONJ ? mfma16x16x4<kF64>(b.re[s][g], minus, acc.im[f][g])
                     : mfma16x16x4<false>(b.re[s][g], ai, acc.im[f][g]);
          else
            acc.im[f][g] = mfma16x16x4<false>(b.im[s][g], ar, acc.im[f][g]);
        }
      }
    }
  }

  __device__ __forceinline__ static void clear(Acc& acc) {
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int g = 0; g < FN; ++g) {
        acc.re[f][g] = V4{S(0), S(0), S(0), S(0)};
        if (CPLX) acc.im[f % (CPLX ? FM : 1)][g % (CPLX ? FN : 1)] = V4{S(0), S(0), S(0), S(0)};
      }
  }
  // total += acc
  __device__ __forceinline__ static void add(Acc& total, const Acc& acc) {
#pragma unroll
    for (int f = 0; f < FM; ++f)
#pragma unroll
      for (int g = 0; g < FN; ++g) {
        total.re[f][g] += acc.re[f][g];
        if (CPLX) {
          constexpr int kM = CPLX ? FM : 1, kN = CPLX ? FN : 1;
          total.im[f % kM][g % kN] += acc.im[f % kM][g % kN];
        }
      }
  }

  // STRETCHES: every `stretch` k-blocks (even, at least 2) the accumulators are added to
  // totals and start anew, so that rounding errors grow with the length of a stretch and
  // not of the whole range. The totals take as many registers again.
  template <bool STRETCHES = false>
  __device__ __forceinline__ static void run(const TileOperands<S>& op, int row0, int col0,
                                             int64_t kBegin, int64_t kEnd, Smem& sm, Acc& acc,
                                             int stretch = 0) {
    const int wave = threadIdx.x >> 6;
    const int wa = (wave % WAVES_M) * 16 * FM;
    const int wb = (wave / WAVES_M) * 16 * FN;
    const int64_t k0 = kBegin / kComps, k1 = kEnd / kComps;
    const int nk = static_cast<int>((k1 - k0 + StageA::kBK - 1) / StageA::kBK);
    StageA sa;
    StageB sb;
    sa.init(op.A, op.lda, row0, op.m, k0, k1);
    sb.init(op.B, op.ldb, col0, op.n, k0, k1);
    auto load = [&](typename StageA::Regs& ra, typename StageB::Regs& rb, int kb) {
      sa.load(ra, kb);
      sb.load(rb, kb);
    };

    // Small wave tiles load two k-blocks ahead through two register sets, the
    // larger ones one and a half (k-block it + 2 as soon as it + 1 is stored).
    constexpr bool kTwoAhead = FM * FN * kComps <= 4;
    // Left to itself the compiler begins a k-block's loads between the stores of the one in
    // front, for which the large real double tiles with one MN-major operand lack the
    // registers: 5 spilled, two of them read back in the loop (2048 x 2048 x 2e4 A B 2.50
    // ms, 2.39 with the loads last). The others have them and lose 1 % with the loads last.
    constexpr bool kLoadsLast = kF64 && !CPLX && LA != LB;
    typename StageA::Regs ra[kTwoAhead ? 2 : 1];
    typename StageB::Regs rb[kTwoAhead ? 2 : 1];
    FragsA fa[2];
    FragsB fb[2];
    const int whole = min(sa.fast, sb.fast);
    if (nk > 0) {
      typename StageA::Regs pa = {};
      typename StageB::Regs pb = {};
      constexpr int kSet = kTwoAhead ? 1 : 0;  // register set of k-block 1
      if (whole >= 2) {  // both in flight together
        sa.load_fast(pa, 0);
        sb.load_fast(pb, 0);
        sa.load_fast(ra[kSet], 1);
        sb.load_fast(rb[kSet], 1);
        StageA::store(pa, sm.a[0]);
        StageB::store(pb, sm.b[0]);
      } else {
        load(pa, pb, 0);
        load(ra[kSet], rb[kSet], 1);
        StageA::store(pa, sm.a[0]);
        StageB::store(pb, sm.b[0]);
      }
    }
    clear(acc);
    if (nk == 0) return;
    Acc total;
    if constexpr (STRETCHES) clear(total);
    int edge = stretch;  // k-blocks in front of the next stretch
    auto stretch_end = [&](int done) {
      if constexpr (STRETCHES) {
        if (done != edge) return;
        add(total, acc);
        clear(acc);
        edge += stretch;
      }
    };
    __syncthreads();
    fa[0].read(sm.a[0], wa, 0);
    fb[0].read(sm.b[0], wb, 0);

    // One k-block over LDS buffer CUR: sub-block 0's first half with the reads of
    // sub-block 1; the staged stores into the other buffer; its second half, which
    // covers the stores' completion; the barrier; the next k-block's sub-block 0
    // reads; sub-block 1, which covers those reads. The stores and the reads after
    // the barrier are unconditional (branches make the wait counts conservative):
    // in the last k-block they store staged registers into the buffer that is no
    // longer read, and read values that are not used.
    // next(set): loads k-block it + 2 into register set `set`; tail: these loads
    // may be partial.
    auto kblock = [&](auto cur, auto tail, auto next) {
      constexpr bool kTail = decltype(tail)::value;
      constexpr int CUR = decltype(cur)::value;
      constexpr int kStored = kTwoAhead ? CUR ^ 1 : 0;  // register set of k-block it + 1
      fa[1].read(sm.a[CUR], wa, 1);
      fb[1].read(sm.b[CUR], wb, 1);
      if (kTwoAhead) next(CUR);
#pragma unroll
      for (int p = 0; p < kPasses / 2; ++p) mfma_pass(acc, fa[0], fb[0], p);
      __builtin_amdgcn_sched_barrier(0);
      StageA::store(ra[kStored], sm.a[CUR ^ 1]);
      StageB::store(rb[kStored], sm.b[CUR ^ 1]);
      if (!kTwoAhead && !kTail) {
        if constexpr (kLoadsLast) __builtin_amdgcn_sched_barrier(0);
        next(0);
      }
#pragma unroll
      for (int p = kPasses / 2; p < kPasses; ++p) mfma_pass(acc, fa[0], fb[0], p);
      __builtin_amdgcn_sched_barrier(0);  // these MFMAs cover the stores' completion
      __syncthreads();
      if (!kTwoAhead && kTail) next(0);  // fewer registers are live here
      fa[0].read(sm.a[CUR ^ 1], wa, 0);
      fb[0].read(sm.b[CUR ^ 1], wb, 0);
#pragma unroll
      for (int p = 0; p < kPasses; ++p) mfma_pass(acc, fa[1], fb[1], p);
      __builtin_amdgcn_sched_barrier(0);  // the next k-block's reads stay behind these (registers)
    };
    // While both k-blocks that an iteration loads are whole, the loads are
    // unconditional: the wait counts stay exact (a load that may not be issued
    // makes every later wait a full one) and the loop holds no branch.
    int it = 0;
    for (; it + 3 < whole; it += 2) {
      auto next = [&](int kb) {
        return [&, kb](int set) {
          sa.load_fast(ra[set], kb);
          sb.load_fast(rb[set], kb);
        };
      };
      kblock(Index<0>(), Index<0>(), next(it + 2));
      kblock(Index<1>(), Index<0>(), next(it + 3));
      stretch_end(it + 2);
    }
    auto next = [&](int kb) {
      return [&, kb](int set) {
        if (kb < nk) load(ra[set], rb[set], kb);
      };
    };
    for (; it < nk; it += 2) {
      kblock(Index<0>(), Index<1>(), next(it + 2));
      if (it + 1 < nk) kblock(Index<1>(), Index<1>(), next(it + 3));
      stretch_end(it + 2);
    }
    if constexpr (STRETCHES) {
      add(total, acc);
      acc = total;
    }
  }

  // Calls f(i, j, re, im) for every element of the tile inside m x n; `flip`:
  // see flip_result.
  template <typename F>
  __device__ __forceinline__ static void for_each(int row0, int col0, int m, int n, bool flip,
                                                  const Acc& acc, F&& f) {
    const int wave = threadIdx.x >> 6;
    const int l16 = threadIdx.x & 15;
    const int kk = (threadIdx.x & 63) >> 4;
    const int wr = row0 + (wave % WAVES_M) * 16 * FM;
    const int wc = col0 + (wave / WAVES_M) * 16 * FN;
#pragma unroll
    for (int g = 0; g < FN; ++g)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = wc + FragsB::row(g, kF64 ? kk + 4 * r : 4 * kk + r);
        if (j >= n) continue;
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
          const int i = wr + FragsA::row(fm, l16);
          if (i >= m) continue;
          S im = S(0);
          if (CPLX) {
            im = acc.im[fm % (CPLX ? FM : 1)][g % (CPLX ? FN : 1)][r];
            im = flip ? -im : im;
          }
          f(i, j, acc.re[fm][g][r], im);
        }
      }
  }

  // The same for f(i, j, re, im, cr, ci) with the element (cr, ci) of C at C + j ldc + i.
  // A column group's elements are all loaded before the group in front of it is stored:
  // read one by one between the stores, which may alias, each waits out its own memory
  // latency (real 100003 x 260 x 260, beta = 0.5: 326 -> 308 us).
  template <typename F>
  __device__ __forceinline__ static void for_each_update(int row0, int col0, int m, int n,
                                                         bool flip, const Acc& acc, const S* C,
                                                         int64_t ldc, F&& f) {
    const int wave = threadIdx.x >> 6;
    const int l16 = threadIdx.x & 15;
    const int kk = (threadIdx.x & 63) >> 4;
    const int wr = row0 + (wave % WAVES_M) * 16 * FM;
    const int wc = col0 + (wave / WAVES_M) * 16 * FN;
    using Elem = typename VecOf<S, kComps>::loose;
    Elem c[2][4][FM];
    auto row = [&](int fm) { return wr + FragsA::row(fm, l16); };
    auto col = [&](int g, int r) { return wc + FragsB::row(g, kF64 ? kk + 4 * r : 4 * kk + r); };
    auto load = [&](int g) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int fm = 0; fm < FM; ++fm)
          c[g % 2][r][fm] = *reinterpret_cast<const Elem*>(
              C + (min(col(g, r), n - 1) * ldc + min(row(fm), m - 1)) * kComps);
    };
    load(0);
#pragma unroll
    for (int g = 0; g < FN; ++g) {
      if (g + 1 < FN) load(g + 1);
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int fm = 0; fm < FM; ++fm) {
          const int i = row(fm), j = col(g, r);
          if (i >= m || j >= n) continue;
          const Elem v = c[g % 2][r][fm];
          if constexpr (CPLX) {
            const S im = acc.im[fm][g][r];
            f(i, j, acc.re[fm][g][r], flip ? -im : im, v[0], v[1]);
          } else {
            f(i, j, acc.re[fm][g][r], S(0), v, S(0));
          }
        }
    }
  }
};

template <typename S, bool CPLX>
__device__ __forceinline__ void store_work(S* w, int64_t Mp, int i, int j, S re, S im) {
  S* p = w + static_cast<int64_t>(j) * Mp + (CPLX ? 2 * i : i);
  p[0] = re;
  if (CPLX) p[1] = im;
}

}  // namespace tile
}  // namespace spla_amd
