// screen.hpp -- operands and bounds of the MFMA distance screens.
//
// A screen distance s = (|a|^2 + |b|^2) - 2 a'.b' on screen copies a', b' comes with a rigorous
// bound |s - d| <= kappa (|a|^2 + |b|^2), d the canonical FP32 distance; only candidates that
// the bound leaves undecided are evaluated canonically.  The 16-bit copy is BF16 when that
// holds every value exactly, else FP16 of the values scaled by a power of two: with 11 bits
// its bound is an eighth of BF16's, so that about one candidate per decision is left.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.hpp"
#include "rules.hpp"

namespace tg {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// Staging of R rows (ids in LDS) through LDS, DC elements at a time, by a 256-thread
// workgroup.  PREC 1: FP32 rows; 2: 16-bit rows; 3: FP8 rows.
template <int PREC, int DC, int R>
struct ScreenStage {
  static constexpr int ESZ = PREC == 3 ? 1 : (PREC == 2 ? 2 : 4);
  static constexpr int RS = DC * ESZ + 16;  // padded row stride in bytes: 16-byte reads of 16
                                            // rows touch every bank once
  static constexpr int BYTES = R * RS;
  static constexpr int EPP = 16 / ESZ;      // elements of a 16-byte piece
  static constexpr int PPR = DC / EPP;      // pieces per row
  static constexpr int NP = R * PPR / 256;  // pieces per thread
  static_assert(R * PPR % 256 == 0 && NP >= 1, "whole pieces per thread");
  uint4 v[NP];

  // loads chunk [d0, d0 + DC) of the rows r with valid(r); the others read as zero
  template <class Valid>
  __device__ __forceinline__ void load(const void* src, const uint32_t* ids, int D, int d0,
                                       Valid valid) {
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int e = int(threadIdx.x) + 256 * q, r = e / PPR, col = d0 + (e % PPR) * EPP;
      v[q] = make_uint4(0u, 0u, 0u, 0u);
      if (valid(r) && col < D)
        v[q] = *reinterpret_cast<const uint4*>(static_cast<const unsigned char*>(src) +
                                               (size_t(ids[r]) * D + col) * ESZ);
    }
  }
  __device__ __forceinline__ void store(unsigned char* sm) const {
#pragma unroll
    for (int q = 0; q < NP; ++q) {
      const int e = int(threadIdx.x) + 256 * q;
      *reinterpret_cast<uint4*>(sm + (e / PPR) * RS + (e % PPR) * 16) = v[q];
    }
  }
};

// acc += one 16 x 16 block of products over a staged chunk: rows at pa against rows at pb
// (each the first of 16 staged rows).  mfma layout: lane l, register r holds row
// 4 (l / 16) + r, column l % 16.  BF: 16-bit rows are BF16, else FP16.
template <int PREC, bool BF, int DC>
__device__ __forceinline__ void screen_block(const unsigned char* pa, const unsigned char* pb,
                                             int l, f32x4& acc) {
  constexpr int RS = ScreenStage<PREC, DC, 256>::RS;
  pa += (l & 15) * RS;
  pb += (l & 15) * RS;
  if constexpr (PREC == 1) {
    // a lane's four consecutive elements feed four products: both operands take element
    // k0 + 4 (l / 16) + q in product q
#pragma unroll
    for (int k0 = 0; k0 < DC; k0 += 16) {
      const int kb = (k0 + 4 * (l >> 4)) * 4;
      const f32x4 fa = *reinterpret_cast<const f32x4*>(pa + kb);
      const f32x4 fb = *reinterpret_cast<const f32x4*>(pb + kb);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[q], fb[q], acc, 0, 0, 0);
    }
  } else if constexpr (PREC == 2) {
#pragma unroll
    for (int k0 = 0; k0 < DC; k0 += 32) {
      const int kb = (k0 + 8 * (l >> 4)) * 2;
      if constexpr (BF)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(pa + kb),
                                                      *reinterpret_cast<const bf16x8*>(pb + kb),
                                                      acc, 0, 0, 0);
      else
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const f16x8*>(pa + kb),
                                                     *reinterpret_cast<const f16x8*>(pb + kb),
                                                     acc, 0, 0, 0);
    }
  } else {
#pragma unroll
    for (int k0 = 0; k0 < DC; k0 += 32) {
      const int kb = k0 + 8 * (l >> 4);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(*reinterpret_cast<const long*>(pa + kb),
                                                       *reinterpret_cast<const long*>(pb + kb),
                                                       acc, 0, 0, 0);
    }
  }
}

// Runs chunk(): the products of every staged chunk of the D elements, the next chunk's loads
// in flight meanwhile.  sm: ScreenStage::BYTES of LDS; ends with a barrier (sm is free again).
template <int PREC, int DC, int R, class Valid, class Chunk>
__device__ __forceinline__ void screen_chunks(const void* src, const uint32_t* ids, int D,
                                              Valid valid, unsigned char* sm, Chunk chunk) {
  ScreenStage<PREC, DC, R> st;
  st.load(src, ids, D, 0, valid);
  for (int d0 = 0; d0 < D; d0 += DC) {
    st.store(sm);
    __syncthreads();
    if (d0 + DC < D) st.load(src, ids, D, d0 + DC, valid);
    chunk();
    __syncthreads();
  }
}

}  // namespace tg
