// Pieces of the register-staged tile kernels (gemm_any.hip, conv_any.hip): 16-byte chunks at the edge of
// a row and the MFMA of one pair of chunk fragments.
#pragma once
#include "common.hpp"

namespace uk::kern {

// Elements [x, x + E) of a line of X elements at `line` (E = 16 / sizeof(T)), zero past the end.
// A chunk that crosses the end reads the line's last E elements and shifts them down.
template <typename T>
__device__ __forceinline__ u32x4 any_load16_edge(const T* line, int x, int X) {
  constexpr int E = 16 / sizeof(T);
  u32x4 v = u32x4{0, 0, 0, 0};
  if (X - x >= E) {
    v = any_load16(line + x);
  } else if (x < X) {
    if (X >= E) {
      unsigned __int128 q = __builtin_bit_cast(unsigned __int128, any_load16(line + (X - E)));
      q >>= (x + E - X) * (int)sizeof(T) * 8;
      v = __builtin_bit_cast(u32x4, q);
    } else {
      T e[E];
#pragma unroll
      for (int i = 0; i < E; ++i) e[i] = i < X - x ? line[x + i] : T(0);
      __builtin_memcpy(&v, e, 16);
    }
  }
  return v;
}

// One fragment pair: lane (i = lane & 15, g = lane >> 4) holds 16 bytes of row i at k group g.
// f16: one 16x16x32 MFMA. f32: four 16x16x4 MFMAs, MFMA e taking element e of every chunk (any
// assignment of k to MFMA steps gives the same sum when both operands agree). B first: the tile
// comes out transposed, so a lane holds four consecutive columns n of one row m.
template <typename T>
__device__ __forceinline__ f32x4 any_mfma(u32x4 b, u32x4 a, f32x4 acc) {
  if constexpr (sizeof(T) == 2) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, b), __builtin_bit_cast(f16x8, a), acc, 0, 0,
                                                  0);
  } else {
    const f32x4 bf = __builtin_bit_cast(f32x4, b), af = __builtin_bit_cast(f32x4, a);
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(bf[e], af[e], acc, 0, 0, 0);
    return acc;
  }
}

}  // namespace uk::kern
