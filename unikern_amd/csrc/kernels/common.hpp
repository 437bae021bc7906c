// Device helpers shared by the gfx950 kernel families: 64-wide wavefront reductions built
// on DPP row operations, ds_swizzle and readlane, and small vector types.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../variants.hpp"

namespace uk::kern {

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// DPP controls (GCN/CDNA encoding).
constexpr int kDppQuadXor1 = 0xB1;     // quad_perm [1,0,3,2]
constexpr int kDppQuadXor2 = 0x4E;     // quad_perm [2,3,0,1]
constexpr int kDppRowHalfMirror = 0x141;
constexpr int kDppRowMirror = 0x140;
constexpr int kSwizzleXor16 = 0x401F;  // ds_swizzle bit mode: and 0x1F, xor 0x10

template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float swizzle_xor16(float v) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), kSwizzleXor16));
}
__device__ __forceinline__ float readlane(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// Sum over the 64 lanes of a wavefront. Butterfly within 16-lane rows (DPP), across the two
// rows of each half (swizzle), then across halves (readlane). Every lane gets the same value.
__device__ __forceinline__ float wave_sum(float v) {
  v += dpp<kDppQuadXor1>(v);
  v += dpp<kDppQuadXor2>(v);
  v += dpp<kDppRowHalfMirror>(v);
  v += dpp<kDppRowMirror>(v);
  v += swizzle_xor16(v);
  return readlane(v, 0) + readlane(v, 32);
}

// The same in binary64 over groups of N lanes (4, 16 or the 64), the halves of each value moved alike.
template <int N>
__device__ __forceinline__ double lanes_sum(double v) {
  static_assert(N == 4 || N == 16 || N == 64, "a quad, a row or the wavefront");
  auto moved = [](double x, auto move) __attribute__((always_inline)) {
    const uint64_t b = __builtin_bit_cast(uint64_t, x);
    const uint32_t lo = __builtin_bit_cast(uint32_t, move(__builtin_bit_cast(float, (uint32_t)b)));
    const uint32_t hi = __builtin_bit_cast(uint32_t, move(__builtin_bit_cast(float, (uint32_t)(b >> 32))));
    return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
  };
  v += moved(v, [](float x) { return dpp<kDppQuadXor1>(x); });
  v += moved(v, [](float x) { return dpp<kDppQuadXor2>(x); });
  if constexpr (N >= 16) {
    v += moved(v, [](float x) { return dpp<kDppRowHalfMirror>(x); });
    v += moved(v, [](float x) { return dpp<kDppRowMirror>(x); });
  }
  if constexpr (N == 64) {
    v += moved(v, [](float x) { return swizzle_xor16(x); });
    v = moved(v, [](float x) { return readlane(x, 0); }) + moved(v, [](float x) { return readlane(x, 32); });
  }
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp<kDppQuadXor1>(v));
  v = fmaxf(v, dpp<kDppQuadXor2>(v));
  v = fmaxf(v, dpp<kDppRowHalfMirror>(v));
  v = fmaxf(v, dpp<kDppRowMirror>(v));
  v = fmaxf(v, swizzle_xor16(v));
  return fmaxf(readlane(v, 0), readlane(v, 32));
}

// 16 bytes at any element-aligned global address (one unaligned 128-bit load).
__device__ __forceinline__ u32x4 any_load16(const void* p) {
  u32x4 v;
  __builtin_memcpy(&v, p, 16);
  return v;
}

// Workgroup barrier that waits for this wavefront's LDS operations only: global loads into registers
// stay in flight across it (the compiler waits for them where their values are used).
__device__ __forceinline__ void lds_barrier() {
  __asm__ volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// The workgroup's number in a grid of folded_grid(). The row is a constant, not gridDim.x: a kernel that reads
// gridDim takes hidden arguments, which cost the host 0.3 us a launch (4.2 -> 4.5 us at the smallest calls).
__device__ __forceinline__ int folded_id() { return (int)(blockIdx.y * (unsigned)kFoldedRow + blockIdx.x); }

__device__ __forceinline__ int lane_id() { return __lane_id(); }

}  // namespace uk::kern
