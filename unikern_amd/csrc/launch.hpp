// Host-side launchers of the kernel families (internal to libunikern_hip.so).
// Every launcher validates what its kernel's grid and indexing assume before it enqueues,
// and returns hipErrorInvalidValue instead of launching a shape the kernel does not cover.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "host/uk_core.hpp"
#include "variants.hpp"

namespace uk {

// The grid of `wgs` workgroups (at most 2^31 - 1): a grid dimension holds fewer than 2^32 work items, so more
// than kFoldedRow workgroups fold into y. A kernel launched so takes its id from kern::folded_id() and returns
// where that is past the last workgroup.
inline dim3 folded_grid(int64_t wgs) {
  return wgs <= kFoldedRow ? dim3((unsigned)wgs) : dim3(kFoldedRow, (unsigned)((wgs + kFoldedRow - 1) / kFoldedRow));
}

enum class RowOp : int { Sum = 0, RmsNorm = 1, Softmax = 2 };

hipError_t launch_rows(const Plan& p, RowOp op, const float* X, const float* W, float* Y, int64_t L, int64_t C,
                       float eps, hipStream_t s);
hipError_t launch_channelscale(const float* X, const float* S, float* Y, int64_t L, int64_t C, hipStream_t s);
// partials: kReduceParts floats; not used where n <= kReduceOneMax.
hipError_t launch_reduce1d(const float* X, float* partials, float* Y, int64_t n, hipStream_t s);

hipError_t launch_gemm_f16(const Plan& p, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                           hipStream_t s);
// variant 1: gemm_f32_kernel (f32, M, N, K multiples of 64); others: the kGemmAnyVariants entry with
// that id (any shape).
hipError_t launch_gemm_generic(int variant, DType dt, Layout lay, const void* A, const void* B, void* C, int64_t M,
                               int64_t N, int64_t K, hipStream_t s);
hipError_t launch_gemm_any(int variant, DType dt, Layout lay, const void* A, const void* B, void* C, int64_t M, int64_t N,
                           int64_t K, hipStream_t s);
bool gemm_f32_tiled_supported(int64_t M, int64_t N, int64_t K);
hipError_t launch_q8_gemm(const Plan& p, const void* X, const void* Wq, float* Y, int64_t M, int64_t N, int64_t K,
                          hipStream_t s);
// Matrix-core ceiling probe (kernels/probe.hip): per loop iteration eight
// v_mfma_f32_16x16x32_f16 (form 16) or four v_mfma_f32_32x32x16_f16 (form 32), 2^17 flops per
// wavefront either way; out receives (shader cycles, 100 MHz ticks, 0) per wavefront, four
// wavefronts per workgroup.
constexpr int probe_mfmas_per_iter(int form) { return form == 16 ? 8 : 4; }
hipError_t launch_mfma_probe(int form, int workgroups, int iters, unsigned long long* out, hipStream_t s);
hipError_t launch_conv_any(int variant, const Shape& sh, Layout lay, const float* X, const float* Wt, const float* scale,
                           float* Y, hipStream_t s);
hipError_t launch_conv_igemm(const Plan& p, const Shape& sh, Layout lay, const float* X, const float* Wt,
                             const float* scale, float* Y, hipStream_t s);

}  // namespace uk
