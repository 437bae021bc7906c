// conv2d as an implicit GEMM on gfx950 f32 matrix cores, with the channelscale epilogue fused.
//
// Replaces the reference's SIMT uk_conv<OCB> / uk_conv_g<OCB> (src/codegen_hip.cpp:337-411)
// and its separate channelscale program (:2329-2335). GEMM view: rows = output channels,
// columns = output pixels, reduction k = (input channel, kernel tap):
//   Y[oc][pix] = scale[oc] * sum_k W[oc][k] * X_im2col[k][pix]
// computed with v_mfma_f32_32x32x2f32. Weights are the MFMA A operand and pixels the B operand,
// so each accumulator register holds 32 consecutive pixels of one output channel and the
// epilogue stores coalesce along the pixel axis of Y.
//
// Work split: one wavefront owns 32 output pixels of one image (a plane of Ho*Wo pixels is cut
// into 32-pixel strips) and 64 output channels (two 32x32 tiles); a workgroup is WAVES strips.
// The weights of one channel chunk ([cb channels][taps][64 oc] floats) are staged once per
// workgroup in LDS with coalesced reads of the weight rows. The input is gathered straight
// from global memory with the reduction ordered channel-outer / tap-inner, so the taps of one
// channel pair re-read the same few cache lines from L1; the next channel pair's gathers are
// issued before the current pair's MFMAs. Padding taps read as zero.
//
// The solver takes conv_igemm_kernel and conv_tile_kernel for few shapes now: conv_any.hip, whose tiles gather
// an input once, is faster at nearly all of them. They serve small launches (2x2 kernels, 1x1 over a few
// pixels), images of 2 GiB and more, which conv_any's 32-bit offsets do not cover, and plans that name them.
//
// Layouts: NCHW (X[N][C][H][W], W[Oc][C][Kh][Kw], Y[N][Oc][Ho][Wo], zero padding, stride) and
// the reference's NT conv (X[H][W][C], Wt[Oc][Kh][Kw][C], Y[Oc][Ho][Wo], valid padding,
// src/reference.cpp:6-22).
#include "../launch.hpp"
#include "../variants.hpp"
#include "common.hpp"

namespace uk::kern {

struct ConvArgs {
  const float* x;
  const float* w;
  const float* scale;
  float* y;
  int N, C, H, W, Oc, Kh, Kw, pad, stride, Ho, Wo;
  int strips;  // 32-pixel strips per image
  int cb;      // channels per staged weight chunk (even)
  int gp;      // conv_lds16_kernel: 16-pixel groups per image
  int wpi;     // conv_lds16_kernel: workgroups per image
  int gq, gr;  // conv_lds16_kernel: gp / wpi and gp % wpi (run j has gq + (j < gr) groups)
};

// Weight index of (oc, c, tap) in the caller's layout.
template <bool NCHW>
__device__ __forceinline__ int64_t widx(const ConvArgs& a, int oc, int c, int t) {
  const int taps = a.Kh * a.Kw;
  if constexpr (NCHW) return ((int64_t)oc * a.C + c) * taps + t;  // OIHW
  else return ((int64_t)oc * taps + t) * a.C + c;                 // [Oc][Kh][Kw][C]
}

template <bool NCHW, int TAPS, int WAVES>
__global__ void __launch_bounds__(WAVES * 64)
    conv_igemm_kernel(ConvArgs a) {
  extern __shared__ float wl[];  // [cb][taps][64]
  constexpr int kMaxTaps = TAPS > 0 ? TAPS : 49;
  const int taps = TAPS > 0 ? TAPS : a.Kh * a.Kw;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int unit = blockIdx.x * WAVES + wave;
  const bool active = unit < a.N * a.strips;
  const int n = active ? unit / a.strips : 0;
  const int P = a.Ho * a.Wo;
  const int p = (active ? unit % a.strips : 0) * 32 + (lane & 31);
  const bool pvalid = active && p < P;
  const int ho = pvalid ? p / a.Wo : 0, wo = pvalid ? p % a.Wo : 0;
  const int kk = lane >> 5;  // k parity within an MFMA k-step: channel c + kk
  const int oc0 = blockIdx.y * 64;

  // Per-lane input offset of every tap (-1: the tap reads padding).
  int off[kMaxTaps];
#pragma unroll
  for (int t = 0; t < kMaxTaps; ++t) {
    if (t >= taps) {
      off[t] = -1;
      continue;
    }
    const int kh = t / a.Kw, kw = t % a.Kw;
    const int hi = ho * a.stride + kh - a.pad, wi = wo * a.stride + kw - a.pad;
    const bool ok = pvalid && hi >= 0 && hi < a.H && wi >= 0 && wi < a.W;
    off[t] = ok ? (NCHW ? hi * a.W + wi : (hi * a.W + wi) * a.C) : -1;
  }
  const int64_t HW = (int64_t)a.H * a.W;
  const float* xb = NCHW ? a.x + (int64_t)n * a.C * HW : a.x;
  const int64_t cstride = NCHW ? HW : 1;  // distance between channels

  f32x16 acc[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j) acc[j][0] = acc[j][1] = f32x16{};

  for (int c0 = 0; c0 < a.C; c0 += a.cb) {
    const int cn = (a.C - c0) < a.cb ? (a.C - c0) : a.cb;
    __syncthreads();  // the previous chunk's weight reads are done
    // Stage W[oc0 .. oc0+63][c0 .. c0+cn)[taps] as wl[c][t][oc]: lane = output channel, so the
    // LDS writes are conflict-free; each wavefront walks the chunk's (c, t) elements, 16 loads in
    // flight at a time. Each lane reads along its own weight row, so the 64 rows' cache lines
    // are fetched into L1 once and reused across consecutive elements.
    {
      const int per_oc = a.cb * taps;
      const bool ook = oc0 + lane < a.Oc;
      const int oc = ook ? oc0 + lane : 0;
      for (int e0 = wave * 16; e0 < per_oc; e0 += WAVES * 16) {
        float v[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int e = e0 + j;
          int cl, t;
          if constexpr (NCHW) {
            cl = e / taps;
            t = e - cl * taps;
          } else {
            t = e / a.cb;
            cl = e - t * a.cb;
          }
          const bool ok = ook && e < per_oc && cl < cn;
          const float val = a.w[ok ? widx<NCHW>(a, oc, c0 + cl, t) : 0];
          v[j] = ok ? val : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const int e = e0 + j;
          if (e < per_oc) {
            int cl, t;
            if constexpr (NCHW) {
              cl = e / taps;
              t = e - cl * taps;
            } else {
              t = e / a.cb;
              cl = e - t * a.cb;
            }
            wl[(cl * taps + t) * 64 + lane] = v[j];
          }
        }
      }
    }
    __syncthreads();

    // Reduction over this chunk: channel pairs (c, c+1) outer, taps inner. Gathers use clamped
    // addresses (always inside the input) and a select, so no load is predicated. The next pair's
    // activations (global) and weights (LDS) are loaded before the current pair's MFMAs, so
    // neither latency sits in front of the matrix pipe.
    float xv[kMaxTaps], xn[kMaxTaps];
    auto gather = [&](float (&dst)[kMaxTaps], int c) {
      const int cc = c + kk;
      const bool cok = cc < cn;
      const float* base = xb + (int64_t)(c0 + (cok ? cc : 0)) * cstride;
#pragma unroll
      for (int t = 0; t < kMaxTaps; ++t) {
        const int o = off[t];
        const bool ok = t < taps && cok && o >= 0;
        const float val = base[ok ? o : 0];
        dst[t] = ok ? val : 0.f;
      }
    };
    if constexpr (TAPS > 0) {
      // Weight operands of pair c: w[t] for output channels 0-31 and 32-63 of the tile. Pairs
      // past the chunk read channel 0's row (inside the staged chunk; their activations are 0).
      float wv0[TAPS], wv1[TAPS], wn0[TAPS], wn1[TAPS];
      auto wload = [&](float (&w0)[TAPS], float (&w1)[TAPS], int c) {
        const int cc = c + kk;
        const float* wr = wl + (cc < cn ? cc : 0) * taps * 64 + (lane & 31);
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
          w0[t] = wr[t * 64];
          w1[t] = wr[t * 64 + 32];
        }
      };
      auto mfma_pair = [&](const float (&w0)[TAPS], const float (&w1)[TAPS], f32x16& acc0, f32x16& acc1) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
          acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(w0[t], xv[t], acc0, 0, 0, 0);
          acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(w1[t], xv[t], acc1, 0, 0, 0);
        }
      };
      gather(xv, 0);
      wload(wv0, wv1, 0);
      for (int c = 0; c < cn; c += 4) {
        // pair c into accumulator set 0, pair c+2 into set 1 (independent MFMA chains)
        gather(xn, c + 2);
        wload(wn0, wn1, c + 2);
        mfma_pair(wv0, wv1, acc[0][0], acc[1][0]);
#pragma unroll
        for (int t = 0; t < kMaxTaps; ++t) xv[t] = xn[t];
        if (c + 2 < cn) {
          gather(xn, c + 4);
          wload(wv0, wv1, c + 4);
          mfma_pair(wn0, wn1, acc[0][1], acc[1][1]);
#pragma unroll
          for (int t = 0; t < kMaxTaps; ++t) xv[t] = xn[t];
        }
      }
    } else {
      auto step = [&](int c, f32x16& acc0, f32x16& acc1) {
#pragma unroll
        for (int t = 0; t < kMaxTaps; ++t) {
          if (t < taps) {
            const float* wr = wl + ((c + kk) * taps + t) * 64 + (lane & 31);
            acc0 = __builtin_amdgcn_mfma_f32_32x32x2f32(wr[0], xv[t], acc0, 0, 0, 0);
            acc1 = __builtin_amdgcn_mfma_f32_32x32x2f32(wr[32], xv[t], acc1, 0, 0, 0);
          }
        }
      };
      gather(xv, 0);
      for (int c = 0; c < cn; c += 4) {
        gather(xn, c + 2);
        step(c, acc[0][0], acc[1][0]);
#pragma unroll
        for (int t = 0; t < kMaxTaps; ++t) xv[t] = xn[t];
        if (c + 2 < cn) {
          gather(xn, c + 4);
          step(c + 2, acc[0][1], acc[1][1]);
#pragma unroll
          for (int t = 0; t < kMaxTaps; ++t) xv[t] = xn[t];
        }
      }
    }
  }

  // Epilogue: lane -> pixel p (column), rows oc = oc0 + j*32 + 8*(r/4) + 4*(lane>>5) + r%4.
  if (!pvalid) return;
  float* yb = NCHW ? a.y + (int64_t)n * a.Oc * P : a.y;
  // The scales are all read before the first store (read between stores, each would wait for
  // the store before it: as far as the compiler knows Y may alias them).
  float sc[2][16];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int oc = oc0 + j * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
      sc[j][r] = a.scale && oc < a.Oc ? a.scale[oc] : 1.f;
    }
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int oc = oc0 + j * 32 + (r >> 2) * 8 + (lane >> 5) * 4 + (r & 3);
      if (oc < a.Oc) {
        const float s = acc[j][0][r] + acc[j][1][r];
        yb[(int64_t)oc * P + p] = a.scale ? s * sc[j][r] : s;
      }
    }
}

// ---------------------------------------------------------------------------------------
// conv_tile_kernel: the same implicit GEMM with a wavefront per 32 pixels x 32 output channels
// and a workgroup of S strips x 2 channel halves, so twice as many wavefronts share the SIMDs and
// hide each other's latency. The weights stream through LDS in chunks of CB input channels,
// loaded coalesced along each output channel's contiguous (channel, tap) row and written
// transposed as wl[(c, tap)][oc] with an odd pitch (kPitch = 97 floats) that keeps both the
// transposing writes and the MFMA operand reads (two channel rows 9 * 97 floats apart) nearly free
// of bank conflicts. The next chunk's loads are in flight while the current chunk is reduced.
// TAPS is a compile-time kernel size (9 or 1); the reduction order per output is the same as the
// wide kernel's (channel pairs alternating between two accumulators, taps ascending).
template <bool NCHW, int TAPS, int S, int CB>
__global__ void __launch_bounds__(S * 2 * 64)
    conv_tile_kernel(ConvArgs a) {
  constexpr int kWaves = S * 2;
  constexpr int kOcs = 64;                   // output channels per workgroup (two halves)
  constexpr int kPitch = kOcs + 33;          // odd: conflict-free transposing writes
  constexpr int kRow = CB * TAPS;            // (channel, tap) entries of one chunk
  static_assert(CB % 2 == 0, "channel pairs");
  __shared__ float wl[kRow * kPitch];
  const int tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63;
  const int sidx = wave >> 1, half = wave & 1;
  const int unit = blockIdx.x * S + sidx;
  const bool active = unit < a.N * a.strips;
  const int n = active ? unit / a.strips : 0;
  const int P = a.Ho * a.Wo;
  const int p = (active ? unit % a.strips : 0) * 32 + (lane & 31);
  const bool pvalid = active && p < P;
  const int ho = pvalid ? p / a.Wo : 0, wo = pvalid ? p % a.Wo : 0;
  const int kk = lane >> 5;
  const int oc_base = blockIdx.y * kOcs;

  int off[TAPS];
#pragma unroll
  for (int t = 0; t < TAPS; ++t) {
    const int kh = t / a.Kw, kw = t % a.Kw;
    const int hi = ho * a.stride + kh - a.pad, wi = wo * a.stride + kw - a.pad;
    const bool ok = pvalid && hi >= 0 && hi < a.H && wi >= 0 && wi < a.W;
    off[t] = ok ? (NCHW ? hi * a.W + wi : (hi * a.W + wi) * a.C) : -1;
  }
  const int64_t HW = (int64_t)a.H * a.W;
  const float* xb = NCHW ? a.x + (int64_t)n * a.C * HW : a.x;
  const int64_t cstride = NCHW ? HW : 1;

  // Chunk staging: wavefront w copies output-channel rows ocl = w, w + kWaves, ...; lane l takes
  // entries r = l + 64 q of the row, r the (channel, tap) index in the order the caller's layout
  // stores contiguously for one output channel (NCHW/OIHW: channel-major; NT: tap-major), so a
  // load instruction reads consecutive floats of one row and the per-lane (channel, tap) split is
  // computed once. The LDS entry is wl[(channel * TAPS + tap) * kPitch + ocl].
  constexpr int kRowsW = kOcs / kWaves;  // rows per wavefront
  constexpr int kQ = (kRow + 63) / 64;   // 64-entry pieces of a row
  static_assert(kOcs % kWaves == 0, "rows split evenly over the wavefronts");
  int cl_q[kQ], t_q[kQ], lds_q[kQ];
#pragma unroll
  for (int q = 0; q < kQ; ++q) {
    const int r = lane + 64 * q;
    int cl, t;
    if constexpr (NCHW) {
      cl = r / TAPS;
      t = r - cl * TAPS;
    } else {
      t = r / CB;
      cl = r - t * CB;
    }
    cl_q[q] = r < kRow ? cl : CB;  // CB marks a lane past the row
    t_q[q] = t;
    lds_q[q] = (cl * TAPS + t) * kPitch;
  }
  float wreg[kRowsW][kQ];
  auto load_chunk = [&](int c0) {
#pragma unroll
    for (int i = 0; i < kRowsW; ++i) {
      const int oc = oc_base + wave + i * kWaves;
#pragma unroll
      for (int q = 0; q < kQ; ++q) {
        const int c = c0 + cl_q[q];
        const bool ok = cl_q[q] < CB && oc < a.Oc && c < a.C;
        const int64_t gi = NCHW ? ((int64_t)oc * a.C + c) * TAPS + t_q[q] : ((int64_t)oc * TAPS + t_q[q]) * a.C + c;
        const float v = a.w[ok ? gi : 0];
        wreg[i][q] = ok ? v : 0.f;
      }
    }
  };
  auto store_chunk = [&]() {
#pragma unroll
    for (int i = 0; i < kRowsW; ++i)
#pragma unroll
      for (int q = 0; q < kQ; ++q)
        if (cl_q[q] < CB) wl[lds_q[q] + wave + i * kWaves] = wreg[i][q];
  };

  f32x16 acc[2] = {f32x16{}, f32x16{}};
  float xv[TAPS], xn[TAPS], wv[TAPS], wn[TAPS];
  const int ocl = half * 32 + (lane & 31);
  load_chunk(0);
  for (int c0 = 0; c0 < a.C; c0 += CB) {
    const int cn = (a.C - c0) < CB ? (a.C - c0) : CB;
    __syncthreads();  // every read of the previous chunk is done
    store_chunk();
    __syncthreads();
    if (c0 + CB < a.C) load_chunk(c0 + CB);  // in flight while this chunk is reduced

    auto gather = [&](float (&dst)[TAPS], int c) {
      const int cc = c + kk;
      const bool cok = cc < cn;
      const float* base = xb + (int64_t)(c0 + (cok ? cc : 0)) * cstride;
#pragma unroll
      for (int t = 0; t < TAPS; ++t) {
        const int o = off[t];
        const bool ok = cok && o >= 0;
        const float v = base[ok ? o : 0];
        dst[t] = ok ? v : 0.f;
      }
    };
    auto wload = [&](float (&dst)[TAPS], int c) {
      const int cc = c + kk;
      const float* wr = wl + (cc < cn ? cc : 0) * TAPS * kPitch + ocl;
#pragma unroll
      for (int t = 0; t < TAPS; ++t) dst[t] = wr[t * kPitch];
    };
    gather(xv, 0);
    wload(wv, 0);
    for (int c = 0; c < cn; c += 2) {
      const bool more = c + 2 < cn;
      if (more) {
        gather(xn, c + 2);
        wload(wn, c + 2);
      }
      f32x16& ac = acc[(c >> 1) & 1];
#pragma unroll
      for (int t = 0; t < TAPS; ++t) ac = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[t], xv[t], ac, 0, 0, 0);
      if (more) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
          xv[t] = xn[t];
          wv[t] = wn[t];
        }
      }
    }
  }

  // Epilogue: lane -> pixel p (column), rows oc = oc_base + 32 half + 8 (r / 4) + 4 kk + r % 4.
  if (!pvalid) return;
  float* yb = NCHW ? a.y + (int64_t)n * a.Oc * P : a.y;
  float sc[16];  // all scales read before the first store
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int oc = oc_base + half * 32 + (r >> 2) * 8 + kk * 4 + (r & 3);
    sc[r] = a.scale && oc < a.Oc ? a.scale[oc] : 1.f;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int oc = oc_base + half * 32 + (r >> 2) * 8 + kk * 4 + (r & 3);
    if (oc < a.Oc) {
      const float v = acc[0][r] + acc[1][r];
      yb[(int64_t)oc * P + p] = a.scale ? v * sc[r] : v;
    }
  }
}

// conv_lds_kernel<PT>: NCHW, 3x3, stride 1. Both MFMA operands come from LDS: a workgroup of
// 4 PT wavefronts owns 64 PT consecutive output pixels of one image (flattened Ho*Wo order) x 64
// output channels, each wavefront a 32 x 32 quarter of a 64-pixel tile. Per chunk of 8 input
// channels it stages
//   * the input rows those pixels touch, zero-padded, as xl[quad][row][col][4 channels] (the 8
//     channels split in two quads of 4; one 16-byte entry per (quad, row, col)), and
//   * the chunk's weights as wl[oc][tap][8 channels] (pitch 76 floats per oc: 16 lanes reading
//     16 bytes at consecutive oc hit 16 distinct bank groups),
// so that for each tap one ds_read_b128 of each gives a lane four k values for four
// v_mfma_f32_32x32x2f32: MFMA j of a tap pairs channel j (lanes 0-31, k = 0) with channel 4 + j
// (lanes 32-63, k = 1). The gathered-input kernels issue one global load per MFMA, and a load
// costs its wavefront about as many issue cycles as the MFMA itself; here each tap's input
// entries are read from LDS by the nine taps that share them. The next chunk's global loads are
// in flight (in registers) while the current chunk is multiplied; one barrier per chunk. With
// PT = 2 the chunk's weights (the same for every pixel) are staged once per 128 pixels.
// Requires: 3x3 kernel, stride 1, pad 0 or 1, W + 2*pad <= kLdsCols, W and C multiples of 4 and
// 8 (16-byte rows and whole channel chunks), 16-byte aligned X and W, and 64 PT consecutive
// output pixels spanning at most kLdsRows - 2 output rows; the launcher checks.
constexpr int kLdsRows = kConvLdsRows;
constexpr int kLdsCols = kConvLdsCols;
constexpr int kWPitch = 76;                                    // floats per output channel in wl
constexpr int kXlFloats = 2 * kLdsRows * kLdsCols * 4;         // 4096 floats = 16 KiB
constexpr int kWlFloats = 64 * kWPitch;                        // 4864 floats = 19 KiB
constexpr int kConvLdsBuf = kXlFloats + kWlFloats;

// PT = 2: taps multiplied before the next chunk (loaded two chunks ahead, so landed) is written
// to LDS; the rest of the chunk's MFMAs follow the writes (3, 5 and 7 measured within 1%).
constexpr int kMidTap = 5;

template <int PT>
__global__ void __launch_bounds__(256 * PT)
    conv_lds_kernel(ConvArgs a) {
  constexpr int kThreads = 256 * PT, kPix = 64 * PT;
  __shared__ __attribute__((aligned(16))) float lds[2 * kConvLdsBuf];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int oh = wave & 1, ph = wave >> 1;  // output-channel half, 32-pixel group
  const int P = a.Ho * a.Wo;
  const int tiles = (P + kPix - 1) / kPix;
  // XCD-aware order: workgroup b runs on XCD b % 8, so XCD x takes a contiguous run of tiles
  // (runs of G / 8 or G / 8 + 1) and neighbouring tiles' shared input rows hit its L2.
  const int G = gridDim.x, q8 = G >> 3, r8 = G & 7;
  const int xcd = blockIdx.x & 7;
  const int lin = xcd * q8 + (xcd < r8 ? xcd : r8) + (blockIdx.x >> 3);
  const int n = lin / tiles;
  const int p0 = (lin - n * tiles) * kPix;
  const int r0 = p0 / a.Wo;
  const int rlast = ((p0 + kPix - 1 < P) ? p0 + kPix - 1 : P - 1) / a.Wo;
  const int in_rows = rlast - r0 + 3;  // padded input rows r0 .. rlast + 2
  const int oc_base = blockIdx.y * 64;
  const float* xn = a.x + (int64_t)n * a.C * a.H * a.W;
  const int64_t HW = (int64_t)a.H * a.W;

  // Input staging: task (quad q, row rr, column group g) loads the four channels of the quad at
  // input columns kXW g .. kXW g + kXW - 1 of one row (four vector loads along W, one per
  // channel), transposes them in registers and writes kXW 16-byte entries
  // [q][rr][pad + kXW g + i][0..3]; the padding columns stay zero from the prologue. PT = 1 takes
  // four columns (at most 256 tasks for 256 threads); PT = 2 two columns (at most 512 tasks for
  // 512 threads), so adjacent lanes write entries 32 bytes apart instead of 64 (2-way instead of
  // 4-way bank conflicts) and fewer threads repeat a task. Every thread takes input task
  // tid mod in_tasks: threads that share a task write the same values, and no staging step is
  // under a branch, so the compiler's wait counting keeps the loads in flight across the MFMAs.
  // Loads always use valid addresses (rows outside the image read row 0, output channels past
  // Oc read channel 0); the zero masks apply when the registers are written to LDS.
  constexpr int kXW = PT == 1 ? 4 : 2;
  const int groups = a.W / kXW;
  const int it = tid % (2 * in_rows * groups);
  const int iq = it / (in_rows * groups);
  const int irr = (it / groups) % in_rows, ig = it % groups;
  const int ihi = r0 + irr - a.pad;
  const bool in_ok = ihi >= 0 && ihi < a.H;
  const int64_t in_off = (int64_t)4 * iq * HW + (int64_t)(in_ok ? ihi : 0) * a.W + kXW * ig;
  float* const in_dst0 = lds + ((iq * kLdsRows + irr) * kLdsCols + a.pad + kXW * ig) * 4;
  // Weight staging. PT = 1: task (oc, channel quad h) = tid mod 128 loads the 36 contiguous floats
  // W[oc][c0 + 4h .. +4][0..9] (nine float4) and writes one 16-byte entry wl[oc][t][4h .. 4h+3]
  // per tap. PT = 2: task (oc, channel j) = tid loads the nine floats W[oc][c0 + j][0..9] and
  // writes them to wl[oc][t][j], so the 512 threads share the chunk's weights evenly and no
  // register transposition is needed.
  constexpr int kWv = PT == 1 ? 9 : 2;  // float4 registers per weight task (PT = 2: plus one float)
  const int wocl = PT == 1 ? (tid & 127) >> 1 : tid >> 3;
  const int wch = PT == 1 ? 4 * (tid & 1) : tid & 7;
  const bool w_ok = oc_base + wocl < a.Oc;
  const float* const w_src0 = a.w + ((int64_t)(w_ok ? oc_base + wocl : 0) * a.C + wch) * 9;
  float* const w_dst0 = lds + kXlFloats + wocl * kWPitch + wch;
  // One chunk's staging registers (PT = 2 alternates two sets, see the main loop).
  // Members are float4 vectors (for PT = 2 the input uses two lanes of each, the weights nine
  // floats of wv and wl): arrays of floats or float2, filled and read through vectors of another
  // width, kept the staging registers in scratch memory.
  struct Stage {
    f32x4 xs[4];
    f32x4 wv[kWv];
    float wl;
  };
  auto load_chunk = [&](Stage& r, int c0) __attribute__((always_inline)) {
    const float* src = xn + (int64_t)c0 * HW + in_off;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (kXW == 4) {
        r.xs[j] = *reinterpret_cast<const f32x4*>(src + j * HW);
      } else {
        const f32x2 v = *reinterpret_cast<const f32x2*>(src + j * HW);
        r.xs[j] = f32x4{v.x, v.y, 0.f, 0.f};
      }
    }
    const float* wsrc = w_src0 + (int64_t)c0 * 9;
    if constexpr (PT == 1) {
#pragma unroll
      for (int i = 0; i < 9; ++i) r.wv[i] = *reinterpret_cast<const f32x4*>(wsrc + 4 * i);
    } else {
      // W[oc][c0 + j][0..9] is 4-byte aligned; the compiler merges the nine loads.
      r.wv[0] = f32x4{wsrc[0], wsrc[1], wsrc[2], wsrc[3]};
      r.wv[1] = f32x4{wsrc[4], wsrc[5], wsrc[6], wsrc[7]};
      r.wl = wsrc[8];
    }
  };
  auto store_chunk = [&](const Stage& r, int b) __attribute__((always_inline)) {
    // Rows above or below the image are zero padding (a select: the loaded row may hold inf).
    float* dst = in_dst0 + b * kConvLdsBuf;
    auto entry = [&](int i, f32x4 v) __attribute__((always_inline)) {
      *reinterpret_cast<f32x4*>(dst + 4 * i) = in_ok ? v : f32x4{0.f, 0.f, 0.f, 0.f};
    };
    entry(0, f32x4{r.xs[0].x, r.xs[1].x, r.xs[2].x, r.xs[3].x});
    entry(1, f32x4{r.xs[0].y, r.xs[1].y, r.xs[2].y, r.xs[3].y});
    if constexpr (kXW == 4) {
      entry(2, f32x4{r.xs[0].z, r.xs[1].z, r.xs[2].z, r.xs[3].z});
      entry(3, f32x4{r.xs[0].w, r.xs[1].w, r.xs[2].w, r.xs[3].w});
    }
    // Output channels past Oc get zero weights.
    float* wdst = w_dst0 + b * kConvLdsBuf;
    if constexpr (PT == 1) {
      // Flat float i of wv is W[oc][c0 + 4 h + i / 9][i % 9].
      auto f = [&](int i) { return r.wv[i >> 2][i & 3]; };
#pragma unroll
      for (int t = 0; t < 9; ++t)
        *reinterpret_cast<f32x4*>(wdst + 8 * t) =
            w_ok ? f32x4{f(t), f(9 + t), f(18 + t), f(27 + t)} : f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const float v = t < 4 ? r.wv[0][t & 3] : t < 8 ? r.wv[1][t & 3] : r.wl;  // t is a constant here
        wdst[8 * t] = w_ok ? v : 0.f;
      }
    }
  };

  // This lane's pixel (column of the MFMA tile) and k half.
  const int pix = p0 + 32 * ph + (lane & 31);
  const bool pvalid = pix < P;
  const int prow = pvalid ? pix / a.Wo - r0 : 0, pcol = pvalid ? pix % a.Wo : 0;
  const int kk = lane >> 5;
  const int xbase = ((kk * kLdsRows + prow) * kLdsCols + pcol) * 4;  // tap (0, 0), this lane's quad
  const int wbase = kXlFloats + (oh * 32 + (lane & 31)) * kWPitch + 4 * kk;

  f32x16 acc[4] = {f32x16{}, f32x16{}, f32x16{}, f32x16{}};
  auto multiply = [&](const float* cur, int t0, int t1) __attribute__((always_inline)) {
#pragma unroll
    for (int t = t0; t < t1; ++t) {
      const int kh = t / 3, kw = t % 3;
      const f32x4 xv = *reinterpret_cast<const f32x4*>(cur + xbase + (kh * kLdsCols + kw) * 4);
      const f32x4 wv = *reinterpret_cast<const f32x4*>(cur + wbase + t * 8);
      // One accumulator per channel slot j: the four MFMAs of a tap are independent.
      acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv.x, xv.x, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv.y, xv.y, acc[1], 0, 0, 0);
      acc[2] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv.z, xv.z, acc[2], 0, 0, 0);
      acc[3] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv.w, xv.w, acc[3], 0, 0, 0);
    }
  };
  const int chunks = a.C / 8;
  Stage sa, sb;
  load_chunk(sa, 0);
  if constexpr (PT == 2) load_chunk(sb, chunks > 1 ? 8 : 0);
  for (int i = tid; i < 2 * kXlFloats / 4; i += kThreads) {  // zero padding in both input buffers
    const int b = i / (kXlFloats / 4), e = i % (kXlFloats / 4);
    *reinterpret_cast<f32x4*>(lds + b * kConvLdsBuf + 4 * e) = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  __syncthreads();
  store_chunk(sa, 0);
  __syncthreads();
  // In both schedules below every load and store of the loop is unconditional: a store after the
  // last chunk writes a buffer nobody reads, and loads past the last chunk repeat it. A load or
  // store under a branch lets the compiler sink loads behind the MFMAs, or makes its wait
  // counting (which cannot tell that a skipped step also leaves the loop) wait for loads that
  // should stay in flight. The other buffer's last readers (chunk k - 1) all passed the previous
  // barrier when chunk k + 1 is written to it.
  if constexpr (PT == 2) {
    // Two chunks ahead: chunk k's `mine` set (already in LDS) takes chunk k + 2's loads and
    // `next` (chunk k + 1, loaded during chunk k - 1) is written between chunk k's MFMAs. The
    // input streams from HBM and one chunk's MFMAs do not cover its load latency. With an odd
    // chunk count the last step (k = chunks) only repeats loads and a store.
    auto step = [&](int k, Stage& mine, const Stage& next) __attribute__((always_inline)) {
      load_chunk(mine, 8 * (k + 2 < chunks ? k + 2 : chunks - 1));
      __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the MFMAs
      if (k < chunks) multiply(lds + (k & 1) * kConvLdsBuf, 0, kMidTap);
      __builtin_amdgcn_sched_barrier(0);  // no use of the loaded registers ahead of the MFMAs
      store_chunk(next, (k + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
      if (k < chunks) multiply(lds + (k & 1) * kConvLdsBuf, kMidTap, 9);
      if (k + 1 < chunks) __syncthreads();
    };
    for (int k = 0; k < chunks; k += 2) {
      step(k, sa, sb);
      step(k + 1, sb, sa);
    }
  } else {
    // One chunk ahead (a second register set would cost the second workgroup per CU); the
    // store follows all of the chunk's MFMAs (writing it halfway through, before its loads have
    // had a whole chunk to land, measured slower).
    for (int k = 0; k < chunks; ++k) {
      load_chunk(sa, 8 * (k + 1 < chunks ? k + 1 : k));
      __builtin_amdgcn_sched_barrier(0);
      multiply(lds + (k & 1) * kConvLdsBuf, 0, 9);
      __builtin_amdgcn_sched_barrier(0);
      store_chunk(sa, (k + 1) & 1);
      if (k + 1 < chunks) __syncthreads();
    }
  }

  // Epilogue: lane -> pixel (column), rows oc = oc_base + 32 oh + 8 (r / 4) + 4 kk + r % 4.
  if (!pvalid) return;
  float* yb = a.y + (int64_t)n * a.Oc * P;
  float sc[16];  // all scales read before the first store
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int oc = oc_base + oh * 32 + (r >> 2) * 8 + kk * 4 + (r & 3);
    sc[r] = a.scale && oc < a.Oc ? a.scale[oc] : 1.f;
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int oc = oc_base + oh * 32 + (r >> 2) * 8 + kk * 4 + (r & 3);
    if (oc < a.Oc) {
      const float v = (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
      yb[(int64_t)oc * P + pix] = a.scale ? v * sc[r] : v;
    }
  }
}

// conv_lds16_kernel: NCHW, 3x3, stride 1, on v_mfma_f32_16x16x4f32 (the f32 rate of the 32x32x2
// form in a quarter of the tile). The output pixels of an image are cut into 16-pixel groups and
// a workgroup owns a contiguous run of G <= 8 groups x 64 output channels; the runs are balanced
// to within one group (the first gp % wpi runs of an image take one more) and sized for one
// workgroup per CU (conv_l16_geom). Whole 32 x 32 tiles
// over the full reduction leave the busiest SIMD two tiles where the average is 1.53 at the
// BASELINE shape (76.6% of the chip); 16-pixel groups leave it 7 where the average is 6.125.
// Eight wavefronts: wavefront w takes output channels 16 (w % 4) .. + 15 of half the run's groups
// (the first ceil(G / 2) or the rest), so the two wavefronts of a SIMD together cover its channel
// tile over the whole run. Per chunk of 16 input channels both operands are staged in LDS as
// 16-byte entries of 4 channels (quads):
//   * input xl[quad][row][col] for the input rows the run touches, zero-padded, kConvL16Pitch
//     entries per row (8 mod 16: a 16-pixel group wrapping onto the next row reads 16 distinct
//     4-bank groups), and
//   * weights wl[tap][quad][oc], quads kL16WQuad entries apart (64 oc + 4: the quads of one
//     8-byte staging write land on distinct banks), so that 16 consecutive output channels are
//     256 contiguous bytes.
// MFMA lane (16 rows or columns, k quarter q = lane / 16): for each tap one ds_read_b128 of each
// operand gives quad q's 4 channels; MFMA j of the tap takes channel 4 q + j, so one read feeds
// four MFMAs per group. The next tap's fragments are read before this tap's MFMAs. The next
// chunk's loads are in registers while the current chunk is multiplied and are written to the
// other buffer after it; one barrier per chunk. (Measured with the staging switched off in a
// copy: the LDS writes, 4-way bank conflicts in both layouts before the padding and the rotation
// below, cost more than the loads.)
constexpr int kL16Rows = kConvL16Rows;
constexpr int kL16Pitch = kConvL16Pitch;
constexpr int kL16WQuad = kConvL16WQuad;          // weight entries per quad
constexpr int kL16WTap = 4 * kL16WQuad;           // weight entries per tap
constexpr int kL16Xl = 4 * kL16Rows * kL16Pitch;  // input entries per buffer
constexpr int kL16Wl = 9 * kL16WTap;              // weight entries per buffer
constexpr int kL16Buf = kL16Xl + kL16Wl;          // 16-byte entries per buffer (65.25 KiB)

// floor(a / d) for 0 <= a < 2^21 and d >= 1 from rd = l16_rcp(d). The hardware reciprocal (the
// compiler emits v_rcp_iflag_f32 for it) is within one ulp, so (a + 0.5) rd is within 1.8e-7
// (relative) of (a + 0.5) / d, whose distance to the nearest integer is at least 0.5 / d: the
// truncation is exact for any a below 2.79e6. Four instructions where an integer division expands
// to about thirty; the launcher keeps every numerator below 2^21.
__device__ __forceinline__ float l16_rcp(int d) { return __builtin_amdgcn_rcpf((float)d); }
__device__ __forceinline__ int l16_div(int a, float rd) { return (int)(((float)a + 0.5f) * rd); }

template <int G>
__device__ __forceinline__ void l16_frags(const f32x4* cur, const int (&xb)[4], int wb, int t, f32x4& av,
                                          f32x4 (&bv)[4]) {
  av = cur[wb + t * kL16WTap];
#pragma unroll
  for (int gi = 0; gi < G; ++gi) bv[gi] = cur[xb[gi] + (t / 3) * kL16Pitch + t % 3];
}

template <int G>
__device__ __forceinline__ void l16_mfma(const f32x4& av, const f32x4 (&bv)[4], f32x4 (&acc)[4]) {
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int gi = 0; gi < G; ++gi) acc[gi] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[c], bv[gi][c], acc[gi], 0, 0, 0);
}

__global__ void __launch_bounds__(512) conv_lds16_kernel(ConvArgs a) {
  // Every argument field the kernel reads, in scalar registers before anything else: left to
  // the compiler, the fields were loaded one by one between the index computations that need
  // them, each load waited for in turn (about 4000 cycles before the first data load issued).
  asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.scale), "s"(a.y), "s"(a.C), "s"(a.H), "s"(a.W), "s"(a.Oc), "s"(a.pad),
               "s"(a.Ho), "s"(a.Wo), "s"(a.wpi), "s"(a.gq), "s"(a.gr), "s"(gridDim.x));
  __shared__ f32x4 lds[2 * kL16Buf];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ot = wave & 3, half = wave >> 2;  // channel tile, half of the run
  const int P = a.Ho * a.Wo;
  // Weight staging: task (oc, channel pair) = (tid / 8, tid % 8) loads the 18 contiguous floats
  // W[oc][c0 + 2 pr .. + 1][0..9] and writes, per tap, the pair as one half of entry
  // wl[t][pr / 2][oc]: every thread carries the same share. Output channels past Oc load
  // channel 0 and write zeros. The first chunk's weight loads go out before any index
  // arithmetic: they need none.
  const int oc_base = blockIdx.y * 64;
  const int woc = tid >> 3, wpr = tid & 7;
  const bool w_ok = oc_base + woc < a.Oc;
  const float* const w_src0 = a.w + ((int64_t)(w_ok ? oc_base + woc : 0) * a.C + 2 * wpr) * 9;
  const int w_dst = kL16Xl + (wpr >> 1) * kL16WQuad + woc;  // entry of tap 0
  struct Stage {
    f32x4 xs[4];
    f32x2 wv[9];
  };
  auto load_w = [&](Stage& r, int c0) __attribute__((always_inline)) {
    const float* wsrc = w_src0 + (int64_t)c0 * 9;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.wv[i] = *reinterpret_cast<const f32x2*>(wsrc + 2 * i);
  };
  Stage st;
  load_w(st, 0);
  __builtin_amdgcn_sched_barrier(0);
  // XCD-aware order: workgroup b runs on XCD b % 8, so XCD x takes a contiguous span of runs
  // (neighbouring runs share input rows in its L2).
  const int NG = gridDim.x, q8 = NG >> 3, r8 = NG & 7, xcd = blockIdx.x & 7;
  const int lin = xcd * q8 + (xcd < r8 ? xcd : r8) + (blockIdx.x >> 3);
  const int n = l16_div(lin, l16_rcp(a.wpi)), j = lin - n * a.wpi;
  const int g0 = j * a.gq + (j < a.gr ? j : a.gr), g1 = g0 + a.gq + (j < a.gr ? 1 : 0);
  const int ga = (g1 - g0 + 1) >> 1;
  const int myg = g0 + (half ? ga : 0);                                      // this wavefront's first group
  const int ng = __builtin_amdgcn_readfirstlane(half ? g1 - g0 - ga : ga);  // its groups, 0..4
  const int pend = (16 * g1 < P ? 16 * g1 : P);
  const float rwo = l16_rcp(a.Wo);
  const int r0 = l16_div(16 * g0, rwo), rlast = l16_div(pend - 1, rwo);
  const int in_rows = rlast - r0 + 3;  // padded input rows r0 - pad .. rlast + 2 - pad
  const int64_t HW = (int64_t)a.H * a.W;
  const float* xn = a.x + (int64_t)n * a.C * HW;

  // Input staging: task (quad, row, 4-column group) loads the quad's four channels at four
  // columns of one input row (a float4 per channel) and writes four entries; threads beyond the
  // task count in a wavefront that has tasks repeat a task's loads but write nothing. The launcher keeps
  // tasks <= 512. Rows outside the image load row 0 and write zeros. Write i of a task goes to
  // column (icg / 4 + i) % 4 of its group: the 16 lanes of one write phase (16 consecutive
  // groups) then hit 16 distinct 4-bank groups instead of 4.
  const int cgs = a.W >> 2;
  const int tasks = 4 * in_rows * cgs;
  const int it = tid - l16_div(tid, l16_rcp(tasks)) * tasks;
  const int iq = l16_div(it, l16_rcp(in_rows * cgs)), itc = l16_div(it, l16_rcp(cgs));
  const int irr = itc - l16_div(itc, l16_rcp(in_rows)) * in_rows, icg = it - itc * cgs;
  const int ihi = r0 + irr - a.pad;
  const bool in_ok = ihi >= 0 && ihi < a.H;
  const bool in_mine = tid < tasks;
  const bool in_wave = __builtin_amdgcn_readfirstlane(tid & ~63) < tasks;  // the wavefront has a task
  const int in_rot = (icg >> 2) & 3;
  const int64_t in_off = (int64_t)4 * iq * HW + (int64_t)(in_ok ? ihi : 0) * a.W + 4 * icg;
  const int in_dst = (iq * kL16Rows + irr) * kL16Pitch + a.pad + 4 * icg;
  auto load_x = [&](Stage& r, int c0) __attribute__((always_inline)) {
    // Wavefronts wholly past the input tasks issue no input loads: issuing the chunk's loads is
    // a cost per load instruction and wavefront, whatever the bytes.
    if (in_wave) {
      const float* src = xn + (int64_t)c0 * HW + in_off;
#pragma unroll
      for (int q = 0; q < 4; ++q) r.xs[q] = *reinterpret_cast<const f32x4*>(src + q * HW);
    }
  };
  auto store_chunk = [&](const Stage& r, int b) __attribute__((always_inline)) {
    if (in_mine) {
      f32x4* xd = lds + b * kL16Buf + in_dst;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = (in_rot + i) & 3;  // column of the group this write covers
        auto pick = [&](const f32x4& v) __attribute__((always_inline)) {
          return c == 0 ? v.x : c == 1 ? v.y : c == 2 ? v.z : v.w;
        };
        const f32x4 e = f32x4{pick(r.xs[0]), pick(r.xs[1]), pick(r.xs[2]), pick(r.xs[3])};
        xd[c] = in_ok ? e : f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    // Flat float k of wv is W[oc][c0 + 2 pr + k / 9][k % 9]; tap t pairs floats t and 9 + t.
    float* wd = reinterpret_cast<float*>(lds + b * kL16Buf + w_dst) + 2 * (wpr & 1);
#pragma unroll
    for (int t = 0; t < 9; ++t) {
      const f32x2 v = f32x2{r.wv[t >> 1][t & 1], r.wv[(9 + t) >> 1][(9 + t) & 1]};
      *reinterpret_cast<f32x2*>(wd + t * kL16WTap * 4) = w_ok ? v : f32x2{0.f, 0.f};
    }
  };

  auto load_chunk = [&](Stage& r, int c0) __attribute__((always_inline)) {
    load_w(r, c0);
    load_x(r, c0);
  };
  // The first chunk's input loads go out before the lane geometry below is computed.
  const int chunks = a.C >> 4;
  load_x(st, 0);

  // MFMA lane roles: pixel or output channel lane & 15, k quarter (channel quad) lane >> 4.
  const int px = lane & 15, kq = lane >> 4;
  int xb[4];
#pragma unroll
  for (int gi = 0; gi < 4; ++gi) {
    const int p = 16 * (myg + gi) + px;
    const bool ok = gi < ng && p < pend;
    const int pr = l16_div(p, rwo);
    xb[gi] = (kq * kL16Rows + (ok ? pr - r0 : 0)) * kL16Pitch + (ok ? p - pr * a.Wo : 0);
  }
  const int wb = kL16Xl + kq * kL16WQuad + ot * 16 + px;
  // This lane's four output-channel scales, read now: at the end of the kernel they were a cold
  // read behind every workgroup's traffic (about 3 us), here they land during the first chunk.
  float sc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int oc = oc_base + 16 * ot + 4 * kq + i;
    sc[i] = a.scale && oc < a.Oc ? a.scale[oc] : 1.f;
  }
  f32x4 acc[4] = {};

  // Zero padding: the MFMA reads of a staged row span columns 0 .. W + 2 pad - 1 and the staging
  // writes columns pad .. pad + W - 1, so only the pad columns (0 and W + 1, pad = 1) need zeros:
  // 2 buffers x 2 sides x 4 quads x kL16Rows rows. Rows past the run's staged rows are never
  // read. These entries are disjoint from the staging writes, so one barrier after both suffices.
  if (a.pad && tid < 2 * 2 * 4 * kL16Rows) {
    const int b = tid / (2 * 4 * kL16Rows), side = (tid / (4 * kL16Rows)) & 1, qr = tid % (4 * kL16Rows);
    lds[b * kL16Buf + qr * kL16Pitch + (side ? a.W + 1 : 0)] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  store_chunk(st, 0);
  __syncthreads();
  // Every load of the loop is unconditional, so the compiler's wait counting keeps the loads in
  // flight across the MFMAs; the last chunk is multiplied after the loop with no loads or LDS
  // writes (a final step that repeated the loads and wrote a buffer nobody reads cost their issue
  // and writes just before the epilogue). Buffer (k + 1) & 1 was last read in chunk k - 1, whose
  // readers all passed the previous barrier. Per tap: the next tap's fragment reads, then this
  // tap's MFMAs.
  auto multiply = [&]<int G>(int k) __attribute__((always_inline)) {
    if constexpr (G > 0) {
      const f32x4* cur = lds + (k & 1) * kL16Buf;
      f32x4 av[2], bv[2][4];
      l16_frags<G>(cur, xb, wb, 0, av[0], bv[0]);
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        if (t + 1 < 9) l16_frags<G>(cur, xb, wb, t + 1, av[(t + 1) & 1], bv[(t + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
        l16_mfma<G>(av[t & 1], bv[t & 1], acc);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  auto run = [&]<int G>() __attribute__((always_inline)) {
    for (int k = 0; k + 1 < chunks; ++k) {
      load_chunk(st, 16 * (k + 1));
      __builtin_amdgcn_sched_barrier(0);
      multiply.template operator()<G>(k);
      store_chunk(st, (k + 1) & 1);
      __syncthreads();
    }
    multiply.template operator()<G>(chunks - 1);
  };
  switch (ng) {
    case 4: run.template operator()<4>(); break;
    case 3: run.template operator()<3>(); break;
    case 2: run.template operator()<2>(); break;
    case 1: run.template operator()<1>(); break;
    default: run.template operator()<0>(); break;
  }

  // Epilogue: lane -> pixel (column), rows oc = oc_base + 16 ot + 4 kq + i (scales read at the
  // start).
  float* yb = a.y + (int64_t)n * a.Oc * P;
  if (((P & 3) | (((uintptr_t)a.y) & 15)) == 0) {
    // Through this wavefront's own 16 x kL16TPitch tile in the buffer the last chunk did not use
    // (its last readers passed the last barrier; nobody writes it after that barrier): four
    // 16-byte stores of four consecutive pixels per lane instead of sixteen 4-byte stores. Rows
    // kL16TPitch = 68 floats apart put the 64 lanes of each 4-byte write on distinct banks. With
    // P a multiple of 4 the run's end is too, so every float4 is whole or wholly outside.
    constexpr int kL16TPitch = 68;
    float* tw = reinterpret_cast<float*>(lds + (chunks & 1) * kL16Buf) + wave * (16 * kL16TPitch);
#pragma unroll
    for (int gi = 0; gi < 4; ++gi) {
      if (gi >= ng) break;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        tw[(4 * kq + i) * kL16TPitch + 16 * gi + px] = a.scale ? acc[gi][i] * sc[i] : acc[gi][i];
    }
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const int f = 64 * s4 + lane, ocl = f >> 4, q = f & 15, gi = q >> 2;
      const int p = 16 * (myg + gi) + 4 * (q & 3), oc = oc_base + 16 * ot + ocl;
      const f32x4 v = *reinterpret_cast<const f32x4*>(tw + ocl * kL16TPitch + 4 * q);
      if (gi < ng && p < pend && oc < a.Oc) *reinterpret_cast<f32x4*>(yb + (int64_t)oc * P + p) = v;
    }
    return;
  }
#pragma unroll
  for (int gi = 0; gi < 4; ++gi) {
    const int p = 16 * (myg + gi) + px;
    if (gi >= ng || p >= pend) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int oc = oc_base + 16 * ot + 4 * kq + i;
      if (oc < a.Oc) yb[(int64_t)oc * P + p] = a.scale ? acc[gi][i] * sc[i] : acc[gi][i];
    }
  }
}

}  // namespace uk::kern

namespace uk {

namespace {
template <bool NCHW, int TAPS, int WAVES>
hipError_t conv_go(const kern::ConvArgs& a, int64_t units, int oc_tiles, size_t lds, hipStream_t s) {
  const unsigned grid = (unsigned)((units + WAVES - 1) / WAVES);
  if (!grid_dim_holds(grid, WAVES * 64)) return hipErrorInvalidValue;
  // Dynamic LDS above the default limit must be requested per kernel (once).
  static hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&kern::conv_igemm_kernel<NCHW, TAPS, WAVES>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 163840);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((kern::conv_igemm_kernel<NCHW, TAPS, WAVES>), dim3(grid, (unsigned)oc_tiles), dim3(WAVES * 64),
                     lds, s, a);
  return hipGetLastError();
}

template <bool NCHW, int WAVES>
hipError_t conv_taps(const kern::ConvArgs& a, int64_t units, int oc_tiles, size_t lds, hipStream_t s) {
  const int taps = a.Kh * a.Kw;
  if (taps == 9) return conv_go<NCHW, 9, WAVES>(a, units, oc_tiles, lds, s);
  if (taps == 1) return conv_go<NCHW, 1, WAVES>(a, units, oc_tiles, lds, s);
  return conv_go<NCHW, 0, WAVES>(a, units, oc_tiles, lds, s);
}
}  // namespace

namespace {
template <bool NCHW, int TAPS, int S, int CB>
hipError_t conv_tile_go(const kern::ConvArgs& a, int64_t units, int oc_tiles, hipStream_t s) {
  const unsigned grid = (unsigned)((units + S - 1) / S);
  if (!grid_dim_holds(grid, S * 128)) return hipErrorInvalidValue;
  hipLaunchKernelGGL((kern::conv_tile_kernel<NCHW, TAPS, S, CB>), dim3(grid, (unsigned)oc_tiles), dim3(S * 128), 0,
                     s, a);
  return hipGetLastError();
}
template <int S, int CB>
hipError_t conv_tile_dispatch(bool nchw, int taps, const kern::ConvArgs& a, int64_t units, int oc_tiles,
                              hipStream_t s) {
  if (taps == 9)
    return nchw ? conv_tile_go<true, 9, S, CB>(a, units, oc_tiles, s) : conv_tile_go<false, 9, S, CB>(a, units, oc_tiles, s);
  if (taps == 1)
    return nchw ? conv_tile_go<true, 1, S, CB>(a, units, oc_tiles, s) : conv_tile_go<false, 1, S, CB>(a, units, oc_tiles, s);
  return hipErrorInvalidValue;
}
}  // namespace

hipError_t launch_conv_igemm(const Plan& p, const Shape& sh, Layout lay, const float* X, const float* Wt,
                             const float* scale, float* Y, hipStream_t s) {
  if (p.family != Family::ConvIgemm || p.variant < 0 || p.variant >= kNumConvVariants + kNumConvAnyVariants)
    return hipErrorInvalidValue;
  if (p.variant >= kNumConvVariants) return launch_conv_any(p.variant - kNumConvVariants, sh, lay, X, Wt, scale, Y, s);
  const ConvVariant v = kConvVariants[p.variant];
  const bool nchw = lay == Layout::NCHW;
  if (!nchw && lay != Layout::NT) return hipErrorInvalidValue;
  if (sh.Ho <= 0 || sh.Wo <= 0 || sh.Ci <= 0 || sh.Co <= 0 || sh.Kh <= 0 || sh.Kw <= 0) return hipErrorInvalidValue;
  const int64_t taps = sh.Kh * sh.Kw;
  if (taps > 49) return hipErrorInvalidValue;  // per-lane tap table
  // Input offsets and plane sizes are 32-bit inside the kernel.
  if (sh.H * sh.W * sh.Ci > INT32_MAX || sh.Ho * sh.Wo > INT32_MAX || sh.Nb * sh.Ci * sh.H * sh.W > (int64_t(1) << 40))
    return hipErrorInvalidValue;
  kern::ConvArgs a;
  a.x = X;
  a.w = Wt;
  a.scale = scale;
  a.y = Y;
  a.N = (int)sh.Nb;
  a.C = (int)sh.Ci;
  a.H = (int)sh.H;
  a.W = (int)sh.W;
  a.Oc = (int)sh.Co;
  a.Kh = (int)sh.Kh;
  a.Kw = (int)sh.Kw;
  a.pad = (int)sh.pad;
  a.stride = (int)sh.stride;
  a.Ho = (int)sh.Ho;
  a.Wo = (int)sh.Wo;
  a.strips = (int)((sh.Ho * sh.Wo + 31) / 32);
  if (v.tile_strips == kConvL16) {  // conv_lds16_kernel: 16-pixel groups, runs balanced over the CUs
    if (!conv_l16_supported(nchw, sh.Kh, sh.Kw, sh.stride, sh.pad, sh.Nb, sh.W, sh.Ho, sh.Wo, sh.Ci, sh.Co))
      return hipErrorInvalidValue;
    if ((((uintptr_t)X) | ((uintptr_t)Wt)) & 15) return hipErrorInvalidValue;
    const ConvL16Geom g = conv_l16_geom(sh.Nb, sh.Ho, sh.Wo, (sh.Co + 63) / 64);
    const int64_t oc_blocks = (sh.Co + 63) / 64;
    // Input staging tasks (4 quads x rows x W / 4 columns) fit the 512 threads.
    if (4 * kConvL16Rows * (sh.W / 4) > 512 || !grid_dim_holds(sh.Nb * g.wpi, 512) || oc_blocks > 65535)
      return hipErrorInvalidValue;
    a.gp = (int)g.gp;
    a.wpi = (int)g.wpi;
    a.gq = (int)(g.gp / g.wpi);
    a.gr = (int)(g.gp % g.wpi);
    hipLaunchKernelGGL(kern::conv_lds16_kernel, dim3((unsigned)(sh.Nb * g.wpi), (unsigned)oc_blocks), dim3(512), 0, s,
                       a);
    return hipGetLastError();
  }
  if (v.tile_strips < 0) {  // conv_lds_kernel: NCHW 3x3 stride 1, both operands staged in LDS
    const int pt = -v.tile_strips;
    if (pt != 1 && pt != 2) return hipErrorInvalidValue;
    if (!conv_lds_supported(nchw, sh.Kh, sh.Kw, sh.stride, sh.pad, sh.W, sh.Ho, sh.Wo, sh.Ci, 64 * pt))
      return hipErrorInvalidValue;
    if ((((uintptr_t)X) | ((uintptr_t)Wt)) & 15) return hipErrorInvalidValue;
    const int64_t tiles = (sh.Ho * sh.Wo + 64 * pt - 1) / (64 * pt);
    const int oc_tiles = (int)((sh.Co + 63) / 64);
    if (!grid_dim_holds(sh.Nb * tiles, 256 * pt) || oc_tiles > 65535) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(sh.Nb * tiles), (unsigned)oc_tiles);
    if (pt == 1) hipLaunchKernelGGL(kern::conv_lds_kernel<1>, grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL(kern::conv_lds_kernel<2>, grid, dim3(512), 0, s, a);
    return hipGetLastError();
  }
  if (v.tile_strips > 0) {  // 32 x 32 wavefront tiles, chunked coalesced weight staging
    if (taps != 9 && taps != 1) return hipErrorInvalidValue;
    a.cb = v.bk_bytes;  // channels per chunk
    const int64_t units = sh.Nb * a.strips;
    const int oc_tiles = (int)((sh.Co + 63) / 64);
    if ((units + v.tile_strips - 1) / v.tile_strips > INT32_MAX || oc_tiles > 65535) return hipErrorInvalidValue;
    if (v.tile_strips == 2 && v.bk_bytes == 16) return conv_tile_dispatch<2, 16>(nchw, (int)taps, a, units, oc_tiles, s);
    if (v.tile_strips == 2 && v.bk_bytes == 8) return conv_tile_dispatch<2, 8>(nchw, (int)taps, a, units, oc_tiles, s);
    if (v.tile_strips == 4 && v.bk_bytes == 8) return conv_tile_dispatch<4, 8>(nchw, (int)taps, a, units, oc_tiles, s);
    return hipErrorInvalidValue;
  }
  // Channel chunk: as many (even) channels as the LDS budget of the variant allows.
  const int64_t per_channel = taps * 64 * 4;
  int64_t cb = v.bk_bytes / per_channel;
  cb &= ~int64_t(1);
  if (cb < 2) return hipErrorInvalidValue;
  const int64_t cpad = (sh.Ci + 1) & ~int64_t(1);
  if (cb > cpad) cb = cpad;
  a.cb = (int)cb;
  const size_t lds = (size_t)(cb * per_channel);
  const int64_t units = sh.Nb * a.strips;
  const int oc_tiles = (int)((sh.Co + 63) / 64);
  if ((units + v.waves - 1) / v.waves > INT32_MAX || oc_tiles > 65535) return hipErrorInvalidValue;
  switch (v.waves) {
    case 2: return nchw ? conv_taps<true, 2>(a, units, oc_tiles, lds, s) : conv_taps<false, 2>(a, units, oc_tiles, lds, s);
    case 4: return nchw ? conv_taps<true, 4>(a, units, oc_tiles, lds, s) : conv_taps<false, 4>(a, units, oc_tiles, lds, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace uk
