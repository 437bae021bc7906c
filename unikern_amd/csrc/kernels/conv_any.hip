// conv2d of any kernel size (up to 49 taps), stride, padding and channel count as an implicit GEMM on
// f32 matrix cores: Y[oc][pixel] = scale[oc] * sum_k W[oc][k] * X_im2col[k][pixel] (reference
// src/codegen_hip.cpp:337-411, its separate channelscale :2329-2335), in both layouts of conv.hip.
//
// conv_any_kernel is gemm_any.hip's tile (weights as A, both operands' 32-k segments in swizzled
// 128-byte LDS rows, operands stored before the multiply, loads a step ahead) with the input gathered
// into the B rows: k runs in the order the layout stores a weight row, so the weights load as they lie.
// A table of the input offset of every (tap, pixel) of the tile, -1 in the padding, is built in LDS
// once per workgroup. MODE 0 (NCHW) and 2 (HWC): lane = pixel and the k of a load are uniform, so the
// channel is scalar arithmetic and the 64 lanes read neighbouring pixels. MODE 1 (HWC, C a multiple of 4,
// no padding): four channels of a pixel are one 16-byte load, eight lanes to a 128-byte row segment.
//
// Why: the gathering kernels (conv_igemm, conv_tile) load every input element straight into the MFMA
// operands of each wavefront that needs it, one load per MFMA; here a tile's input is loaded once
// and an element costs one load instead of one per 32 output channels. Bound by the f32 MFMA of the CU (0.62 of
// its cycles at HWC 256x256x32, 14 of 16 wavefronts resident: the fill at the start, when every tile
// builds its table and loads, and the stores at the end are the rest) and, in NCHW, by the gather's loads.
// HWC 256x256x32, 3x3, 64 channels: 89.7 -> 26.5 us (90 TFLOP/s, 57% of the f32 MFMA
// peak; 29.0 from HBM); NCHW 8x64x56x56 stride 2 53.8 -> 17.3, 8x64x56x56 1x1 to 256 56.2 -> 20.7, 8x256x14x14 3x3
// 174 -> 54.5, 4x3x112x112 7x7 stride 2 35.9 -> 11.9. NCHW 3x3 stride 1 of aligned rows stays on the
// kernels that stage whole input rows (conv_lds16: 20.7 us at 8x64x56x56, 36.0 here).
#include "../launch.hpp"
#include "../variants.hpp"
#include "common.hpp"
#include "tile.hpp"

#include <type_traits>
#include <utility>

namespace uk::kern {

struct ConvAnyArgs {
  const float* x;
  const float* w;
  const float* scale;
  float* y;
  int C, H, W, Oc, Kw, pad, stride, Wo;
  int taps, P, K;          // Kh Kw, Ho Wo, C taps
  int inner;               // k = outer * inner + rest: taps (NCHW) or C (HWC)
  unsigned magic;          // ceil(2^32 / inner): k / inner = mulhi(k, magic) (inner > 1)
  int tiles_m, tiles_n;    // tiles of output channels and of one image's pixels
  int tiles;               // of all images
  int64_t xstep, ystep;    // floats of one image of X and Y
};

template <int BM, int BN, int WM, int WN, int S>
struct ConvAnyCfg {
  static constexpr int kGroup = WM * WN * 64;
  static constexpr int kThreads = kGroup * S;
  static constexpr int kFM = BM / WM / 16, kFN = BN / WN / 16;
  static constexpr int kNA = BM * 8 / kGroup, kNB = BN * 8 / kGroup;
  static constexpr int kSlot = (BM + BN) * 128;
  static constexpr int kPitch = BN / WN + 4;  // floats
  static constexpr int kPipe = 2 * S * kSlot;
  static constexpr int kRed = (S - 1) * BM * BN * 4;
  static constexpr int kStage = WM * WN * (BM / WM) * kPitch * 4;
  static constexpr int kMax = kPipe > kRed ? (kPipe > kStage ? kPipe : kStage) : (kRed > kStage ? kRed : kStage);
};

template <int MODE, int BM, int BN, int WM, int WN, int S, bool PAD>
__global__ void __launch_bounds__(WM* WN* S * 64, 4)
    conv_any_kernel(ConvAnyArgs a) {
  using Cfg = ConvAnyCfg<BM, BN, WM, WN, S>;
  constexpr int FM = Cfg::kFM, FN = Cfg::kFN, NA = Cfg::kNA, NB = Cfg::kNB;
  constexpr int KT_ELEMS = S * 32;
  asm volatile("" ::"s"(a.x), "s"(a.w), "s"(a.y), "s"(a.C), "s"(a.H), "s"(a.W), "s"(a.Oc), "s"(a.P), "s"(a.K), "s"(a.inner),
               "s"(a.magic));
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  int* const tab = reinterpret_cast<int*>(lds + Cfg::kMax);  // [taps][BN]: offset of (pixel, tap), -1: padding
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = w / (WM * WN), wg = w % (WM * WN), wm = wg / WN, wn = wg % WN;
  const int tg = tid - kh * Cfg::kGroup;

  const int per_image = a.tiles_m * a.tiles_n;
  const int id = folded_id();
  if (id >= a.tiles) return;
  const int image = id / per_image, in_image = id - image * per_image;
  const int m0 = in_image % a.tiles_m * BM, n0 = in_image / a.tiles_m * BN;
  const float* const xb = a.x + image * a.xstep;

  // Offset table: a thread's pixel is fixed, its taps tid / BN, tid / BN + threads / BN, ...
  {
    static_assert(Cfg::kThreads % BN == 0, "a thread's pixel is fixed");
    const int pix = tid % BN;
    const int p = n0 + pix < a.P ? n0 + pix : a.P - 1;
    const int ho = p / a.Wo, wo = p - ho * a.Wo;
    for (int t = tid / BN; t < a.taps; t += Cfg::kThreads / BN) {
      const int y = t / a.Kw, x = t - y * a.Kw;
      const int hi = ho * a.stride + y - a.pad, wi = wo * a.stride + x - a.pad;
      const int o = MODE == 0 ? hi * a.W + wi : (hi * a.W + wi) * a.C;
      tab[t * BN + pix] = !PAD || (hi >= 0 && hi < a.H && wi >= 0 && wi < a.W) ? o : -1;
    }
  }

  const int crow = tg >> 3, cc = tg & 7;
  const float* arow[NA];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int r = m0 + u * (Cfg::kGroup / 8) + crow;
    arow[u] = a.w + (int64_t)(r < a.Oc ? r : a.Oc - 1) * a.K;
  }
  // Scalar gather (MODE 0, 2): lane = pixel, a wavefront's chunks (four consecutive k) are uniform.
  constexpr int kPixWaves = BN / 64;
  static_assert(BN % 64 == 0 && (WM * WN) % kPixWaves == 0, "wavefronts tile the pixels");
  constexpr int kChunkWaves = WM * WN / kPixWaves;
  const int gpix = (wg % kPixWaves) * 64 + lane, gchunk = wg / kPixWaves;

  const int whole_steps = a.K / KT_ELEMS;
  u32x4 ra[NA], rb[NB];
  uint32_t bad = 0;  // PAD: bit 4 u + e: element e of chunk u lies in the padding
  auto split = [&](int k, int& outer, int& rest) __attribute__((always_inline)) {
    outer = a.inner == 1 ? k : (int)__umulhi((unsigned)k, a.magic);
    rest = k - outer * a.inner;
  };
  auto load = [&]<bool TAIL>(int t) __attribute__((always_inline)) {
    const int k0 = t * KT_ELEMS + kh * 32;
#pragma unroll
    for (int u = 0; u < NA; ++u)
      ra[u] = TAIL ? any_load16_edge(arow[u], k0 + cc * 4, a.K) : any_load16(arow[u] + k0 + cc * 4);
    if constexpr (MODE == 1) {
      int tap, c;
      const int k = !TAIL || k0 + cc * 4 < a.K ? k0 + cc * 4 : 0;
      split(k, tap, c);
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const unsigned o = (unsigned)(tab[tap * BN + u * (Cfg::kGroup / 8) + crow] + c) * 4u;
        rb[u] = any_load16(reinterpret_cast<const char*>(xb) + o);
      }
    } else {
      if constexpr (PAD) bad = 0;
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int kc = k0 + 4 * (gchunk + u * kChunkWaves);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = !TAIL || kc + e < a.K ? kc + e : 0;
          int outer, rest;
          split(k, outer, rest);
          const int o = tab[(MODE == 0 ? rest : outer) * BN + gpix];
          const float* base = MODE == 0 ? xb + (int64_t)outer * a.H * a.W : xb + rest;
          const unsigned off = (unsigned)(PAD && o < 0 ? 0 : o) * 4u;
          rb[u][e] = *reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(base) + off);
          if constexpr (PAD) bad |= (o < 0 ? 1u : 0u) << (4 * u + e);
        }
      }
    }
  };
  auto store = [&]<bool TAIL>(int slot) __attribute__((always_inline)) {
    char* as = lds + (slot * S + kh) * Cfg::kSlot;
    char* bs = as + BM * 128;
    const int k0 = whole_steps * KT_ELEMS + kh * 32;  // of the tail
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const int r = u * (Cfg::kGroup / 8) + crow;
      *reinterpret_cast<u32x4*>(as + r * 128 + ((cc ^ ((r >> 1) & 7)) << 4)) = ra[u];
    }
    if constexpr (MODE == 1) {
      if (TAIL && k0 + cc * 4 >= a.K) {  // K is a multiple of 4: chunks past it are whole
#pragma unroll
        for (int u = 0; u < NB; ++u) rb[u] = u32x4{0, 0, 0, 0};
      }
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int r = u * (Cfg::kGroup / 8) + crow;
        *reinterpret_cast<u32x4*>(bs + r * 128 + ((cc ^ ((r >> 1) & 7)) << 4)) = rb[u];
      }
    } else {
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int c = gchunk + u * kChunkWaves;
        u32x4 v = rb[u];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (PAD && (bad >> (4 * u + e) & 1)) v[e] = 0;
          if (TAIL && k0 + 4 * c + e >= a.K) v[e] = 0;
        }
        *reinterpret_cast<u32x4*>(bs + gpix * 128 + ((c ^ ((gpix >> 1) & 7)) << 4)) = v;
      }
    }
  };
  const int fi = lane & 15, fg = lane >> 4;
  // Summation in blocks: the even and the odd pairs of k of a chunk run apart (as the gathered kernels' channel
  // pairs do) over eight steps, then go into `acc`. Against 64 bits no further off than those kernels at any
  // K (2.0e-7 against 2.2e-7 at K = 288); with halves of a segment apart over all of K, 1.2 times at K <= 16.
  f32x4 part[2][FM][FN], acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = part[0][i][j] = part[1][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto fold = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] += part[0][i][j][r] + part[1][i][j][r];
        part[0][i][j] = part[1][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  auto multiply = [&](int slot) __attribute__((always_inline)) {
    const char* as = lds + (slot * S + kh) * Cfg::kSlot + (wm * (BM / WM) + fi) * 128;
    const char* bs = lds + (slot * S + kh) * Cfg::kSlot + BM * 128 + (wn * (BN / WN) + fi) * 128;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int c = ((4 * ks + fg) ^ ((fi >> 1) & 7)) << 4;
      u32x4 fa[FM], fb[FN];
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[j] = *reinterpret_cast<const u32x4*>(bs + j * 16 * 128 + c);
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[i] = *reinterpret_cast<const u32x4*>(as + i * 16 * 128 + c);
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const f32x4 b = __builtin_bit_cast(f32x4, fb[j]), a = __builtin_bit_cast(f32x4, fa[i]);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            f32x4& sum = part[e >> 1][i][j];
            sum = __builtin_amdgcn_mfma_f32_16x16x4f32(b[e], a[e], sum, 0, 0, 0);
          }
        }
    }
  };

  // Step t: its operands sit in slot t % 2; the next step's go into the other slot, the loads after that
  // are issued (past the last whole step they repeat it, so that no branch surrounds a load), and only
  // then does it multiply. The partial last step, if any, follows by itself.
  __syncthreads();  // the table
  if (whole_steps > 0) {
    load.template operator()<false>(0);
    store.template operator()<false>(0);
    load.template operator()<false>(whole_steps > 1 ? 1 : 0);
    lds_barrier();
    for (int t = 0; t < whole_steps;) {
      for (const int end = t + 8 < whole_steps ? t + 8 : whole_steps; t < end; ++t) {
        store.template operator()<false>((t + 1) & 1);
        load.template operator()<false>(t + 2 < whole_steps ? t + 2 : whole_steps - 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(t & 1);
        lds_barrier();
      }
      fold();
    }
  }
  if (whole_steps * KT_ELEMS < a.K) {
    load.template operator()<true>(whole_steps);
    store.template operator()<true>(0);
    lds_barrier();
    multiply(0);
    fold();
    lds_barrier();
  }

  if constexpr (S > 1) {
    f32x4* red = reinterpret_cast<f32x4*>(lds);
    if (kh > 0) {
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) red[(((kh - 1) * FM + i) * FN + j) * Cfg::kGroup + tg] = acc[i][j];
    }
    __syncthreads();
    if (kh == 0) {
#pragma unroll
      for (int s = 0; s < S - 1; ++s)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const f32x4 p = red[((s * FM + i) * FN + j) * Cfg::kGroup + tg];
            acc[i][j] = f32x4{acc[i][j][0] + p[0], acc[i][j][1] + p[1], acc[i][j][2] + p[2], acc[i][j][3] + p[3]};
          }
    }
    __syncthreads();
    if (kh > 0) return;
  }
  const int mw = m0 + wm * (BM / WM), nw = n0 + wn * (BN / WN);
  float* stage = reinterpret_cast<float*>(lds) + wg * (BM / WM) * Cfg::kPitch;
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int oc = mw + i * 16 + fi;
    const float s = a.scale && oc < a.Oc ? a.scale[oc] : 1.f;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const f32x4 v = acc[i][j];
      *reinterpret_cast<f32x4*>(stage + (i * 16 + fi) * Cfg::kPitch + j * 16 + 4 * fg) =
          a.scale ? f32x4{v[0] * s, v[1] * s, v[2] * s, v[3] * s} : v;
    }
  }
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int kRowChunks = BN / WN / 4;
  float* const yb = a.y + image * a.ystep;
#pragma unroll 4
  for (int id = lane; id < BM / WM * kRowChunks; id += 64) {
    const int r = id / kRowChunks, q = id % kRowChunks;
    const int m = mw + r, n = nw + q * 4;
    if (m >= a.Oc || n >= a.P) continue;
    const f32x4 v = *reinterpret_cast<const f32x4*>(stage + r * Cfg::kPitch + q * 4);
    float* dst = yb + (int64_t)m * a.P + n;
    if (a.P - n >= 4) {
      __builtin_memcpy(dst, &v, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (e < a.P - n) dst[e] = v[e];
    }
  }
}

}  // namespace uk::kern

namespace uk {
namespace {
template <int MODE, int BM, int BN, int WM, int WN, int S, bool PAD>
hipError_t conv_any_go(const kern::ConvAnyArgs& a, hipStream_t s) {
  using Cfg = kern::ConvAnyCfg<BM, BN, WM, WN, S>;
  static hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(&kern::conv_any_kernel<MODE, BM, BN, WM, WN, S, PAD>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, 163840);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL((kern::conv_any_kernel<MODE, BM, BN, WM, WN, S, PAD>), folded_grid(a.tiles), dim3(Cfg::kThreads),
                     Cfg::kMax + a.taps * BN * 4, s, a);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_conv_any(int variant, const Shape& sh, Layout lay, const float* X, const float* Wt, const float* scale,
                           float* Y, hipStream_t s) {
  if (variant < 0 || variant >= kNumConvAnyVariants) return hipErrorInvalidValue;
  const ConvAnyVariant v = kConvAnyVariants[variant];
  const bool nchw = lay == Layout::NCHW;
  if (!conv_any_supported(nchw, sh.Nb, sh.Ci, sh.H, sh.W, sh.Co, sh.Kh, sh.Kw, sh.Ho, sh.Wo)) return hipErrorInvalidValue;
  kern::ConvAnyArgs a{};
  a.x = X;
  a.w = Wt;
  a.scale = scale;
  a.y = Y;
  a.C = (int)sh.Ci;
  a.H = (int)sh.H;
  a.W = (int)sh.W;
  a.Oc = (int)sh.Co;
  a.Kw = (int)sh.Kw;
  a.pad = (int)sh.pad;
  a.stride = (int)sh.stride;
  a.Wo = (int)sh.Wo;
  a.taps = (int)(sh.Kh * sh.Kw);
  a.P = (int)(sh.Ho * sh.Wo);
  a.K = (int)(sh.Ci * a.taps);
  a.inner = nchw ? a.taps : a.C;
  a.magic = a.inner > 1 ? (unsigned)(((uint64_t(1) << 32) + a.inner - 1) / a.inner) : 0;
  a.tiles_m = (int)((sh.Co + v.bm - 1) / v.bm);
  a.tiles_n = (int)((a.P + v.bn - 1) / v.bn);
  a.xstep = sh.Ci * sh.H * sh.W;
  a.ystep = sh.Co * int64_t(a.P);
  const int64_t grid = sh.Nb * a.tiles_m * int64_t(a.tiles_n);
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  a.tiles = (int)grid;
  const bool pad = sh.pad != 0;
  const bool vec = !nchw && sh.Ci % 4 == 0 && !pad;
  hipError_t e = hipErrorInvalidValue;
  auto go = [&](auto i_c) {
    constexpr ConvAnyVariant c = kConvAnyVariants[decltype(i_c)::value];
    if (nchw)
      e = pad ? conv_any_go<0, c.bm, c.bn, c.wm, c.wn, c.ks, true>(a, s)
              : conv_any_go<0, c.bm, c.bn, c.wm, c.wn, c.ks, false>(a, s);
    else if (vec)
      e = conv_any_go<1, c.bm, c.bn, c.wm, c.wn, c.ks, false>(a, s);
    else
      e = conv_any_go<2, c.bm, c.bn, c.wm, c.wn, c.ks, true>(a, s);
  };
  [&]<int... Is>(std::integer_sequence<int, Is...>) {
    (void)((Is == variant && (go(std::integral_constant<int, Is>{}), true)) || ...);
  }(std::make_integer_sequence<int, kNumConvAnyVariants>{});
  return e;
}
}  // namespace uk
