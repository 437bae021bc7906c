// Compiled kernel variant tables. The solver enumerates exactly these (its candidate set is
// what was compiled, so a plan can never name a kernel that does not exist) and the kernel
// files instantiate exactly these.
#pragma once

namespace uk {

// Work items of one grid dimension. The runtime takes a launch of more without an error and runs what is
// left of the number modulo 2^32.
constexpr long kGridDimItems = 0xffffffffL;
constexpr int kFoldedRow = 1 << 20;  // workgroups in x of a grid that folds into y
inline bool grid_dim_holds(long workgroups, int threads) { return workgroups <= kGridDimItems / threads; }

// Row family (row-sum, RMSNorm, softmax with the row held in registers).
// tpr: threads per row (whole wavefronts), nv: float4 registers per thread.
// A workgroup is max(tpr, 256) threads, i.e. 256/tpr rows per workgroup when tpr < 256.
// nt: loads and stores carry the non-temporal hint (streamed data bypasses cache retention).
// rpb: rows a workgroup walks in turn, the next row's loads in flight during this row's reduction.
// grp: one wavefront per row (tpr = 64, rpb = 1), the workgroup's rows stored together after one
// barrier, a row-length vector staged in LDS per workgroup (the RMSNorm or channelscale gain; for
// softmax a library-owned vector of ones, which the stores multiply by).
// eff: calibrated fraction of the HBM peak the variant sustains for row-sum, RMSNorm and softmax
// (kernel-only median at 4096 x 4096 f32 on one MI355X, rotating buffers > 512 MiB); 0 where the
// variant cannot hold a 4096-wide row, and the solver's bytes-in-flight model prices it alone.
struct RowsVariant {
  int tpr, nv, nt, rpb;
  double eff_sum, eff_rms, eff_softmax;
  int grp = 0;
};
constexpr RowsVariant kRowsVariants[] = {
    {64, 1, 0, 1, 0, 0, 0},
    {64, 2, 0, 1, 0, 0, 0},
    {64, 4, 0, 1, 0, 0, 0},
    {64, 8, 0, 1, 0, 0, 0},
    {64, 16, 0, 1, 0.653, 0.622, 0.625},
    {128, 4, 0, 1, 0, 0, 0},
    {128, 8, 0, 1, 0.697, 0.658, 0.661},
    {256, 1, 0, 1, 0, 0, 0},
    {256, 2, 0, 1, 0, 0, 0},
    {256, 4, 0, 1, 0.707, 0.679, 0.690},
    {256, 8, 0, 1, 0.706, 0.683, 0.681},
    {512, 2, 0, 1, 0.715, 0.694, 0.698},
    {512, 4, 0, 1, 0.715, 0.690, 0.684},
    {1024, 1, 0, 1, 0.549, 0.585, 0.672},
    {1024, 2, 0, 1, 0.552, 0.583, 0.639},
    {1024, 4, 0, 1, 0.544, 0.597, 0.526},
    {256, 4, 1, 1, 0.754, 0.717, 0.718},
    {512, 2, 1, 1, 0.762, 0.713, 0.735},
    {1024, 1, 1, 1, 0.558, 0.598, 0.683},
    {512, 4, 1, 1, 0.759, 0.702, 0.717},
    {1024, 2, 1, 1, 0.562, 0.606, 0.642},
    {128, 8, 1, 1, 0.740, 0.704, 0.709},
    {256, 4, 1, 2, 0.731, 0.718, 0.698},
    {512, 2, 1, 2, 0.742, 0.700, 0.681},
    {64, 16, 1, 1, 0.707, 0.771, 0.759, 1},
};
constexpr int kNumRowsVariants = sizeof(kRowsVariants) / sizeof(kRowsVariants[0]);

// Standalone channelscale in the grouped-store row form (one wavefront per row of at most 4096
// floats, more than half of its lanes busy).
inline bool channelscale_rows_form(long L, long C) { return C % 4 == 0 && C > 2048 && C <= 4096 && L <= 0x7fffffffL; }
// Other shapes go as a flat array (channelscale_flat_kernel): workgroups of 4096 floats, or of 1024 where
// there would be fewer than two of those per CU. Rows of 2049-4096 floats in multiples of 4 keep the row
// form (4096 x 4096: 21.4 us; 4096 x 4097, flat, 24.8).
constexpr long kChannelScaleSmall = 512L * 4096;
inline long channelscale_grid(long n) {
  const long per = n <= kChannelScaleSmall ? 1024 : 4096;
  return (n + per - 1) / per;
}
constexpr int kRowsStreamThreads = 256;

// Rows of any length that the variants above do not hold (C not a multiple of 4, or longer):
// rows_any_kernel keeps the row in registers, tpr threads with nv unaligned float4 each. The entry is
// the smallest that holds the row (rows_any_pick); few rows take the widest teams, because a CU holds
// one row at a time then and its loads all go out at once.
struct RowsAnyVariant {
  int tpr, nv;
};
constexpr RowsAnyVariant kRowsAny[] = {{64, 1},   {64, 2},   {64, 3},   {64, 4},   {64, 6},    {64, 8},    {256, 3},
                                       {256, 4},  {256, 5},  {256, 6},  {256, 8},  {256, 10},  {256, 12},  {256, 16},
                                       {1024, 1}, {1024, 2}, {1024, 3}, {1024, 4}, {1024, 5},  {1024, 6},  {1024, 8},
                                       {1024, 10}, {1024, 12}, {1024, 15}, {1024, 18}};
constexpr int kNumRowsAny = sizeof(kRowsAny) / sizeof(kRowsAny[0]);
constexpr long kRowsAnyFew = 512;  // rows up to which 1024 threads take a row of more than 2048 floats
inline int rows_any_pick(long L, long C) {
  for (int i = 0; i < kNumRowsAny; ++i) {
    if (kRowsAny[i].tpr == 256 && L <= kRowsAnyFew) continue;
    if (C <= long(kRowsAny[i].tpr) * kRowsAny[i].nv * 4) return i;
  }
  return -1;  // longer rows are streamed
}
// The entry a plan of the family names by its tpr and nv, or, where it names none that holds the row, the pick.
inline int rows_any_entry(int tpr, int nv, long L, long C) {
  for (int i = 0; i < kNumRowsAny; ++i)
    if (kRowsAny[i].tpr == tpr && kRowsAny[i].nv == nv && C <= long(tpr) * nv * 4) return i;
  return rows_any_pick(L, C);
}

// 1-D reduce: pass-1 partial count and threads of the two-pass form, and the length up to which one
// workgroup sums the vector in one launch instead: that takes 4.1 us up to 65536 floats and 1.5 us per
// 65536 more until 262144 (8.8 us; the CU's cache no longer serves it beyond, 17.3 us at 400001), the two
// launches ordered by an event 9.0-10.2 us whatever the length up to 4 Mi floats.
constexpr int kReduceParts = 2048;
constexpr int kReduceThreads = 256;
constexpr int kReduceOneThreads = 1024;
constexpr long kReduceOneMax = 1L << 18;

// f16 MFMA GEMM, layout TN (A[M][K], B stored [N][K]).
// bm x bn x bk macro tile; wm x wn waves; stages of LDS buffering; swz selects the LDS
// XOR swizzle (0: row, 1: row >> 1, 2: row >> 2) for the bank geometry. pp = 0: every wavefront
// interleaves copies, fragment reads and v_mfma_f32_32x32x16_f16 (gemm_f16_tn_kernel); pp = 1:
// ping-pong wavefront groups on v_mfma_f32_16x16x32_f16 (gemm_f16_pp_kernel, 256x256x32 with 8
// wavefronts); pp = 2: four wavefronts of 128x128 on v_mfma_f32_32x32x16_f16 with copies sharing
// one M0 and a fence-free barrier (gemm_f16_w4_kernel, 256x256x32); pp = 3: the same four
// wavefronts on v_mfma_f32_16x16x32_f16 with a rolling A fragment (gemm_f16_w4s_kernel); pp = 4:
// the pp = 2 tiling with 64-deep k-tiles in 128-byte rows, two A and three B tile slots
// (gemm_f16_w4k_kernel; stages counts the A slots); pp = 5: the same on v_mfma_f32_16x16x32_f16
// (gemm_f16_w4k16_kernel); pp = 6: that tile with eight wavefronts of 128x64, two per SIMD
// (gemm_f16_w8k16_kernel). eff is
// the calibrated fraction of the dense f16 MFMA peak the variant sustains when every CU holds a
// tile (kernel-only median at M = N = K = 4096 on one MI355X, clocks settled); the solver's cost
// model scales it by wave quantisation for other shapes.
struct GemmF16Variant {
  int bm, bn, bk, wm, wn, stages, swz;
  double eff;
  int pp;
};
constexpr GemmF16Variant kGemmF16Variants[] = {
    {256, 256, 32, 2, 2, 4, 1, 0.431, 0},
    {256, 256, 32, 2, 2, 4, 2, 0.436, 0},
    {256, 256, 32, 2, 2, 4, 0, 0.432, 0},
    {256, 256, 32, 2, 4, 4, 2, 0.446, 0},
    {256, 128, 32, 2, 2, 4, 2, 0.354, 0},
    {256, 128, 64, 2, 2, 3, 1, 0.336, 0},
    {128, 128, 64, 2, 2, 3, 1, 0.231, 0},
    {128, 128, 32, 2, 2, 4, 2, 0.314, 0},
    {256, 256, 32, 2, 4, 5, 2, 0.445, 0},
    {256, 256, 32, 2, 2, 5, 2, 0.425, 0},
    {256, 256, 32, 2, 4, 4, 2, 0.479, 1},
    {256, 256, 32, 2, 4, 5, 2, 0.475, 1},
    {256, 256, 32, 2, 2, 4, 2, 0.448, 2},
    {256, 256, 32, 2, 2, 5, 2, 0.446, 2},
    {256, 256, 32, 2, 4, 4, 1, 0.477, 1},
    {256, 256, 32, 2, 4, 5, 1, 0.473, 1},
    {256, 256, 32, 2, 2, 4, 1, 0.440, 3},
    {256, 256, 64, 2, 2, 2, 1, 0.487, 4},
    {256, 256, 64, 2, 2, 2, 1, 0.545, 5},
    {256, 256, 64, 2, 4, 2, 1, 0.517, 6},
};
constexpr int kNumGemmF16Variants = sizeof(kGemmF16Variants) / sizeof(kGemmF16Variants[0]);

// GEMM of any M, N, K, either B layout, fp16 or fp32, element-aligned operands (kernels/gemm_any.hip).
// tile (mt == 0): a bm x bn tile per workgroup, wm x wn wavefronts per k group and ks k groups, each
// multiplying its own 128-byte k segment of the rows. skinny (mt > 0): 16 mt rows of A per workgroup,
// `waves` wavefronts splitting k over 16 nt columns of B ([N][K]) or 64 ([K][N], with twice the
// wavefronts up to 16), operands straight into registers.
// The cost of a variant is fixed_us + (iterations + tail) * sum over rounds of max(lat_us, n * work),
// with n the workgroups a CU holds in that round: lat_us is one iteration's load latency, work its
// share of the CU's time (work_f16 / work_f32, times nt_factor where B is [K][N], times `unaligned`
// where the rows of B are not whole 16-byte chunks), tail the fold and stores in iterations. Fitted
// over 515 shapes drawn from M 1-4096, N 64-11008, K 64-4096 (every variant measured at each, both
// types and layouts) whose inputs stayed in the MALL: the pick's time is about 2% over the fastest variant's
// on average (26% at 16x11008x4096 TN: 23.4 us for variant 7 where variant 2 takes 17.0). Whatever the
// sum says, no variant has sustained more than kGemmAnyPeakF16 / F32 of the matrix-core peak.
// The 64x64 variant 0 is the one any shape falls back to; a product of a single tile of it (M, N <= 64) is offered
// variant 7 in its place, whose 16-row workgroups spread it over CUs (64x64x96 f32: 3.9 against 5.1 us).
// nt_factor 0: not compiled for B [K][N].
// Variant 11 (256x192, TN only) is for products whose 256x256 tiles leave a quarter of the CUs idle or
// spill into a new round: 1000x11008x4096 (232 tiles for 172) 107 -> 97 us, 1454x5888x1408 43 -> 37,
// 3637x2887x3584 98 -> 86; picked at five of 49 drawn TN shapes and the fastest at each. For B [K][N] its
// three chunks per thread do not split into pairs of k, and the 128x192 tile that would, in two k groups,
// gained 1% at best over 256x128 there (46.5 against 46.8 us at 512x9728x2560): not compiled.
// id: the plan's variant number (1 is gemm_f32_kernel). resident: the workgroups per CU the costs were fitted with.
struct GemmAnyVariant {
  int id, bm, bn, wm, wn, ks, mt, nt, waves, unroll, resident, f16_only;
  double lat_us, work_f16, work_f32, nt_factor, fixed_us, tail, unaligned;
};
constexpr GemmAnyVariant kGemmAnyVariants[] = {
    {0, 64, 64, 2, 2, 1, 0, 0, 0, 0, 4, 0, 0.270, 0.297, 0.600, 1.255, 2.860, 1.045, 1.135},
    {2, 64, 64, 2, 2, 2, 0, 0, 0, 0, 2, 0, 0.361, 0.531, 1.150, 1.120, 2.502, 1.396, 1.172},
    {3, 64, 64, 2, 2, 4, 0, 0, 0, 0, 1, 0, 0.600, 1.346, 2.450, 1.050, 1.224, 1.315, 1.110},
    {4, 128, 64, 2, 2, 1, 0, 0, 0, 0, 3, 0, 0.662, 0.473, 1.183, 1.020, 2.908, 0.854, 1.099},
    {5, 256, 128, 4, 2, 1, 0, 0, 0, 0, 1, 1, 0.600, 0.926, 0.000, 1.096, 0.000, 4.178, 1.156},
    {6, 256, 256, 2, 4, 1, 0, 0, 0, 0, 1, 1, 0.600, 1.573, 0.000, 1.089, 0.000, 3.277, 1.138},
    {11, 256, 192, 2, 4, 1, 0, 0, 0, 0, 1, 1, 0.600, 1.280, 0.000, 0.000, 0.000, 5.214, 1.221},
    {7, 16, 16, 0, 0, 0, 1, 1, 8, 4, 2, 0, 0.720, 0.766, 0.794, 2.324, 1.485, 0.000, 1.147},
    {8, 16, 32, 0, 0, 0, 1, 2, 4, 4, 4, 0, 0.608, 0.596, 0.649, 1.443, 1.606, 0.500, 1.237},
    {9, 32, 32, 0, 0, 0, 2, 2, 8, 2, 2, 0, 0.600, 1.473, 1.933, 1.493, 0.951, 0.230, 1.171},
    {10, 32, 64, 0, 0, 0, 2, 4, 8, 2, 2, 0, 0.600, 2.481, 3.245, 0.853, 0.494, 0.452, 1.189},
};
constexpr double kGemmAnyPeakF16 = 0.467, kGemmAnyPeakF32 = 0.80;
constexpr int kNumGemmAnyVariants = sizeof(kGemmAnyVariants) / sizeof(kGemmAnyVariants[0]);
// Products of many whole tiles (f16 TN: of 128x128x32; f32: of 64x64x64) ask for 16-byte aligned operands, whichever
// kernel the plan names: the direct-to-LDS kernels, which share these shapes, need it, and whether a call is
// taken must not hang on which of them a cost constant prefers. Few whole tiles (fewer than 16 or 32, which
// those kernels rarely get), other shapes and variant 0 take any element alignment.
inline bool gemm_whole_tiles(bool f16, bool tn, long M, long N, long K) {
  return f16 ? tn && M % 128 == 0 && N % 128 == 0 && K % 32 == 0 : M % 64 == 0 && N % 64 == 0 && K % 64 == 0;
}
inline bool gemm_few_tiles(bool f16, bool tn, long M, long N, long K) {
  return gemm_whole_tiles(f16, tn, M, N, K) && (f16 ? (M / 128) * (N / 128) < 16 : (M / 64) * (N / 64) < 32);
}
inline bool gemm_any_asks_alignment(int variant, bool f16, bool tn, long M, long N, long K) {
  return variant != 0 && gemm_whole_tiles(f16, tn, M, N, K) && !gemm_few_tiles(f16, tn, M, N, K);
}
constexpr int gemm_skinny_nt_waves(int waves) { return 2 * waves <= 16 ? 2 * waves : 16; }

// Q8_0 skinny GEMM: a workgroup owns 16 nt weight rows; each of its wavefronts copies `pairs`
// block pairs of those rows per round into its own LDS area (nt * pairs * 1088 bytes) and
// computes them; a round covers waves * pairs block pairs. vec: dwords per lane per copy
// instruction (4 needs K divisible by 64 * pairs). db: two LDS buffers per wavefront, the next
// round's copies in flight while the current round is computed. nt: 16-row weight tiles that
// share each activation fragment.
// gemv: the M = 1 kernel instead (one weight row per wavefront, vector-ALU dot products, `waves`
// rows per workgroup sharing the activation row in LDS, one block pair per lane: K <= 4096).
// many: more than 16 activation rows, where a workgroup's compute sets the time: fixed_us +
// (rounds of k + tail) * sum over rounds of workgroups of max(lat_us, n * work), n the workgroups a
// CU holds (the form of kGemmAnyVariants' cost), fitted over 170 shapes of M 17-512, N 64-11008, K
// 64-11008 together with the tile kernels' (below): the pick is 2% over the fastest on average.
struct Q8Many {
  double lat_us, work, fixed_us, tail;
};
struct Q8Variant {
  int waves, pairs, vec, db, nt, gemv;
  Q8Many many;
};
constexpr Q8Variant kQ8Variants[] = {
    {16, 4, 4, 0, 1, 0, {0.600, 3.633, 1.427, 0.000}}, {16, 4, 1, 0, 1, 0, {3.894, 0.000, 0.893, 0.260}},
    {8, 8, 4, 0, 1, 0, {0.600, 3.102, 2.961, 0.000}},  {8, 4, 1, 0, 1, 0, {0.600, 1.999, 2.706, 0.000}},
    {8, 4, 4, 1, 1, 0, {0.600, 1.826, 2.657, 0.000}},  {4, 4, 4, 1, 1, 0, {1.354, 1.016, 2.460, 0.000}},
    {4, 8, 4, 1, 1, 0, {0.600, 2.249, 3.102, 0.000}},  {8, 4, 4, 0, 4, 0, {0.600, 4.217, 0.000, 0.365}},
    {8, 4, 4, 0, 1, 0, {0.600, 1.846, 1.948, 0.000}},  {8, 4, 4, 0, 3, 0, {0.600, 3.443, 0.000, 0.455}},
    {4, 1, 4, 0, 1, 1, {}}};
constexpr int kNumQ8Variants = sizeof(kQ8Variants) / sizeof(kQ8Variants[0]);
// Q8_0 GEMM tiles for more than 16 activation rows (q8_0_tile_kernel): bm x bn outputs per workgroup,
// wm x wn wavefronts per k group, ks k groups. The plan's variant number is kNumQ8Variants + index.
struct Q8TileVariant {
  int bm, bn, wm, wn, ks, resident;
  Q8Many many;
};
constexpr Q8TileVariant kQ8TileVariants[] = {
    {32, 64, 1, 4, 4, 1, {0.730, 0.510, 0.000, 5.206}},
    {64, 64, 2, 2, 4, 1, {0.930, 0.300, 0.000, 4.433}},
    {32, 32, 1, 2, 4, 2, {0.509, 0.470, 2.264, 1.818}},
};
constexpr int kNumQ8TileVariants = sizeof(kQ8TileVariants) / sizeof(kQ8TileVariants[0]);

// Implicit-GEMM conv on f32 MFMA (v_mfma_f32_32x32x2f32). Wide kernel (tile_strips 0): a
// wavefront owns 32 output pixels x 64 output channels, `waves` wavefronts per workgroup, and
// bk_bytes is the LDS budget of one staged weight chunk (channels = budget / (taps * 64 * 4 B),
// even). Tile kernel (tile_strips S > 0, 3x3 and 1x1 only): wavefronts of 32 pixels x 32 output
// channels, S strips x 2 channel halves per workgroup, bk_bytes channels per weight chunk. LDS
// kernel (tile_strips -T for T = 1, 2, NCHW 3x3 stride 1 only, see conv_lds_supported): 64 T
// pixels x 64 output channels per workgroup of 4 T wavefronts, input rows and weights of 8
// channels staged in LDS. 16-pixel-group kernel (tile_strips kConvL16, see conv_l16_geom): runs of
// 16-pixel groups x 64 output channels per workgroup of 8 wavefronts on v_mfma_f32_16x16x4f32,
// bk_bytes channels per staged chunk. eff is the calibrated fraction of the f32 MFMA rate the
// busiest SIMD sustains (kernel-only median at the BASELINE conv shape on one MI355X).
struct ConvVariant {
  int waves;
  int bk_bytes;
  int tile_strips;
  double eff;
};
constexpr ConvVariant kConvVariants[] = {
    {4, 147456, 0, 0.273}, {2, 73728, 0, 0.175}, {4, 73728, 0, 0.260}, {2, 36864, 0, 0.170},
    {4, 16, 2, 0.130},     {4, 8, 2, 0.130},     {8, 8, 4, 0.310},     {4, 8, -1, 0.472},
    {8, 8, -2, 0.619},     {8, 16, -16, 0.696},
};
// LDS kernel geometry: input rows and padded columns one staged tile holds.
constexpr int kConvLdsRows = 8;
constexpr int kConvLdsCols = 64;
// The LDS kernel covers NCHW, 3x3, stride 1, pad 0 or 1, W + 2 pad <= kConvLdsCols, W a multiple
// of 4 and C of 8 (16-byte staging loads, whole channel chunks), and pix (64 or 128) consecutive
// output pixels spanning at most kConvLdsRows - 2 output rows.
inline bool conv_lds_supported(bool nchw, long kh, long kw, long stride, long pad, long W, long Ho, long Wo, long C,
                               long pix) {
  if (!nchw || kh != 3 || kw != 3 || stride != 1 || (pad != 0 && pad != 1)) return false;
  if (W + 2 * pad > kConvLdsCols || W % 4 != 0 || C % 8 != 0 || C <= 0 || Wo <= 0 || Ho <= 0) return false;
  return (pix - 1 + Wo - 1) / Wo + 1 + 2 <= kConvLdsRows;
}
constexpr int kNumConvVariants = sizeof(kConvVariants) / sizeof(kConvVariants[0]);

// 16-pixel-group kernel (conv_lds16_kernel, tile_strips kConvL16): the output pixels of an image
// (flattened Ho*Wo order) cut into gp groups of 16, and each image's groups into wpi contiguous
// runs, run j of gp / wpi + (j < gp % wpi) <= kConvL16MaxGroups groups, one workgroup (x 64
// output channels) each. wpi aims the launch at kConvL16Target workgroups (the CU count of
// MI355X: one workgroup per CU, runs balanced to within one group). rows: the most output rows
// a run spans; the kernel stages rows + 2 input rows per channel chunk, at most kConvL16Rows.
constexpr int kConvL16 = -16;
constexpr int kConvL16Target = 256;
constexpr int kConvL16MaxGroups = 8;
constexpr int kConvL16Rows = 6;
constexpr int kConvL16Pitch = 72;  // 16-byte entries per staged input row (8 mod 16: see the kernel)
constexpr int kConvL16WQuad = 68;  // 16-byte weight entries per channel quad (64 oc + 4: see the kernel)
struct ConvL16Geom {
  long gp, wpi, gmax, rows;
};
inline ConvL16Geom conv_l16_geom(long N, long Ho, long Wo, long oc_blocks) {
  ConvL16Geom g{0, 0, 0, 0};
  if (N <= 0 || Ho <= 0 || Wo <= 0 || oc_blocks <= 0) return g;
  const long P = Ho * Wo;
  g.gp = (P + 15) / 16;
  long wpi = (kConvL16Target + N * oc_blocks - 1) / (N * oc_blocks);
  const long least = (g.gp + kConvL16MaxGroups - 1) / kConvL16MaxGroups;
  if (wpi < least) wpi = least;
  if (wpi > g.gp) wpi = g.gp;
  g.wpi = wpi;
  const long q = g.gp / wpi, r = g.gp % wpi;
  for (long j = 0; j < wpi; ++j) {
    const long a = j * q + (j < r ? j : r), b = a + q + (j < r ? 1 : 0);
    const long pend = (16 * b < P ? 16 * b : P) - 1;
    const long rows = pend / Wo - (16 * a) / Wo + 1;
    if (b - a > g.gmax) g.gmax = b - a;
    if (rows > g.rows) g.rows = rows;
  }
  return g;
}
// NCHW, 3x3, stride 1, pad 0 or 1, W + 2 pad <= kConvL16Pitch, W a multiple of 4 and C of 16
// (16-byte staging loads, whole 16-channel chunks), every run within kConvL16Rows - 2 rows, and
// the kernel's index quotients (pixel indices up to 16 (gp + 4), workgroup indices up to N wpi)
// below kConvL16IndexLimit, where its reciprocal division is exact.
constexpr long kConvL16IndexLimit = 1L << 21;
inline bool conv_l16_supported(bool nchw, long kh, long kw, long stride, long pad, long N, long W, long Ho, long Wo,
                               long C, long Oc) {
  if (!nchw || kh != 3 || kw != 3 || stride != 1 || (pad != 0 && pad != 1)) return false;
  if (W + 2 * pad > kConvL16Pitch || W % 4 != 0 || C % 16 != 0 || C <= 0 || Oc <= 0) return false;
  const ConvL16Geom g = conv_l16_geom(N, Ho, Wo, (Oc + 63) / 64);
  return g.wpi > 0 && g.gmax <= kConvL16MaxGroups && g.rows + 2 <= kConvL16Rows &&
         16 * (g.gp + 4) < kConvL16IndexLimit && N * g.wpi < kConvL16IndexLimit;
}

// Implicit-GEMM conv of any kernel size, stride, padding and channel count (conv_any_kernel): bm output
// channels x bn pixels of one image per workgroup, wm x wn wavefronts per k group, ks k groups. The
// plan's variant number is kNumConvVariants + index. Cost: fixed_us + (32 ks-deep steps of k + tail) *
// sum over rounds of max(lat, n * work), n the workgroups a CU holds (the form of kGemmAnyVariants'
// cost), fitted over 220 drawn shapes (7-256 pixels a side, 3-256 channels, kernels of 1, 3 and 5): the
// pick is 1.2% over the fastest on average. resident is what the fit took (a CU holds four of the first
// variant: 14.2 of 16 wavefronts counted at 256x256x32). work: NCHW, HWC with C a multiple of 4 (16-byte loads), HWC.
struct ConvAnyVariant {
  int bm, bn, wm, wn, ks, resident;
  double lat_us, lat_vec_us, work_nchw, work_vec, work_hwc, fixed_us, tail;
};
constexpr ConvAnyVariant kConvAnyVariants[] = {
    {64, 64, 2, 2, 1, 3, 1.198, 0.692, 0.957, 0.630, 1.097, 2.843, 0.832},
    {64, 64, 2, 2, 2, 2, 0.800, 0.500, 1.987, 1.294, 2.203, 2.689, 0.453},
    {32, 64, 1, 4, 2, 2, 0.800, 0.500, 1.425, 0.772, 1.684, 2.823, 0.312},
    {32, 64, 2, 2, 1, 4, 0.901, 0.426, 0.671, 0.384, 0.930, 3.175, 0.561},
};
constexpr int kNumConvAnyVariants = sizeof(kConvAnyVariants) / sizeof(kConvAnyVariants[0]);
// Byte offsets within one image's X are 32-bit, k and pixel indices 31-bit, and the quotient k / inner by
// mulhi is exact for k * inner < 2^32.
inline bool conv_any_supported(bool nchw, long N, long C, long H, long W, long Oc, long kh, long kw, long Ho, long Wo) {
  const long taps = kh * kw, K = C * taps, inner = nchw ? taps : C;
  if (N <= 0 || C <= 0 || Oc <= 0 || Ho <= 0 || Wo <= 0 || taps <= 0 || taps > 49) return false;
  if ((nchw ? H * W : H * W * C) * 4 > 0x7fffffffL || Ho * Wo > 0x3fffffffL) return false;
  return K < 0x1000000L && K * inner < 0xffffffffL;
}

// Sustained shader clock (GHz) of the matrix-core probe (uk_probe_mfma: one wavefront per SIMD
// issuing only v_mfma_f32_16x16x32_f16 on switching random operands, its primary form) on the
// parts where the GEMM and conv efficiencies above were fitted (2.01-2.03 GHz measured; the same
// parts settle at 1.66 GHz under the 32x32x16 form). A part whose probe sustains less under that
// load runs every MFMA-bound kernel proportionally slower; calibration uses the ratio when no
// measured MFMA-bound row is available.
constexpr double kEffFitProbeClockGhz = 2.02;

}  // namespace uk
