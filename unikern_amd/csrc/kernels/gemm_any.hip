// GEMM of any shape on gfx950 matrix cores: C[M][N] = A[M][K] . B with B stored [N][K] (TN) or [K][N]
// (NT, the reference's layout, src/codegen_hip.cpp:1089-1120), f16 or f32 operands with f32 sums, any
// M, N and K, operands aligned to their element only. One template serves both types: a 128-byte row
// segment is 64 halves or 32 floats, a 16-byte chunk of it is one lane's share of a fragment, and
// the chunk's halves feed one 16x16x32 MFMA, its floats four 16x16x4 MFMAs.
//
// Two forms (kGemmAnyVariants lists the compiled ones and their costs):
//
// gemm_any_kernel: a BM x BN tile per workgroup, operands staged through registers into two LDS
//   slots, one barrier per step of k. A step stores the next step's operands, loaded D steps ago,
//   issues the loads that replace them and multiplies: the loads have D whole steps to land, and the
//   barrier waits for LDS only. The loop has no branch around a load (past the end they repeat the last
//   whole step; the partial step has loads of its own), because with one the compiler can no longer
//   count the loads in flight and waits for all of them: storing after the multiply, with branches,
//   256x256 took 117.5 us at 1000x11008x4096 (107 now) and 64x64 in two k groups 32.3 us at f32 NT
//   1000^3 (24.8 now). Registers (not direct-to-LDS copies) because rows of any length start at any
//   address: the unaligned 128-bit loads need no special case, only chunks that cross the end of a row
//   do, and B stored [K][N] is transposed on its way (v_perm on pairs of k). With S > 1, S groups of
//   wavefronts multiply S consecutive 128-byte segments and add their sums in LDS at the end: small
//   grids then have S times the loads in flight. Bound by load latency below about two workgroups per
//   CU; above, no pipe is full (256x192 at 1000x11008x4096: matrix cores 0.50 of a busy CU's cycles, LDS 0.39;
//   row-major B at 512x9728x2560: 0.36, LDS 0.48 of which the transposing stores' conflicts 0.15, vector ALU
//   0.32): a step's stores, fragment reads and MFMAs follow each other in the two wavefronts of a SIMD.
// gemm_skinny_*_kernel: 16-32 rows of A. Wavefronts split k, each lane loads its fragments of both
//   operands straight into registers (no LDS, no barrier until the partial sums are added), several
//   steps' loads in flight. Bound by the vector cache's tag lookups (0.89 a cycle at 16x11008x4096: the lanes of a
//   load are 16 rows apart), then the stream of B.
//
// Measured against the bounds-checked 64x64x16 kernel these replaced (element loads, two barriers per
// 16 k), one box, inputs rotating over three sets: f16 TN 1000x11008x4096 2667 -> 96.8 us (932
// TFLOP/s; 256x192), 16x11008x4096 251 -> 23.9 us (3.8 TB/s; skinny), f16 NT 512x9728x2560 440 ->
// 46.8 us (545 TFLOP/s; 256x128), f32 NT 1000^3 131 -> 24.8 us (81 TFLOP/s; 64x64 in two k groups),
// and against 64 bits the f32 sums are no further off (4.0e-7 against 5.7e-7).
#include "../launch.hpp"
#include "../variants.hpp"
#include "common.hpp"
#include "tile.hpp"

#include <type_traits>
#include <utility>

namespace uk::kern {

// Four f32 sums of consecutive columns, in the output type.
template <typename T>
struct any_out;
template <>
struct any_out<_Float16> {
  typedef f16x4 type;
  static __device__ __forceinline__ type of(f32x4 v) {
    return f16x4{(_Float16)v[0], (_Float16)v[1], (_Float16)v[2], (_Float16)v[3]};
  }
};
template <>
struct any_out<float> {
  typedef f32x4 type;
  static __device__ __forceinline__ type of(f32x4 v) { return v; }
};

template <typename T, int BM, int BN, int WM, int WN, int S>
struct AnyCfg {
  static constexpr int kE = 16 / (int)sizeof(T);   // elements of a 16-byte chunk
  static constexpr int kSlab = 128 / (int)sizeof(T);  // k of one 128-byte row segment
  static constexpr int kGroup = WM * WN * 64;      // threads of one k group
  static constexpr int kThreads = kGroup * S;
  static constexpr int kFM = BM / WM / 16, kFN = BN / WN / 16;
  static constexpr int kNA = BM * 8 / kGroup, kNB = BN * 8 / kGroup;  // chunks per thread and slab
  static constexpr int kOpA = BM * 128, kOpB = BN * 128;
  static constexpr int kSlot = kOpA + kOpB;
  static constexpr int kPitch = BN / WN * (int)sizeof(T) + 16;
  static constexpr int kPipe = 2 * S * kSlot;
  static constexpr int kRed = (S - 1) * BM * BN * 4;
  static constexpr int kStage = WM * WN * (BM / WM) * kPitch;
  static constexpr int kLds = kPipe > kRed ? (kPipe > kStage ? kPipe : kStage) : (kRed > kStage ? kRed : kStage);
};

template <typename T, int BM, int BN, int WM, int WN, int S, int D, bool BT>
__global__ void __launch_bounds__(WM* WN* S * 64)
    gemm_any_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int K, int tiles_m,
                    int tiles_n) {
  using Cfg = AnyCfg<T, BM, BN, WM, WN, S>;
  constexpr int E = Cfg::kE, SLAB = Cfg::kSlab, FM = Cfg::kFM, FN = Cfg::kFN, NA = Cfg::kNA, NB = Cfg::kNB;
  constexpr int KT_ELEMS = S * SLAB;
  asm volatile("" ::"s"(A), "s"(B), "s"(C), "s"(M), "s"(N), "s"(K), "s"(tiles_m), "s"(tiles_n));
  __shared__ __attribute__((aligned(1024))) char lds[Cfg::kLds];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kh = w / (WM * WN), wg = w % (WM * WN), wm = wg / WN, wn = wg % WN;
  const int tg = tid - kh * Cfg::kGroup;

  // Workgroup i runs on XCD i % 8: give each XCD a contiguous range of tiles (the first G % 8 XCDs
  // one more), walked in groups of 4 tile rows.
  const int G = tiles_m * tiles_n;
  const int id = folded_id();
  if (id >= G) return;
  const int xcd = id & 7, per = G >> 3, rem = G & 7;
  const int lin = xcd * per + (xcd < rem ? xcd : rem) + (id >> 3);
  constexpr int kGroupM = 4;
  const int per_group = kGroupM * tiles_n;
  const int group = lin / per_group;
  const int first_m = group * kGroupM;
  const int gm = (tiles_m - first_m) < kGroupM ? (tiles_m - first_m) : kGroupM;
  const int in_group = lin - group * per_group;
  const int m0 = (first_m + in_group % gm) * BM, n0 = (in_group / gm) * BN;

  // Staging lanes. K-contiguous operands: chunk u of a thread is row u * (kGroup / 8) + tg / 8,
  // 16-byte chunk tg % 8 (eight lanes read one 128-byte row segment). Rows past the edge read the
  // last row (they feed only outputs that are not stored).
  const int crow = tg >> 3, cc = tg & 7;
  const T* arow[NA];
#pragma unroll
  for (int u = 0; u < NA; ++u) {
    const int r = m0 + u * (Cfg::kGroup / 8) + crow;
    arow[u] = A + (int64_t)(r < M ? r : M - 1) * K;
  }
  // B stored [K][N]: a thread owns NB rows of k by one chunk of E columns and writes them
  // transposed. Lanes: eight chunks of columns (one 128-byte line) by eight groups of k.
  constexpr int kGroupsK = SLAB / NB;  // k groups of a slab
  constexpr int kGW = kGroupsK / 8;
  const int nc = (tg & 7) + 8 * ((tg >> 6) / kGW);
  const int kg = ((tg >> 3) & 7) + 8 * ((tg >> 6) % kGW);
  const T* brow[BT ? NB : 1];
  if constexpr (BT) {
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const int r = n0 + u * (Cfg::kGroup / 8) + crow;
      brow[u] = B + (int64_t)(r < N ? r : N - 1) * K;
    }
  } else {
    brow[0] = B;
  }
  // B stored [K][N] at the right edge (N >= E there): a chunk that crosses N is read as the row's last
  // E columns and its own moved to their places when it is stored.
  const bool whole_n = BT || N - n0 >= BN;
  const int nb = n0 + nc * E;
  const int nl = N - nb >= E ? nb : N - E;
  const int nshift = nb - nl < E ? (nb - nl) * (int)sizeof(T) * 8 : 0;

  // Whole steps of k, and a last partial one. Loads of whole step t into register set t % D; past the
  // last they read it again: no branch, so the compiler waits for one step's loads by count while the
  // next step's are in flight.
  const int whole_steps = K / KT_ELEMS;
  const bool tail = whole_steps * KT_ELEMS < K;
  u32x4 ra[D][NA], rb[D][NB];
  auto load = [&](auto set_c, int t) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value % D;
    const int k0 = (t < whole_steps ? t : whole_steps - 1) * KT_ELEMS + kh * SLAB;
#pragma unroll
    for (int u = 0; u < NA; ++u) ra[set][u] = any_load16(arow[u] + k0 + cc * E);
    if constexpr (BT) {
#pragma unroll
      for (int u = 0; u < NB; ++u) rb[set][u] = any_load16(brow[u] + k0 + cc * E);
    } else {
#pragma unroll
      for (int u = 0; u < NB; ++u) rb[set][u] = any_load16(B + (int64_t)(k0 + kg * NB + u) * N + nl);
    }
  };
  auto load_tail = [&](u32x4(&ta)[NA], u32x4(&tb)[NB]) __attribute__((always_inline)) {
    const int k0 = whole_steps * KT_ELEMS + kh * SLAB;
#pragma unroll
    for (int u = 0; u < NA; ++u) ta[u] = any_load16_edge(arow[u], k0 + cc * E, K);
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      if constexpr (BT) {
        tb[u] = any_load16_edge(brow[u], k0 + cc * E, K);
      } else {
        const int k = k0 + kg * NB + u;
        tb[u] = k < K ? any_load16(B + (int64_t)k * N + nl) : u32x4{0, 0, 0, 0};
      }
    }
  };
  // 16-byte chunk c of row r sits at c ^ ((r >> 1) & 7): fragment reads (16 rows at one chunk
  // column) spread over the banks.
  auto store = [&](u32x4(&sa)[NA], u32x4(&sb)[NB], auto slot_c) __attribute__((always_inline)) {
    const int slot = slot_c;
    char* as = lds + (slot * S + kh) * Cfg::kSlot;
    char* bs = as + Cfg::kOpA;
#pragma unroll
    for (int u = 0; u < NA; ++u) {
      const int r = u * (Cfg::kGroup / 8) + crow;
      *reinterpret_cast<u32x4*>(as + r * 128 + ((cc ^ ((r >> 1) & 7)) << 4)) = sa[u];
    }
    if constexpr (BT) {
#pragma unroll
      for (int u = 0; u < NB; ++u) {
        const int r = u * (Cfg::kGroup / 8) + crow;
        *reinterpret_cast<u32x4*>(bs + r * 128 + ((cc ^ ((r >> 1) & 7)) << 4)) = sb[u];
      }
    } else {
      if (!whole_n) {
#pragma unroll
        for (int u = 0; u < NB; ++u)
          sb[u] = __builtin_bit_cast(u32x4, (unsigned __int128)(__builtin_bit_cast(unsigned __int128, sb[u]) >> nshift));
      }
#pragma unroll
      for (int j = 0; j < E; ++j) {
        const int r = nc * E + j;
        if constexpr (sizeof(T) == 2) {
          // Halves j of NB rows, in pairs of k.
          uint32_t o[NB / 2];
#pragma unroll
          for (int p = 0; p < NB / 2; ++p)
            o[p] = __builtin_amdgcn_perm(sb[2 * p + 1][j >> 1], sb[2 * p][j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
          const int kb = kg * NB * 2;  // byte of the row segment
          char* dst = bs + r * 128 + (((kb >> 4) ^ ((r >> 1) & 7)) << 4) + (kb & 15);
          if constexpr (NB == 4) *reinterpret_cast<u32x2*>(dst) = u32x2{o[0], o[1]};
          else *reinterpret_cast<uint32_t*>(dst) = o[0];
        } else {
          const int kb = kg * NB * 4;
          char* dst = bs + r * 128 + (((kb >> 4) ^ ((r >> 1) & 7)) << 4) + (kb & 15);
          if constexpr (NB == 4) *reinterpret_cast<u32x4*>(dst) = u32x4{sb[0][j], sb[1][j], sb[2][j], sb[3][j]};
          else *reinterpret_cast<u32x2*>(dst) = u32x2{sb[0][j], sb[1][j]};
        }
      }
    }
  };
  static_assert(BT || NB == 2 || NB == 4, "the transposing store writes 2 or 4 k at a time");

  const int fi = lane & 15, fg = lane >> 4;
  f32x4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](auto slot_c) __attribute__((always_inline)) {
    const int slot = slot_c;
    const char* as = lds + (slot * S + kh) * Cfg::kSlot + (wm * (BM / WM) + fi) * 128;
    const char* bs = lds + (slot * S + kh) * Cfg::kSlot + Cfg::kOpA + (wn * (BN / WN) + fi) * 128;
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
        for (int j = 0; j < FN; ++j) acc[i][j] = any_mfma<T>(fb[j], fa[i], acc[i][j]);
    }
  };

  // Step t: its operands sit in slot t % 2; the next step's, loaded D steps ago, go into the other slot
  // (every wavefront passed the barrier after reading it), the loads of step t + 1 + D take their
  // registers, and only then does it multiply. With D = 2 (tiles whose registers allow it) sets and
  // slots are compile-time constants and the tail's loads, issued first, have registers of their own.
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  auto step = [&](auto set_c, auto slot_c, auto next_c, int t) __attribute__((always_inline)) {
    constexpr int set = decltype(set_c)::value % D;
    store(ra[set], rb[set], next_c);
    load(set_c, t + 1 + D);
    __builtin_amdgcn_sched_barrier(0);
    multiply(slot_c);
    lds_barrier();
  };
  u32x4 ta[D == 2 ? NA : 1], tb[D == 2 ? NB : 1];
  if constexpr (D == 2) {
    if (tail) load_tail(ta, tb);
  }
  if (whole_steps > 0) {
    load(I0{}, 0);
    if constexpr (D == 2) load(I1{}, 1);
    store(ra[0], rb[0], I0{});
    load(I0{}, D);
    lds_barrier();
    if constexpr (D == 2) {
      int t = 0;
      for (; t + 1 < whole_steps; t += 2) {
        step(I1{}, I0{}, I1{}, t);
        step(I0{}, I1{}, I0{}, t + 1);
      }
      if (t < whole_steps) step(I1{}, I0{}, I1{}, t);
    } else {
      for (int t = 0; t < whole_steps; ++t) step(I0{}, t & 1, (t + 1) & 1, t);
    }
  }
  if (tail) {
    if constexpr (D == 2) {
      store(ta, tb, I0{});
    } else {
      load_tail(ra[0], rb[0]);
      store(ra[0], rb[0], I0{});
    }
    lds_barrier();
    multiply(I0{});
    lds_barrier();
  }

  // k groups 1 .. S - 1 hand their sums to group 0, which adds them in order.
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
  // Stage the wavefront's tile in LDS and store whole rows, 16 bytes per lane (unaligned where N
  // makes the rows so), single elements at the right edge.
  typedef typename any_out<T>::type O;
  char* stage = lds + wg * (BM / WM) * Cfg::kPitch;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
      *reinterpret_cast<O*>(stage + (i * 16 + fi) * Cfg::kPitch + (j * 16 + 4 * fg) * (int)sizeof(T)) =
          any_out<T>::of(acc[i][j]);
  __asm__ volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  constexpr int kRowChunks = BN / WN / E;
  const int mw = m0 + wm * (BM / WM), nw = n0 + wn * (BN / WN);
#pragma unroll 4
  for (int id = lane; id < BM / WM * kRowChunks; id += 64) {
    const int r = id / kRowChunks, q = id % kRowChunks;
    const int m = mw + r, n = nw + q * E;
    if (m >= M || n >= N) continue;
    const u32x4 v = *reinterpret_cast<const u32x4*>(stage + r * Cfg::kPitch + q * 16);
    T* dst = C + (int64_t)m * N + n;
    if (N - n >= E) {
      __builtin_memcpy(dst, &v, 16);
    } else {
      T e[E];
      __builtin_memcpy(e, &v, 16);
#pragma unroll
      for (int i = 0; i < E; ++i)
        if (i < N - n) dst[i] = e[i];
    }
  }
}

// Sum over the wavefronts' partial tiles (in wavefront order) and store: thread o takes lane
// o % 64 of tile o / 64; col(tile, lane) is the first of the columns `cstep` apart it holds.
template <typename T, int W, int TILES, class F>
__device__ __forceinline__ void skinny_fold(const f32x4* red, T* __restrict__ C, int M, int N, F&& place) {
  for (int o = threadIdx.x; o < TILES * 64; o += W * 64) {
    f32x4 v = red[o];
#pragma unroll
    for (int w = 1; w < W; ++w) {
      const f32x4 p = red[w * TILES * 64 + o];
      v = f32x4{v[0] + p[0], v[1] + p[1], v[2] + p[2], v[3] + p[3]};
    }
    int m, n, step;
    place(o >> 6, o & 63, m, n, step);
    if (m < M) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r * step < N - n) C[(int64_t)m * N + n + r * step] = (T)v[r];
    }
  }
}

// Skinny, B stored [N][K]: W wavefronts take the row segments w, w + W, ... of 16 NT columns; U
// segments' loads are issued together (two loads of a lane cover 32 of a row's 128 bytes, so every
// line is fetched once).
template <typename T, int MT, int NT, int W, int U>
__global__ void __launch_bounds__(W * 64)
    gemm_skinny_tn_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int K, int gm,
                          int gn) {
  constexpr int E = 16 / (int)sizeof(T), SLAB = 8 * E;
  asm volatile("" ::"s"(A), "s"(B), "s"(C), "s"(M), "s"(N), "s"(K), "s"(gm), "s"(gn));
  __shared__ f32x4 red[W * MT * NT * 64];
  const int lane = threadIdx.x & 63, fi = lane & 15, fg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int id = folded_id();
  if (id >= gm * gn) return;
  const int n0 = id % gn * 16 * NT, m0 = id / gn * 16 * MT;
  const T* arow[MT];
  const T* brow[NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = A + (int64_t)(m0 + 16 * i + fi < M ? m0 + 16 * i + fi : M - 1) * K;
#pragma unroll
  for (int j = 0; j < NT; ++j) brow[j] = B + (int64_t)(n0 + 16 * j + fi < N ? n0 + 16 * j + fi : N - 1) * K;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  auto slabs = [&]<int CNT, bool EDGE>(int s) __attribute__((always_inline)) {
    u32x4 fb[CNT][NT][2], fa[CNT][MT][2];
#pragma unroll
    for (int u = 0; u < CNT; ++u) {
      const int k = (s + u * W) * SLAB + fg * E;
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          fb[u][j][h] = EDGE ? any_load16_edge(brow[j], k + h * 4 * E, K) : any_load16(brow[j] + k + h * 4 * E);
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          fa[u][i][h] = EDGE ? any_load16_edge(arow[i], k + h * 4 * E, K) : any_load16(arow[i] + k + h * 4 * E);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < CNT; ++u)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i][j] = any_mfma<T>(fb[u][j][h], fa[u][i][h], acc[i][j]);
  };
  const int full = K / SLAB;
  int s = w;
  for (; s + (U - 1) * W < full; s += U * W) slabs.template operator()<U, false>(s);
  for (; s < full; s += W) slabs.template operator()<1, false>(s);
  if (s == full && full * SLAB < K) slabs.template operator()<1, true>(s);

#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) red[((w * MT + i) * NT + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  skinny_fold<T, W, MT * NT>(red, C, M, N, [&](int t, int l, int& m, int& n, int& step) {
    m = m0 + 16 * (t / NT) + (l & 15);
    n = n0 + 16 * (t % NT) + 4 * (l >> 4);
    step = 1;
  });
}

// Skinny, B stored [K][N]: lane (i, g) loads the E rows k of its chunk at columns 4 i .. 4 i + 3 (16
// lanes read one 128-byte (f16) or 256-byte row segment) and gathers four fragments, one per column,
// from them: tile j of the wavefront holds the columns 4 x + j.
template <typename T, int MT, int W, int U>
__global__ void __launch_bounds__(W * 64)
    gemm_skinny_nt_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int M, int N, int K, int gm,
                          int gn) {
  constexpr int E = 16 / (int)sizeof(T), STEP = 4 * E;
  typedef T Quad __attribute__((ext_vector_type(4)));
  asm volatile("" ::"s"(A), "s"(B), "s"(C), "s"(M), "s"(N), "s"(K), "s"(gm), "s"(gn));
  __shared__ f32x4 red[W * MT * 4 * 64];
  const int lane = threadIdx.x & 63, fi = lane & 15, fg = lane >> 4;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int id = folded_id();
  if (id >= gm * gn) return;
  const int n0 = id % gn * 64, m0 = id / gn * 16 * MT;
  const int n = n0 + 4 * fi;
  const T* arow[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = A + (int64_t)(m0 + 16 * i + fi < M ? m0 + 16 * i + fi : M - 1) * K;
  f32x4 acc[MT][4];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // MODE 0: whole steps and columns. 1: whole steps in the last column block (N >= 4): a lane whose
  // four columns cross N reads the row's last four and moves its own to their places. 2: element by
  // element (the last, partial step of k; N < 4).
  const int nl = N - n >= 4 ? n : N - 4;
  const int shift = (n - nl < 4 ? n - nl : 0) * (int)sizeof(T) * 8;
  auto steps = [&]<int CNT, int MODE>(int s) __attribute__((always_inline)) {
    Quad q[CNT][E];
    u32x4 fa[CNT][MT];
#pragma unroll
    for (int u = 0; u < CNT; ++u) {
      const int k = (s + u * W) * STEP + fg * E;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        if constexpr (MODE == 2) {
#pragma unroll
          for (int j = 0; j < 4; ++j) q[u][e][j] = e < K - k && j < N - n ? B[(int64_t)(k + e) * N + n + j] : T(0);
        } else {
          __builtin_memcpy(&q[u][e], B + (int64_t)(k + e) * N + (MODE == 1 ? nl : n), sizeof(Quad));
        }
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) fa[u][i] = MODE == 2 ? any_load16_edge(arow[i], k, K) : any_load16(arow[i] + k);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (MODE == 1) {
      typedef std::conditional_t<sizeof(T) == 2, uint64_t, unsigned __int128> Bits;
#pragma unroll
      for (int u = 0; u < CNT; ++u)
#pragma unroll
        for (int e = 0; e < E; ++e)
          q[u][e] = __builtin_bit_cast(Quad, (Bits)(__builtin_bit_cast(Bits, q[u][e]) >> shift));
    }
#pragma unroll
    for (int u = 0; u < CNT; ++u)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        typedef T Frag __attribute__((ext_vector_type(E)));
        Frag f;
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = q[u][e][j];
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i][j] = any_mfma<T>(__builtin_bit_cast(u32x4, f), fa[u][i], acc[i][j]);
      }
  };
  const int all = K / STEP + (K % STEP != 0);
  const int full = N >= 4 ? K / STEP : 0;
  int s = w;
  if (N - n0 >= 64) {
    for (; s + (U - 1) * W < full; s += U * W) steps.template operator()<U, 0>(s);
    for (; s < full; s += W) steps.template operator()<1, 0>(s);
  } else {
    for (; s + (U - 1) * W < full; s += U * W) steps.template operator()<U, 1>(s);
    for (; s < full; s += W) steps.template operator()<1, 1>(s);
  }
  for (; s < all; s += W) steps.template operator()<1, 2>(s);

#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) red[((w * MT + i) * 4 + j) * 64 + lane] = acc[i][j];
  __syncthreads();
  // Tile j holds the columns n0 + 4 x + j, x < 16: a lane's four sums are four columns apart.
  skinny_fold<T, W, MT * 4>(red, C, M, N, [&](int t, int l, int& m, int& nn, int& step) {
    m = m0 + 16 * (t / 4) + (l & 15);
    nn = n0 + 16 * (l >> 4) + (t & 3);
    step = 4;
  });
}

}  // namespace uk::kern

namespace uk {
namespace {
constexpr int kGemmAnyNarrow = 8;  // the skinny 16x32 entry
static_assert(kGemmAnyVariants[kGemmAnyNarrow].id == 8 && kGemmAnyVariants[kGemmAnyNarrow].mt == 1, "a skinny variant");

template <int I, typename T>
hipError_t any_go(bool bt, const T* a, const T* b, T* c, int64_t M, int64_t N, int64_t K, hipStream_t s) {
  constexpr GemmAnyVariant v = kGemmAnyVariants[I];
  if constexpr (v.f16_only && sizeof(T) != 2) {
    return hipErrorInvalidValue;
  } else if constexpr (v.mt == 0) {
    using Cfg = kern::AnyCfg<T, v.bm, v.bn, v.wm, v.wn, v.ks>;
    // B stored [K][N] is read in 16-byte chunks of a row: narrower products run as skinny ones.
    if (!bt && N * (int64_t)sizeof(T) < 16) return any_go<kGemmAnyNarrow, T>(bt, a, b, c, M, N, K, s);
    const int64_t tm = (M + v.bm - 1) / v.bm, tn = (N + v.bn - 1) / v.bn;
    if (tm * tn > INT32_MAX) return hipErrorInvalidValue;
    constexpr int D = v.bm * v.bn >= 128 * 64 ? 1 : 2;  // registers for two load sets
    auto* k = kern::gemm_any_kernel<T, v.bm, v.bn, v.wm, v.wn, v.ks, D, true>;
    if constexpr (v.nt_factor > 0) {
      if (!bt) k = kern::gemm_any_kernel<T, v.bm, v.bn, v.wm, v.wn, v.ks, D, false>;
    } else {
      if (!bt) return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(k, folded_grid(tm * tn), dim3(Cfg::kThreads), 0, s, a, b, c, (int)M, (int)N, (int)K, (int)tm,
                       (int)tn);
    return hipGetLastError();
  } else {
    const int64_t cols = bt ? 16 * v.nt : 64;
    const int64_t gm = (M + 16 * v.mt - 1) / (16 * v.mt), gn = (N + cols - 1) / cols;
    if (gm * gn > INT32_MAX) return hipErrorInvalidValue;
    constexpr int W2 = gemm_skinny_nt_waves(v.waves), U2 = v.unroll > 1 ? v.unroll / 2 : 1;
    if (bt)
      hipLaunchKernelGGL((kern::gemm_skinny_tn_kernel<T, v.mt, v.nt, v.waves, v.unroll>), folded_grid(gm * gn),
                         dim3(v.waves * 64), 0, s, a, b, c, (int)M, (int)N, (int)K, (int)gm, (int)gn);
    else
      hipLaunchKernelGGL((kern::gemm_skinny_nt_kernel<T, v.mt, W2, U2>), folded_grid(gm * gn), dim3(W2 * 64), 0, s, a, b,
                         c, (int)M, (int)N, (int)K, (int)gm, (int)gn);
    return hipGetLastError();
  }
}

template <typename T, int... Is>
hipError_t any_dispatch(int variant, bool bt, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                        hipStream_t s, std::integer_sequence<int, Is...>) {
  hipError_t e = hipErrorInvalidValue;
  (void)((kGemmAnyVariants[Is].id == variant &&
          (e = any_go<Is, T>(bt, static_cast<const T*>(A), static_cast<const T*>(B), static_cast<T*>(C), M, N, K, s),
           true)) ||
         ...);
  return e;
}
}  // namespace

hipError_t launch_gemm_any(int variant, DType dt, Layout lay, const void* A, const void* B, void* C, int64_t M, int64_t N,
                           int64_t K, hipStream_t s) {
  if (M <= 0 || N <= 0 || K <= 0 || M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return hipErrorInvalidValue;
  if (lay != Layout::NT && lay != Layout::TN) return hipErrorInvalidValue;
  if ((M + 63) / 64 > 65535) return hipErrorInvalidValue;
  const bool bt = lay == Layout::TN;
  if (gemm_any_asks_alignment(variant, dt == DType::F16, bt, M, N, K) &&
      ((((uintptr_t)A) | ((uintptr_t)B) | ((uintptr_t)C)) & 15))
    return hipErrorInvalidValue;
  constexpr auto seq = std::make_integer_sequence<int, kNumGemmAnyVariants>{};
  if (dt == DType::F16) return any_dispatch<_Float16>(variant, bt, A, B, C, M, N, K, s, seq);
  if (dt == DType::F32) return any_dispatch<float>(variant, bt, A, B, C, M, N, K, s, seq);
  return hipErrorInvalidValue;
}
}  // namespace uk
