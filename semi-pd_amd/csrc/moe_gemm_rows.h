// Grouped GEMM of the experts, up to 320 routed rows x 256 weight rows a workgroup (gfx950): gemm4w_kernel's tile with as many row
// fragments as the tile's expert has rows for.  Compiled in moe_gemm_rows_bf16.hip and _f16.hip.
//
//   c[id] = a[id / top_k_div] @ w[expert]^T  for the entries id of sorted_ids, 320 of one expert at a time (moe_align_block_size)
//
//  * Four waves, 2 x 2, one a SIMD; a wave owns 16 (NX0 + NX1) entries x 128 weight rows, NX0 and NX1 = 2 .. 5 row fragments of 16 in the
//    first half and the second, as many or one less: 128, 160, ... 320 entries a tile, whichever the expert fills (chosen by the workgroup
//    from its entries; a body each).
//  * K in steps of 64.  The operands of a step are four half-tiles in LDS (x0, x1 of 32 NX entries, W0, W1 of 128 weight rows; SiLU * up:
//    W0 gate rows, W1 up rows of the same columns), two steps' worth of them: 144 KB.  Phases, order of the half-tiles, swizzle and
//    waits are those of gemm4w_kernel; loads in flight behind a wait are counted with NX0 or NX1 a wave for an x half and 4 for a W half.
//  * Accumulators: 8 (NX0 + NX1) tiles of 4 registers; 64 of them fill the accumulation half of the register file, those behind
//    that are ordinary registers.
// Bound: the flight of its loads: 64 KB + of a step in LDS twice is all there is room for, 108 KB of it in flight, and behind 94 to 281 rows
// an expert's weights come from HBM once (738 MB of 64 experts of 2816 x 2048: 147 us of a read's time).  Why 320 rows: a second, nearly
// empty tile of 256 took 0.4 of a full one; 320 accumulator registers and 144 KB of LDS are what a CU holds.  Why bodies: a wave's products
// follow its rows in steps of 32 (of 64 before: the layer of 2000 tokens 312 -> 307 us, 3001 362 -> 357, 6000 631 -> 617).  64 experts, top
// 6, bf16, both products, tiles of 256 rows / this: 1000 tokens (94 rows an expert) 183 + 95 / 167 + 81 us, 3001 (281) 296 + 182 / 220 +
// 115, 6000 (562) 477 + 265 / 391 + 208, 8192 572 + 332 / 523 + 294.  Results by way of LDS, in 256 bytes of an entry instead of 32: second
// product of 3001 tokens 134 -> 115 us (74 MB of results).
// Around the K loop nothing overlaps, one workgroup a CU: of 71 us of a tile 4 pass before the first products and 9 (SiLU) or 5 behind
// the last.  So a lane has no division and one wait for its places and weights, conversions are in pairs, and what is staged past the end
// or for padding is no access.  The layer, before / after, us: 1000 tokens 277 / 266, 2000 324 / 312, 3001 375 / 362, 6000 655 / 631, 8192 889 / 850.
#pragma once
#include "gemm8p_parts.h"

namespace semipd {

template <int I, int N, typename F> __device__ __forceinline__ void rows_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    rows_for<I + 1, N>(f);
  }
}

// an accumulator tile in the accumulation half (ACC) or in ordinary registers
template <typename T, bool ACC> __device__ __forceinline__ void rows_mma(g8_f32x4& c, const G8Frag& a, const G8Frag& b) {
  if constexpr (ACC) {
    G4Mfma<T>::mma(c, a, b);
  } else if constexpr (std::is_same<T, bf16_t>::value) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a.b), "v"(b.b));
  } else {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(c) : "v"(a.f), "v"(b.f));
  }
}

// its products retire before it is read (see gemm4w_kernel)
template <bool ACC> __device__ __forceinline__ void rows_retire(g8_f32x4& a, g8_f32x4& b, g8_f32x4& c, g8_f32x4& d) {
  if constexpr (ACC) asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+a"(a), "+a"(b), "+a"(c), "+a"(d));
  else asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}

// the low or the high half of a pair, as a float
template <typename T> __device__ __forceinline__ float half_of(uint32_t w, int high) {
  if constexpr (std::is_same<T, bf16_t>::value) return __uint_as_float(high ? w & 0xffff0000u : w << 16);
  else return Elem<T>::to_f(T{(uint16_t)(high ? w >> 16 : w)});
}

struct RowsTile {
  static constexpr int kRows = kMoeRowsTile, kCols = 256;
  static constexpr int kXHalf = 160 * 128, kWHalf = 128 * 128;         // bytes of a half-tile
  static constexpr int kParity = 2 * (kXHalf + kWHalf), kLds = 2 * kParity;
};

template <typename T, int EPI, int NX0, int NX1, bool NT>
__device__ __forceinline__ void moe_rows_body(char* smem, T* __restrict__ out, const T* __restrict__ x, const T* __restrict__ w, int N, int K,
                                              int m0, int n0, const G8Group& grp) {
  using R = RowsTile;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave >> 1, wc = wave & 1;
  const int c16 = lane & 15, q4 = lane >> 4;
  const int n_cols = EPI == G8_SILU_MUL ? N / 2 : N;
  const int nkt = K >> 6;
  static_assert(NX0 - NX1 >= 0 && NX0 - NX1 <= 1 && NX0 <= 5, "the first half is as long as the second, or one fragment longer: the waits count on it");

  // an entry's row: id / top_k_div, by 2^32 / top_k_div and what is left (35 instructions fewer than the division, of which a lane has 2 NX)
  const uint32_t div = grp.top_k_div, inverse = grp.inverse;
  auto row_of = [&](uint32_t id) __attribute__((always_inline)) {
    const uint32_t q = __umulhi(id, inverse);
    return (int)(q + (id - q * div >= div));
  };

  // ---- DMA sources: piece p of a half-tile is its LDS rows 8 p .. + 7, 128 bytes each; chunk c of row r at c ^ ((r >> 1) & 7) ----
  const int x_bytes = (int)((int64_t)(row_of((uint32_t)grp.num_valid - 1) + 1) * K * 2), w_bytes = (int)((int64_t)N * K * 2);
  int off_x[2][NX0], off_w[2][4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int e = 0; e < (h ? NX1 : NX0); ++e) {
      const int rp = 8 * (wave * (h ? NX1 : NX0) + e) + (lane >> 3);
      const int id = grp.sorted_ids[m0 + 32 * NX0 * h + rp];
      // (padding lies behind the operand's end: zeros that nobody fetches, and products that take little power)
      off_x[h][e] = id < grp.num_valid ? (row_of((uint32_t)id) * K + (((lane & 7) ^ ((rp >> 1) & 7)) << 3)) * 2 : (int)0x80000000;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int rp = 8 * (wave * 4 + e) + (lane >> 3);
      const int wrow = EPI == G8_SILU_MUL ? min(h * (N / 2) + n0 + rp, (h + 1) * (N / 2) - 1) : min(n0 + 128 * (rp >> 6) + 64 * h + (rp & 63), N - 1);
      off_w[h][e] = (wrow * K + (((lane & 7) ^ ((rp >> 1) & 7)) << 3)) * 2;
    }
  }
  const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)smem;
  // piece e of this wave's share of half-tile HALF (0: x0, 1: x1, 2: W0, 3: W1) of K step kt.  Past the end, where the waits still count
  // its loads, the operand has no bytes: nothing is fetched for them.
  auto stage1 = [&](auto half_c, auto e_c, int kt) __attribute__((always_inline)) {
    constexpr int HALF = decltype(half_c)::value, E = decltype(e_c)::value;
    const int k = kt < nkt ? kt * 128 : 0;
    const __amdgpu_buffer_rsrc_t from = __builtin_amdgcn_make_buffer_rsrc((void*)(HALF < 2 ? x : w), 0, kt < nkt ? (HALF < 2 ? x_bytes : w_bytes) : 0, 0x00020000);
    const uint32_t at = lds0 + (kt & 1) * R::kParity;
    if constexpr (HALF < 2)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void*)(uintptr_t)(at + HALF * R::kXHalf + (wave * (HALF ? NX1 : NX0) + E) * 1024), 16,
                                               off_x[HALF][E], k, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(from, (__attribute__((address_space(3))) void*)(uintptr_t)(at + 2 * R::kXHalf + (HALF - 2) * R::kWHalf + (wave * 4 + E) * 1024),
                                               16, off_w[HALF - 2][E], k, 0, NT ? 2 : 0);
  };
  auto stage = [&](auto half_c, int kt) __attribute__((always_inline)) {
    rows_for<0, (decltype(half_c)::value == 0 ? NX0 : decltype(half_c)::value == 1 ? NX1 : 4)>([&](auto e) __attribute__((always_inline)) { stage1(half_c, e, kt); });
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  using H2 = std::integral_constant<int, 2>;
  using H3 = std::integral_constant<int, 3>;

  const int swz = (c16 >> 1) & 7;
  uint32_t off_s[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) off_s[s] = c16 * 128 + (((4 * s + q4) ^ swz) << 4);
  const uint32_t xa = lds0 + wr * (16 * NX0 * 128), xb = lds0 + R::kXHalf + wr * (16 * NX1 * 128);     // this wave's 16 NX rows of an x half
  const uint32_t wa = lds0 + 2 * R::kXHalf + wc * (64 * 128);           // ... and 64 of a W half

  g8_f32x4 acc[NX0 + NX1][8];
#pragma unroll
  for (int i = 0; i < NX0 + NX1; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = g8_f32x4{0.f, 0.f, 0.f, 0.f};
  G8Frag fx0[NX0][2], fx1[NX1][2], fw0[4][2], fw1[4][2];

  // One phase: wait for this wave's share of the half to be read (VM loads behind it may be in flight) and for the last phase's reads,
  // barrier; then 8 NX products of one quadrant with the CNT x 2 reads of RF and the DMA of one half-tile between them.
  auto phase = [&](auto vm_c, auto& rf, uint32_t rbase, auto half_c, int kt, auto& xf, auto& wf, auto i0_c, auto j0_c) __attribute__((always_inline)) {
    constexpr int CNT = sizeof(rf) / sizeof(rf[0]), NX = sizeof(xf) / sizeof(xf[0]), I0 = decltype(i0_c)::value, J0 = decltype(j0_c)::value;
    constexpr int DMA = decltype(half_c)::value == 0 ? NX0 : decltype(half_c)::value == 1 ? NX1 : 4;
    g8_wait_vm<decltype(vm_c)::value>();
    g8_wait_lgkm0();
    g8_barrier();
    rows_for<0, 2 * NX>([&](auto g_c) __attribute__((always_inline)) {
      constexpr int G = decltype(g_c)::value, S = G / NX, I = G % NX;
      rows_for<0, 4>([&](auto j_c) __attribute__((always_inline)) {
        constexpr int J = decltype(j_c)::value;
        rows_mma<T, (I0 + I < 8)>(acc[I0 + I][J0 + J], wf[J][S], xf[I][S]);
      });
      if constexpr (S == 0) {
        rows_for<I * 2 * CNT / NX, (I + 1) * 2 * CNT / NX>([&](auto r_c) __attribute__((always_inline)) {
          constexpr int F = decltype(r_c)::value >> 1, Q = decltype(r_c)::value & 1;
          rf[F][Q].u = g8_lds_read16(rbase + off_s[Q], F * 2048);
        });
      } else {
        rows_for<I * DMA / NX, (I + 1) * DMA / NX>([&](auto e_c) __attribute__((always_inline)) { stage1(half_c, e_c, kt); });
      }
    });
  };
  // loads of the six half-tiles behind one that is waited for: of eight in a row, four x and four W, all but itself and the one before
  constexpr int kAll = 2 * (NX0 + NX1) + 16;
  using XX = std::integral_constant<int, kAll - NX0 - NX1>;
  using X0W = std::integral_constant<int, kAll - NX0 - 4>;
  using X1W = std::integral_constant<int, kAll - NX1 - 4>;
  using WW = std::integral_constant<int, kAll - 8>;
  using IX = std::integral_constant<int, NX0>;
  using J4 = std::integral_constant<int, 4>;

  // (the first weights do not wait for the entries' rows)
  stage(H2{}, 0), stage(H3{}, 0), stage(H0{}, 0), stage(H1{}, 0), stage(H0{}, 1), stage(H3{}, 1), stage(H2{}, 1), stage(H1{}, 1);
  g8_wait_vm<kAll - NX0 - 8>();
  g8_barrier();
  rows_for<0, NX0>([&](auto f) __attribute__((always_inline)) {
    fx0[decltype(f)::value][0].u = g8_lds_read16(xa + off_s[0], decltype(f)::value * 2048);
    fx0[decltype(f)::value][1].u = g8_lds_read16(xa + off_s[1], decltype(f)::value * 2048);
  });
  rows_for<0, 4>([&](auto f) __attribute__((always_inline)) {
    fw0[decltype(f)::value][0].u = g8_lds_read16(wa + off_s[0], decltype(f)::value * 2048);
    fw0[decltype(f)::value][1].u = g8_lds_read16(wa + off_s[1], decltype(f)::value * 2048);
  });
  g8_wait_lgkm0();
  g8_barrier();
  stage(H0{}, 2);

  for (int kt = 0; kt < nkt; kt += 2) {                                // (an even count of K steps: the caller sees to it)
    constexpr uint32_t pa = 0, pb = R::kParity;
    phase(WW{}, fw1, wa + pa + R::kWHalf, H2{}, kt + 2, fx0, fw0, H0{}, H0{});      // reads W1(kt);     W0(kt) -> W0(kt + 2)
    phase(X1W{}, fx1, xb + pa, H3{}, kt + 2, fx0, fw1, H0{}, J4{});      // reads x1(kt);     W1(kt) -> W1(kt + 2)
    phase(XX{}, fx0, xa + pb, H1{}, kt + 2, fx1, fw1, IX{}, J4{});                  // reads x0(kt + 1); x1(kt) -> x1(kt + 2)
    phase(X0W{}, fw1, wa + pb + R::kWHalf, H0{}, kt + 3, fx1, fw0, IX{}, H0{});      // reads W1(kt + 1); x0(kt + 1) -> x0(kt + 3)
    phase(WW{}, fw0, wa + pb, H3{}, kt + 3, fx0, fw1, H0{}, J4{});                  // reads W0(kt + 1); W1(kt + 1) -> W1(kt + 3)
    phase(X1W{}, fx1, xb + pb, H2{}, kt + 3, fx0, fw0, H0{}, H0{});      // reads x1(kt + 1); W0(kt + 1) -> W0(kt + 3)
    phase(XX{}, fx0, xa + pa, H1{}, kt + 3, fx1, fw0, IX{}, H0{});                  // reads x0(kt + 2); x1(kt + 1) -> x1(kt + 3)
    phase(X0W{}, fw0, wa + pa, H0{}, kt + 4, fx1, fw1, IX{}, J4{});                  // reads W0(kt + 2); x0(kt + 2) -> x0(kt + 4)
  }
  // ---- epilogue: lane holds, of entry m0 + 32 NX0 h + 16 NX wr + 16 i + c16, columns 16 j + 4 q4 .. + 3 of its wave's.  A half's rows go
  //      through the wave's own quarter of the LDS and leave whole: 256 bytes of an entry (128 of SiLU * up) instead of 32 a store.  All
  //      entries' places, and their weights, are asked for together ----
  constexpr int WCOLS = EPI == G8_SILU_MUL ? 64 : 128, LPR = WCOLS / 8, RPS = 64 / LPR;      // lanes a row, rows a store
  constexpr int OS = WCOLS * 2 + 16;                                                            // bytes between rows in LDS
  static_assert(16 * NX0 * OS <= R::kLds / 4, "a half's rows fit the wave's quarter");
  char* const mine = smem + wave * (R::kLds / 4);
  int to[2][16 * NX0 / RPS], entry[2][NX0];
  float weight[2][NX0];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int NX = h ? NX1 : NX0;
    const int32_t* ids = grp.sorted_ids + m0 + 32 * NX0 * h + 16 * NX * wr;
#pragma unroll
    for (int i = 0; i < NX; ++i) entry[h][i] = EPI == G8_PLAIN ? ids[16 * i + c16] : 0;
#pragma unroll
    for (int u = 0; u < 16 * NX / RPS; ++u) to[h][u] = ids[RPS * u + lane / LPR];
  }
  g8_wait_vm<0>();                    // no DMA may land in LDS that the next workgroup owns
  g8_wait_lgkm0();
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int i = 0; i < (h ? NX1 : NX0); ++i) weight[h][i] = EPI == G8_PLAIN && grp.mul_routed_weight ? grp.topk_weights[min(entry[h][i], grp.num_valid - 1)] : 1.f;   // (padding has none and is not stored)
  rows_for<0, NX1>([&](auto i_c) __attribute__((always_inline)) {
    constexpr int I = NX0 + decltype(i_c)::value;
    rows_retire<(I < 8)>(acc[I][4], acc[I][5], acc[I][6], acc[I][7]);
  });
  g8_barrier();                       // everybody has read its last fragments and has no DMA in flight
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int NX = h ? NX1 : NX0;
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const float scale = weight[h][i];
#pragma unroll
      for (int j = 0; j < WCOLS / 16; ++j) {
        float r[4];
        if (EPI == G8_SILU_MUL) {
          // the unfused pair rounds the GEMM output to T before the activation reads it
#pragma unroll
          for (int e = 0; e < 4; e += 2) {
            const g8_f32x4 &gate = acc[NX0 * h + i][j], &up = acc[NX0 * h + i][(EPI == G8_SILU_MUL ? 4 : 0) + j];
            const uint32_t g2 = pack2<T>(gate[e], gate[e + 1]), u2 = pack2<T>(up[e], up[e + 1]);
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              const float gq = half_of<T>(g2, b), uq = half_of<T>(u2, b);
              r[e + b] = gq / (1.f + __expf(-gq)) * uq;
              asm volatile("" : "+v"(r[e + b]));   // (see gemm8p_kernel's epilogue: two roundings, not one fused one)
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) r[e] = acc[NX0 * h + i][j][e] * scale;
        }
        *reinterpret_cast<uint2*>(mine + (16 * i + c16) * OS + j * 32 + q4 * 8) = uint2{pack2<T>(r[0], r[1]), pack2<T>(r[2], r[3])};
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int n = n0 + WCOLS * wc + lane % LPR * 8;
#pragma unroll
    for (int u = 0; u < 16 * NX / RPS; ++u) {
      const uint4 v = *reinterpret_cast<const uint4*>(mine + (RPS * u + lane / LPR) * OS + lane % LPR * 16);
      if (to[h][u] < grp.num_valid && n < n_cols) *reinterpret_cast<uint4*>(out + (int64_t)to[h][u] * n_cols + n) = v;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

template <typename T, int EPI>
__global__ void __launch_bounds__(256)
moe_gemm_rows_kernel(T* __restrict__ out, const T* __restrict__ x, const T* __restrict__ w, int N, int K, G8Group grp) {
  extern __shared__ __attribute__((aligned(16))) char g8_smem[];
  const int n_cols = EPI == G8_SILU_MUL ? N / 2 : N;
  constexpr int cols_per_tile = EPI == G8_SILU_MUL ? RowsTile::kCols / 2 : RowsTile::kCols;
  const int tiles_n = (n_cols + cols_per_tile - 1) / cols_per_tile;
  // An XCD (workgroup id % 8) takes a contiguous eighth of the tiles there are.  The column tiles of an expert are next to each other: its
  // rows are fetched into one L2, and a second row tile's are near enough to find the weight tiles there.  Where they are more than half
  // the CUs of an XCD, up to eight row tiles of the expert take turns within them (8 experts of 4096 x 28672, 4096 tokens, top 2: 1800 ->
  // 1640 us; with 11 column tiles, second tiles of 64 rows: 328 -> 382, their short tiles no longer come last).
  const int tiles_m = grp.num_post_pad[0] / RowsTile::kRows, lane = threadIdx.x & 63, at = blockIdx.x >> 3, xcd = blockIdx.x & 7;
  if (tiles_m == 0) return;                                              // (no entry is one of these experts': none of expert_ids is written)
  int tile_m, tile_n, expert;
  bool alone;                                                            // no other row tile reads this one's weight rows
  if (tiles_n > 16 || tiles_m > 256) {
    const int total = tiles_m * tiles_n, per = (total + 7) >> 3, logical = xcd * per + at;
    if (at >= per || logical >= total) return;
    const int near = logical / tiles_n, slot = (near & ~7) + (lane & 7);
    expert = grp.expert_ids[near];
    const uint32_t same = (uint32_t)__ballot(grp.expert_ids[min(slot, tiles_m - 1)] == expert && slot < tiles_m) & 255u;
    const int first = (near & ~7) + __builtin_ctz(same), n_rows = __builtin_popcount(same);
    tile_m = near;
    tile_n = logical - near * tiles_n;
    alone = n_rows == 1;
    if (tiles_n > 16) {
      const int in_group = logical - first * tiles_n;
      tile_n = in_group / n_rows;
      tile_m = first + in_group - tile_n * n_rows;
    }
  } else {
    // The last row tiles of experts that have several come behind all others where they are few: a launch that ends in them ends in short
    // tiles (64 experts, 300 rows each on average, 72 row tiles: 262 -> 230 and 151 -> 132 us).  A bit a row tile: its expert is the one
    // before's, and it is such a last one.
    int ids[4];
    uint64_t again[5] = {}, tails[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int t = 64 * c + lane;
      ids[c] = grp.expert_ids[min(t, tiles_m - 1)];
      again[c] = __ballot(t > 0 && t < tiles_m && grp.expert_ids[max(min(t, tiles_m) - 1, 0)] == ids[c]);
    }
    int n_tails = 0;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      tails[c] = again[c] & ~(again[c] >> 1 | again[c + 1] << 63);
      n_tails += __builtin_popcountll(tails[c]);
    }
    if (n_tails * 8 > tiles_m) n_tails = 0;
    const int heads = (tiles_m - n_tails) * tiles_n, ends = n_tails * tiles_n, per = (heads + 7) >> 3, per_end = (ends + 7) >> 3;
    const bool end = at >= per;
    const int logical = end ? (at - per) + xcd * per_end : at + xcd * per;
    if (end ? at - per >= per_end || logical >= ends : logical >= heads) return;
    tile_m = logical / tiles_n;
    tile_n = logical - tile_m * tiles_n;
    if (n_tails > 0) {                                                   // the tile_m-th of its kind
      int left = tile_m;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const uint64_t there = tiles_m >= 64 * (c + 1) ? ~0ull : tiles_m > 64 * c ? (1ull << (tiles_m - 64 * c)) - 1 : 0ull, kind = end ? tails[c] : there & ~tails[c];
        const int n = __builtin_popcountll(kind);
        if (left >= 0 && left < n) tile_m = 64 * c + __builtin_ctzll(__ballot((kind >> lane & 1) && __builtin_popcountll(kind & ((1ull << lane) - 1)) == left));
        left -= n;
      }
    }
    expert = 0;
    alone = true;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (tile_m >> 6 == c) {
        expert = __builtin_amdgcn_readlane(ids[c], tile_m & 63);
        alone = !((again[c] | (again[c] >> 1 | again[c + 1] << 63)) >> (tile_m & 63) & 1);
      }
  }
  const int m0 = tile_m * RowsTile::kRows, n0 = tile_n * cols_per_tile;
  w += (int64_t)expert * N * K;
  int rows = 0;                                                          // up to the tile's last entry that is no padding
#pragma unroll
  for (int i = 0; i < RowsTile::kRows / 64; ++i) {
    const uint64_t there = __ballot(grp.sorted_ids[m0 + 64 * i + (threadIdx.x & 63)] < grp.num_valid);
    if (there) rows = 64 * i + 64 - __builtin_clzll(there);
  }
  // weight rows that no other workgroup reads leave the L2 to the entries' rows (64 experts of 2048 x 1408 behind 94 rows: 97 -> 89 us, 281
  // rows 143 -> 134; of 1408 x 2816 within the noise)
  const int pairs = max(4, (rows + 31) >> 5);                            // of row fragments, the first half's and the second's
#define ROWS_BODY(ALONE)                                                                                         \
  switch (pairs) {                                                                                               \
    case 4: return moe_rows_body<T, EPI, 2, 2, ALONE>(g8_smem, out, x, w, N, K, m0, n0, grp);                    \
    case 5: return moe_rows_body<T, EPI, 3, 2, ALONE>(g8_smem, out, x, w, N, K, m0, n0, grp);                    \
    case 6: return moe_rows_body<T, EPI, 3, 3, ALONE>(g8_smem, out, x, w, N, K, m0, n0, grp);                    \
    case 7: return moe_rows_body<T, EPI, 4, 3, ALONE>(g8_smem, out, x, w, N, K, m0, n0, grp);                    \
    case 8: return moe_rows_body<T, EPI, 4, 4, ALONE>(g8_smem, out, x, w, N, K, m0, n0, grp);                    \
    case 9: return moe_rows_body<T, EPI, 5, 4, ALONE>(g8_smem, out, x, w, N, K, m0, n0, grp);                    \
    default: return moe_rows_body<T, EPI, 5, 5, ALONE>(g8_smem, out, x, w, N, K, m0, n0, grp);                   \
  }
  if (alone) { ROWS_BODY(true) } else { ROWS_BODY(false) }
#undef ROWS_BODY
}

template <typename T, int EPI>
static int launch_rows(T* c, const T* a, const T* w, const G8Group& grp, int64_t max_sorted, int N, int K, hipStream_t st) {
  const int n_cols = EPI == G8_SILU_MUL ? N / 2 : N, cols_per_tile = EPI == G8_SILU_MUL ? RowsTile::kCols / 2 : RowsTile::kCols;
  const int64_t tiles = max_sorted / RowsTile::kRows * ((n_cols + cols_per_tile - 1) / cols_per_tile);
  // (an XCD's share of the tiles and its share of those that come last are rounded up apart)
  static std::atomic<uint64_t> lds_ok{0};
  if (ensure_dynamic_lds((const void*)moe_gemm_rows_kernel<T, EPI>, RowsTile::kLds, lds_ok, "moe_gemm_rows")) return 1;
  hipLaunchKernelGGL((moe_gemm_rows_kernel<T, EPI>), dim3((unsigned)((tiles + 7) / 8 * 8 + 8)), dim3(256), RowsTile::kLds, st, c, a, w, N, K, grp);
  return launch_status("moe_gemm_rows");
}

template <typename T>
int launch_moe_gemm_rows(T* c, const T* a, const T* w, const G8Group& grp, int64_t max_sorted, int N, int K, int epi, hipStream_t st) {
  return epi == G8_SILU_MUL ? launch_rows<T, G8_SILU_MUL>(c, a, w, grp, max_sorted, N, K, st) : launch_rows<T, G8_PLAIN>(c, a, w, grp, max_sorted, N, K, st);
}
}  // namespace semipd
