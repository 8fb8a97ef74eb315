// Block-scaled fp8 GEMM of the experts of prompts (gfx950): blocks of 128 routed rows x 256 weight rows a workgroup, whole scale blocks of K.
//
//   c[id, n] = sum_kb As[row(id), kb] Ws[n / block_n, kb] (sum_(k in kb) Aq[row(id), k] Wq[n, k])      row(id) = id / top_k_div
//   (the grouped form of w8a8 block fp8 inside fused_moe_kernel, fused_moe_triton/fused_moe.py:174-243)
//
//  * Eight waves, each all 128 rows x 32 weight rows: 16 products v_mfma_scale_f32_16x16x128 a scale block of 128 k (hardware scales 2^0), each
//    folded into its accumulators with its own fp32 scale behind them, in the order of k.
//  * The rows go through LDS, two blocks (16 KB and their scales) in turn, asked for a block ahead of their place; a wave's weight rows
//    are read by it alone and stay in its registers, three blocks in turn, asked for two blocks ahead.  One barrier a block.  (Rows by LDS-DMA:
//    the compiler drains all loads in front of the weights' use then.)  Chunk c (16 bytes) of row r lies at c ^ ((r >> 1) & 7), as in gemm8p.hip.
//  * An XCD (workgroup id % 8) takes a contiguous eighth of the tiles there are, the column tiles of a block next to each other: its
//    rows are fetched into one L2, and the weight rows that several blocks of an expert read are found there.  Experts of more than 24 MB
//    are not: of theirs up to 8 column tiles of every block come first, then the next ones, so that the blocks that are at work share weight
//    rows.  8 experts, 520 rows each, product alone, us, column tiles next to each other / in groups (/ the kernel of all block sizes): 28672 x 4096 1184 / 929
//    (1110), 8192 x 8192 680 / 549 (635), 4096 x 14336 539 / 523 (588), 8192 x 5120 428 / 363 (422); 64 of 4096 x 7168 1928 / 1844 (2104); below the
//    line 64 of 7168 x 2048 1042 / 1113 (1202), 16 of 5120 x 1536 with 64 rows 41.5 / 43.2.
// Bound: of a block's 1.0 k cycles of products a SIMD the folds take as many again (80 vector instructions a wave), the rows' way through LDS 1.0 k of
// the CU's and its loads 0.8 k (48 KB; with 128 weight rows a workgroup, two of them a CU, 64 KB and 1.0 k: 2566 tokens 409 us); behind one block an
// expert the weights' stream.  64 experts of 2048 x 1408, top 6, whole layer, us, the kernel of all block sizes (fp8_gemm.hip: weights one block
// ahead, two barriers a block) / this: 513 tokens 190 / 168, 928 227 / 200, 1500 355 / 310, 2100 400 / 331, 2566 452 / 389, 3000 542 / 461.
#include "common.h"

#include <type_traits>

namespace semipd {

typedef float f8r_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t f8r_u32x4 __attribute__((ext_vector_type(4)));
typedef int f8r_i32x8 __attribute__((ext_vector_type(8)));
typedef int f8r_i32x4 __attribute__((ext_vector_type(4)));

constexpr int kF8Rows = 128, kF8Waves = 8, kF8Cols = 32 * kF8Waves, kF8Block = kF8Rows * 128;      // rows, columns of a tile; bytes of a block's rows
constexpr int64_t kF8LargeExpert = 24 << 20;       // bytes of an expert's weight

struct F8RowsArgs {
  void* c;
  const uint8_t *a, *w;
  const float *a_s, *w_s, *topk_weights;
  const int32_t *sorted_ids, *expert_ids, *num_post_pad;
  int num_valid, N, K, block_n, top_k_div, mul_routed_weight;
  int64_t max_sorted;
};

template <typename OutT>
__global__ void __launch_bounds__(64 * kF8Waves, 2) fp8_rows_kernel(F8RowsArgs p) {
  constexpr int NG = 2, MT = kF8Rows / 16, HALF = MT / 2, NX = 16 / kF8Waves;       // NX: 16-byte pieces of the rows a thread
  __shared__ __attribute__((aligned(16))) uint8_t rows_l[2][kF8Block];
  __shared__ __attribute__((aligned(16))) float scale_l[2][kF8Rows];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c16 = lane & 15, q4 = lane >> 4;
  const int64_t entries = p.num_post_pad[0] < p.max_sorted ? p.num_post_pad[0] : p.max_sorted;
  const int tiles_n = (p.N + kF8Cols - 1) / kF8Cols, tiles_m = (int)((entries + kF8Rows - 1) / kF8Rows), total = tiles_m * tiles_n;
  const int per = (total + 7) >> 3, at = blockIdx.x >> 3, logical = (int)(blockIdx.x & 7) * per + at;
  if (at >= per || logical >= total) return;
  int tile_m = logical / tiles_n, tile_n = logical - tile_m * tiles_n;
  if ((int64_t)p.N * p.K > kF8LargeExpert) {
    const int groups = (tiles_n + 7) >> 3, width = (tiles_n + groups - 1) / groups, group = logical / (tiles_m * width);
    const int within = logical - group * tiles_m * width, cols = min(width, tiles_n - group * width);
    tile_m = within / cols, tile_n = group * width + within - tile_m * cols;
  }
  const int m0 = tile_m * kF8Rows, n0 = tile_n * kF8Cols + 32 * wave;
  const int KB = p.K >> 7, NB = (p.N + p.block_n - 1) / p.block_n;
  const int64_t expert = p.expert_ids[tile_m];
  const int32_t* ids = p.sorted_ids + m0;
  const uint32_t valid = (uint32_t)p.num_valid;
  const int last = (int)(entries - m0 < kF8Rows ? entries - m0 : kF8Rows) - 1;
  // the block's entries, a lane the one of its place in either half (a last block may not be whole); both reads at once, everything in front of
  // the loop takes them from here
  uint32_t id[2] = {(uint32_t)ids[min(lane, last)], (uint32_t)ids[min(64 + lane, last)]};
  asm volatile("" : "+v"(id[0]), "+v"(id[1]));
  if (lane > last) id[0] = valid;
  if (64 + lane > last) id[1] = valid;
  const uint64_t low = __ballot(id[0] < valid), high = __ballot(id[1] < valid);
  if ((low | high) == 0) return;
  const bool upper = high != 0;                                   // (entries behind the padding there are none: up to 64 rows are the lower half's)

  // row of an entry; padding reads row 0 and is not stored
  auto row_of = [&](uint32_t id) { return id < valid ? id / (uint32_t)p.top_k_div : 0u; };
  const uint8_t* src[NX];
  uint32_t to[NX];
#pragma unroll
  for (int e = 0; e < NX; ++e) {
    const int r = 8 * kF8Waves * e + (tid >> 3);
    src[e] = p.a + (int64_t)row_of(__shfl(id[e], r & 63, 64)) * p.K + ((tid & 7) << 4);
    to[e] = r * 128 + (((tid & 7) ^ ((r >> 1) & 7)) << 4);
  }
  const float* src_s = p.a_s + (int64_t)row_of(wave & 1 ? id[1] : id[0]) * KB;
  const uint8_t* wp[NG];
  const float* wsp[NG];
#pragma unroll
  for (int g = 0; g < NG; ++g) {
    const int n = min(n0 + 16 * g + c16, p.N - 1), first = min(n0 + 16 * g, p.N - 1);
    wp[g] = p.w + (expert * p.N + n) * p.K + 16 * q4;
    wsp[g] = p.w_s + (expert * NB + first / p.block_n) * KB;      // (16 | block_n: one scale for a group of 16)
  }
  f8r_i32x8 w[3][NG];
  float ws[3][NG];
  f8r_u32x4 x_next[NX];
  float xs_next;
  auto load_w = [&](auto slot_c, int kb) __attribute__((always_inline)) {     // block kb, past the end the last one (nobody multiplies it)
    constexpr int S = decltype(slot_c)::value;
    const int k = min(kb, KB - 1);
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      w[S][g].lo = *reinterpret_cast<const f8r_i32x4*>(wp[g] + (int64_t)k * 128);
      w[S][g].hi = *reinterpret_cast<const f8r_i32x4*>(wp[g] + (int64_t)k * 128 + 64);
      ws[S][g] = wsp[g][k];
    }
  };
  auto load_x = [&](int kb) __attribute__((always_inline)) {
    const int k = min(kb, KB - 1);
#pragma unroll
    for (int e = 0; e < NX; ++e) x_next[e] = *reinterpret_cast<const f8r_u32x4*>(src[e] + (int64_t)k * 128);
    xs_next = src_s[k];
  };
  auto place_x = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < NX; ++e) *reinterpret_cast<f8r_u32x4*>(rows_l[buf] + to[e]) = x_next[e];
    if (tid < kF8Rows) scale_l[buf][tid] = xs_next;
  };
  f8r_f32x4 acc[NG][MT];
#pragma unroll
  for (int g = 0; g < NG; ++g)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[g][t] = f8r_f32x4{0.f, 0.f, 0.f, 0.f};

  const int swz = (c16 >> 1) & 7;
  const uint32_t lo_at = c16 * 128 + ((q4 ^ swz) << 4), hi_at = c16 * 128 + (((q4 + 4) ^ swz) << 4);       // (a lane's k, of both operands alike)
  union Row {
    f8r_u32x4 u[2];
    f8r_i32x8 v;
  };
  // a half of a block's rows: their operands and scales, then the products of one row tile while those of the one before are folded
  auto half = [&](auto slot_c, auto half_c, int buf) __attribute__((always_inline)) {
    constexpr int S = decltype(slot_c)::value, H = decltype(half_c)::value;
    Row x[HALF];
    float xs[HALF];
#pragma unroll
    for (int t = 0; t < HALF; ++t) {
      x[t].u[0] = *reinterpret_cast<const f8r_u32x4*>(rows_l[buf] + lo_at + (H * HALF + t) * 2048);
      x[t].u[1] = *reinterpret_cast<const f8r_u32x4*>(rows_l[buf] + hi_at + (H * HALF + t) * 2048);
      xs[t] = scale_l[buf][(H * HALF + t) * 16 + c16];
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
    f8r_f32x4 blk[HALF][NG];
#pragma unroll
    for (int t = 0; t < HALF; ++t)
#pragma unroll
      for (int g = 0; g < NG; ++g)
        blk[t][g] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(w[S][g], x[t].v, f8r_f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
#pragma unroll
    for (int t = 0; t < HALF; ++t)
#pragma unroll
      for (int g = 0; g < NG; ++g) {
        const float sc = xs[t] * ws[S][g];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[g][H * HALF + t][e] += blk[t][g][e] * sc;
      }
    __builtin_amdgcn_s_setprio(0);
#pragma unroll
    for (int t = 0; t < HALF; ++t)
#pragma unroll
      for (int g = 0; g < NG; ++g) asm volatile("" : "+v"(acc[g][H * HALF + t]));       // (folded here, not sunk to the loop's end with all operands held until then)
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  auto walk = [&](auto both_c) __attribute__((always_inline)) {
    auto step = [&](auto slot_c, auto next_c, int kb) __attribute__((always_inline)) {
      load_w(next_c, kb + 2);
      half(slot_c, I0{}, kb & 1);
      if constexpr (decltype(both_c)::value) half(slot_c, I1{}, kb & 1);
      place_x((kb + 1) & 1);          // (read last in step kb - 1)
      load_x(kb + 2);
      __syncthreads();
    };
    int kb = 0;
    for (; kb + 3 <= KB; kb += 3) {
      step(I0{}, I2{}, kb);
      step(I1{}, I0{}, kb + 1);
      step(I2{}, I1{}, kb + 2);
    }
    if (kb < KB) step(I0{}, I2{}, kb);
    if (kb + 1 < KB) step(I1{}, I0{}, kb + 1);
  };
  load_x(0);
  load_w(I0{}, 0);
  load_w(I1{}, 1);
  place_x(0);
  load_x(1);
  __syncthreads();
  if (upper) walk(std::true_type{});
  else walk(std::false_type{});

  // lane holds c[entry 16 t + c16][n0 + 16 g + 4 q4 .. + 3]
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    if (!((t < MT / 2 ? low : high) >> (16 * (t % (MT / 2)) + c16) & 1)) continue;
    const uint32_t id = (uint32_t)ids[16 * t + c16];
    const float scale = p.mul_routed_weight ? p.topk_weights[id] : 1.f;
    OutT* dst = (OutT*)p.c + (int64_t)id * p.N + n0 + 4 * q4;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (n0 + 16 * g >= p.N) continue;
      const f8r_f32x4 v = acc[g][t] * scale;
      if constexpr (sizeof(OutT) == 4) {
        *reinterpret_cast<float4*>(dst + 16 * g) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
        uint2 u;
        u.x = (uint32_t)Elem<OutT>::from_f(v[0]).v | ((uint32_t)Elem<OutT>::from_f(v[1]).v << 16);
        u.y = (uint32_t)Elem<OutT>::from_f(v[2]).v | ((uint32_t)Elem<OutT>::from_f(v[3]).v << 16);
        *reinterpret_cast<uint2*>(dst + 16 * g) = u;
      }
    }
  }
}

// K % 128 == 0, N % 16 == 0, c aligned to 16 bytes, blocks of 128 entries: the caller sees to it
int launch_fp8_rows_grouped(void* c, const void* a, const float* a_s, const void* w, const float* w_s, const float* topk_weights, const int32_t* sorted_ids,
                            const int32_t* expert_ids, const int32_t* num_post_pad, int num_valid, int N, int K, int64_t max_sorted, int block_n, int top_k_div,
                            int mul_routed_weight, int out_dtype, hipStream_t st) {
  const F8RowsArgs p{c, (const uint8_t*)a, (const uint8_t*)w, a_s, w_s, topk_weights, sorted_ids, expert_ids, num_post_pad, num_valid, N, K, block_n, top_k_div, mul_routed_weight, max_sorted};
  const int64_t tiles = (max_sorted + kF8Rows - 1) / kF8Rows * ((N + kF8Cols - 1) / kF8Cols);
  const dim3 grid((unsigned)((tiles + 7) / 8 * 8));
  switch (out_dtype) {
    case SEMIPD_BF16: hipLaunchKernelGGL((fp8_rows_kernel<bf16_t>), grid, dim3(64 * kF8Waves), 0, st, p); break;
    case SEMIPD_F16: hipLaunchKernelGGL((fp8_rows_kernel<f16_t>), grid, dim3(64 * kF8Waves), 0, st, p); break;
    case SEMIPD_F32: hipLaunchKernelGGL((fp8_rows_kernel<float>), grid, dim3(64 * kF8Waves), 0, st, p); break;
    default:
      set_error("moe_grouped_gemm_fp8: output dtype code %d is not f32 / bf16 / f16", out_dtype);
      return SEMIPD_EDTYPE;
  }
  return launch_status("fp8_rows_grouped");
}

}  // namespace semipd
