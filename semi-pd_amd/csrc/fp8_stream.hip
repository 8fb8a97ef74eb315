// Block-scaled fp8 expert GEMMs of decode batches, weights through LDS-DMA (gfx950): the grouped form of stream_linear.hip's kernel in
// bytes, for semipd_moe_grouped_gemm_fp8 (fp8_gemm.hip).
//
//   c[id, n] = sum_kb (sum_{k in block kb} a_q[row, k] * w_q[expert, n, k]) * a_s[row, kb] * w_s[expert, n / block_n, kb],  row = id / top_k_div,
// for the entries id of a block of 16 MT of sorted_ids (one expert each), times topk_weights[id] where asked.
//
//  * A wave owns 16 weight rows and a private ring of R slots of 256 bytes of each (4 KB, two scale blocks), R - 1 in flight; the activation
//    rows of the same 256 bytes go through a ring of the workgroup's.  A DMA instruction takes four rows' 256 contiguous bytes; chunk c of
//    row r lies at c ^ r of its 256.  A row's activation scales are in LDS ([scale block][row]) from the start, the weight scales of a wave
//    in a register, a lane each.
//  * A scale block of 128 bytes is one v_mfma_scale_f32_16x16x128_f8f6f4 a tile (hardware scales 2^0) and folded in with one product of
//    scales and four multiply-adds.  K of an uneven count of scale blocks: the last slot holds its first 128 bytes twice, the second with scale 0.
// Bound: the weight stream.  The register-fragment form (fp8_block_gemm_kernel: 16 rows x 64 bytes an instruction, blocks of 64 rows) ran it
// at 3.7 TB/s of a whole layer's time: 64 experts of 2048 x 1408, top 6, 32 tokens 142 -> 108 us, 16 122 -> 94, 128 160 -> 126, 320 183 -> 155.
#include "common.h"

namespace semipd {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

template <int MT, int NW> struct F8Stream {
  static constexpr int R = 3;
  static constexpr int kXStage = MT * 4096, kWSlot = 4096;
  static constexpr int kRings = R * (kXStage + NW * kWSlot);
  static constexpr int kNX = (4 * MT + NW - 1) / NW;             // activation pieces a wave issues per slot
  static constexpr int kPerSlot = kNX + 4;
  __host__ __device__ static int scale_pieces(int nkb) { return (2 * nkb * 16 * MT + 63) / 64; }      // of 64 activation scales
  static size_t lds(int K) { return kRings + (size_t)scale_pieces((K + 255) / 256) * 256; }
};

__device__ __forceinline__ i32x4 f8s_read16(uint32_t addr) {
  i32x4 v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}
__device__ __forceinline__ float f8s_read4(uint32_t addr) {
  float v;
  asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}
template <int N> __device__ __forceinline__ void f8s_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
template <int N> __device__ __forceinline__ void f8s_wait_lgkm() {
  asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
  __builtin_amdgcn_sched_barrier(0);
}
#define F8S_DMA(FROM, TO, BYTES, AUX)                                                           \
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(FROM),       \
                                   (__attribute__((address_space(3))) void*)(TO), BYTES, 0, AUX)

template <typename OutT, int MT, int NW>
__global__ void __launch_bounds__(64 * NW)
fp8_stream_grouped_kernel(OutT* __restrict__ c, const uint8_t* __restrict__ a, const float* __restrict__ a_s, const uint8_t* __restrict__ w,
                          const float* __restrict__ w_s, const float* __restrict__ topk_weights, const int32_t* __restrict__ sorted_ids,
                          const int32_t* __restrict__ expert_ids, const int32_t* __restrict__ num_post_pad, int num_valid, int N, int K,
                          int block_n, int top_k_div, int mul_routed_weight) {
  using L = F8Stream<MT, NW>;
  constexpr int R = L::R, BM = 16 * MT;
  static_assert(64 % BM == 0, "a lane's rows of the scales are one row");
  extern __shared__ __attribute__((aligned(16))) char f8_smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c16 = lane & 15, q4 = lane >> 4;
  const int m_blk = (int)blockIdx.y * BM;
  if (m_blk >= num_post_pad[0]) return;
  const int KB = K >> 7, nkb = (K + 255) >> 8;
  const int64_t expert = expert_ids[blockIdx.y];
  const int n0 = ((int)blockIdx.x * NW + wave) * 16;             // (N % 16 == 0: past the end, rows of the last group again, not stored)
  const int n_at = min(n0, N - 16);
  auto row_of = [&](int m) __attribute__((always_inline)) {      // (padding reads row 0)
    const int id = sorted_ids[m_blk + m];
    return (int64_t)(id < num_valid ? id / top_k_div : 0);
  };

  // ---- sources: piece j = rows 4 j .. + 3 of 16, lane -> row 4 j + (lane >> 4), chunk (lane & 15) ^ row of its 256 bytes ----
  const uint8_t* wsrc[4];
  int fold_w[4];                                                 // what a lane steps back by in a last slot of one scale block
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int i = 4 * j + q4, chunk = c16 ^ i;
    wsrc[j] = w + (expert * N + n_at + i) * K + chunk * 16;
    fold_w[j] = chunk >= 8 ? 128 : 0;
  }
  const uint8_t* xsrc[L::kNX];
  int xdst[L::kNX], fold_x[L::kNX];
#pragma unroll
  for (int e = 0; e < L::kNX; ++e) {
    const int piece = (wave + e * NW) % (4 * MT), i = 4 * (piece & 3) + q4, chunk = c16 ^ i;      // (a piece twice where 4 MT % NW != 0: the same bytes)
    xsrc[e] = a + row_of((piece >> 2) * 16 + i) * K + chunk * 16;
    xdst[e] = piece * 1024;
    fold_x[e] = chunk >= 8 ? 128 : 0;
  }
  const float* const srow = a_s + row_of(lane % BM) * KB;
  const float ws_of = w_s[(expert * ((N + block_n - 1) / block_n) + n_at / block_n) * KB + min(lane, KB - 1)];      // (K <= 8192: a lane a scale block)

  char* const xring = f8_smem;
  char* const wring = f8_smem + R * L::kXStage + wave * (R * L::kWSlot);
  char* const scales = f8_smem + L::kRings;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)f8_smem;
  const uint32_t xring_at = lds0, wring_at = lds0 + R * L::kXStage + wave * (R * L::kWSlot), scales_at = lds0 + L::kRings + c16 * 4;
  // (in front of the slots: every wait for one covers these)
  for (int p = wave; p < L::scale_pieces(nkb); p += NW) F8S_DMA(srow + min(p * (64 / BM) + lane / BM, KB - 1), scales + p * 256, 4, 0);
  auto issue = [&](int kb) __attribute__((always_inline)) {
    const int64_t k = (int64_t)kb * 256;
    const bool fold = 2 * kb + 1 >= KB;
#pragma unroll
    for (int e = 0; e < L::kNX; ++e) F8S_DMA(xsrc[e] + (k - (fold ? fold_x[e] : 0)), xring + (kb % R) * L::kXStage + xdst[e], 16, 0);
#pragma unroll
    for (int j = 0; j < 4; ++j) F8S_DMA(wsrc[j] + (k - (fold ? fold_w[j] : 0)), wring + (kb % R) * L::kWSlot + j * 1024, 16, 2);
  };

  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  uint32_t frag[2][2];                                           // scale block, half of this lane's 32 bytes of it
#pragma unroll
  for (int sb = 0; sb < 2; ++sb)
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) frag[sb][hf] = c16 * 256 + (((8 * sb + 2 * q4 + hf) ^ c16) << 4);

#pragma unroll
  for (int p = 0; p < R - 1; ++p)
    if (p < nkb) issue(p);
  for (int kb = 0; kb < nkb; ++kb) {
    if (kb + R - 1 <= nkb) f8s_wait_vm<(R - 2) * L::kPerSlot>();
    else f8s_wait_vm<0>();
    __builtin_amdgcn_s_barrier();       // every wave's share of the slot is in, everybody is done with the one before
    asm volatile("" ::: "memory");
    if (kb + R - 1 < nkb) issue(kb + R - 1);
    const uint32_t xs = xring_at + (kb % R) * L::kXStage, wl = wring_at + (kb % R) * L::kWSlot, sc = scales_at + kb * (2 * BM * 4);
    i32x8 av[2], bv[2][MT];
    float as[2][MT];
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      av[sb].lo = f8s_read16(wl + frag[sb][0]);
      av[sb].hi = f8s_read16(wl + frag[sb][1]);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        bv[sb][t].lo = f8s_read16(xs + t * 4096 + frag[sb][0]);
        bv[sb][t].hi = f8s_read16(xs + t * 4096 + frag[sb][1]);
        as[sb][t] = f8s_read4(sc + (sb * BM + t * 16) * 4);
      }
    }
#pragma unroll
    for (int sb = 0; sb < 2; ++sb) {
      if (sb == 0) f8s_wait_lgkm<2 + 3 * MT>();
      else f8s_wait_lgkm<0>();
      const int at = 2 * kb + sb;
      const float ws = at < KB ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ws_of), at)) : 0.f;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const f32x4 blk = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(av[sb], bv[sb][t], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
        const float s = as[sb][t] * ws;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[t][e] = __builtin_fmaf(blk[e], s, acc[t][e]);
      }
    }
  }

  // ---- lane holds c[m = 16 t + c16][n = n0 + 4 q4 .. + 3] ----
  if (n0 >= N) return;
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int id = sorted_ids[m_blk + t * 16 + c16];
    if (id >= num_valid || id < 0) continue;
    const float scale = mul_routed_weight ? topk_weights[id] : 1.f;
    OutT* dst = c + (int64_t)id * N + n0 + q4 * 4;
    if constexpr (sizeof(OutT) == 4) {
      *reinterpret_cast<float4*>(dst) = make_float4(acc[t][0] * scale, acc[t][1] * scale, acc[t][2] * scale, acc[t][3] * scale);
    } else {
      uint2 p;
      p.x = (uint32_t)Elem<OutT>::from_f(acc[t][0] * scale).v | ((uint32_t)Elem<OutT>::from_f(acc[t][1] * scale).v << 16);
      p.y = (uint32_t)Elem<OutT>::from_f(acc[t][2] * scale).v | ((uint32_t)Elem<OutT>::from_f(acc[t][3] * scale).v << 16);
      *reinterpret_cast<uint2*>(dst) = p;
    }
  }
}

template <typename OutT, int MT, int NW>
static int launch_fp8_stream(void* c, const void* a, const float* a_s, const void* w, const float* w_s, const float* topk_weights,
                             const int32_t* sorted_ids, const int32_t* expert_ids, const int32_t* num_post_pad, int num_valid, int N, int K,
                             int blocks, int block_n, int top_k_div, int mul_routed_weight, hipStream_t st) {
  using L = F8Stream<MT, NW>;
  static std::atomic<uint64_t> lds_ok{0};
  const size_t lds = L::lds(K);
  if (ensure_dynamic_lds((const void*)fp8_stream_grouped_kernel<OutT, MT, NW>, L::lds(8192), lds_ok, "fp8_stream_grouped")) return 1;
  hipLaunchKernelGGL((fp8_stream_grouped_kernel<OutT, MT, NW>), dim3((unsigned)((N + 16 * NW - 1) / (16 * NW)), (unsigned)blocks), dim3(64 * NW),
                     lds, st, (OutT*)c, (const uint8_t*)a, a_s, (const uint8_t*)w, w_s, topk_weights, sorted_ids, expert_ids,
                     num_post_pad, num_valid, N, K, block_n, top_k_div, mul_routed_weight);
  return launch_status("fp8_stream_grouped");
}
#undef F8S_DMA

// blocks of 16, 32 or 64 entries; K % 128, K <= 8192, N % 16, c 16-byte aligned (the caller has checked)
int launch_fp8_stream_grouped(void* c, const void* a, const float* a_s, const void* w, const float* w_s, const float* topk_weights,
                              const int32_t* sorted_ids, const int32_t* expert_ids, const int32_t* num_post_pad, int num_valid, int N, int K,
                              int blocks, int block_m, int block_n, int top_k_div, int mul_routed_weight, int out_dtype, hipStream_t st) {
#define GO(OutT, MT, NW)                                                                                                                       \
  return launch_fp8_stream<OutT, MT, NW>(c, a, a_s, w, w_s, topk_weights, sorted_ids, expert_ids, num_post_pad, num_valid, N, K, blocks, block_n, \
                                         top_k_div, mul_routed_weight, st)
  // (two workgroups of four waves a CU, one of eight where the activations' ring is 16 KB a slot; 32 tokens, blocks of 32: 115 us, in
  // workgroups of eight waves 120, of two 130)
#define GO_MT(OutT)                    \
  do {                                 \
    if (block_m == 16) GO(OutT, 1, 4); \
    if (block_m == 32) GO(OutT, 2, 4); \
    GO(OutT, 4, 8);                    \
  } while (0)
  switch (out_dtype) {
    case SEMIPD_BF16: GO_MT(bf16_t);
    case SEMIPD_F16: GO_MT(f16_t);
    case SEMIPD_F32: GO_MT(float);
  }
#undef GO_MT
#undef GO
  set_error("moe_grouped_gemm_fp8: output dtype code %d is not f32 / bf16 / f16", out_dtype);
  return SEMIPD_EDTYPE;
}

}  // namespace semipd
