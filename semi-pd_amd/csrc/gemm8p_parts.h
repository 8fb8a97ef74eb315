// What the tiled GEMMs of gemm8p.hip and the experts' of moe_gemm_rows.h share: fragments, products, LDS-DMA, waits, the entries of a group.
#pragma once
#include "common.h"
#include "mfma_frag.h"

#include <type_traits>

namespace semipd {

typedef float g8_f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 g8_bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 g8_f16x8 __attribute__((ext_vector_type(8)));

union G8Frag {
  uint4 u;
  g8_bf16x8 b;
  g8_f16x8 f;
};
template <typename T> struct G8Mfma;
template <> struct G8Mfma<bf16_t> {
  __device__ static inline g8_f32x4 mma(const G8Frag& a, const G8Frag& b, g8_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.b, b.b, c, 0, 0, 0);
  }
};
template <> struct G8Mfma<f16_t> {
  __device__ static inline g8_f32x4 mma(const G8Frag& a, const G8Frag& b, g8_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a.f, b.f, c, 0, 0, 0);
  }
};

enum { G8_PLAIN = 0, G8_SILU_MUL = 1 };

#define G8_GLDS(gp, lp, aux) \
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(gp), \
                                   (__attribute__((address_space(3))) void*)(lp), 16, 0, aux)

__device__ inline uint4 g8_lds_read16(uint32_t addr, int imm) {
  uint4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(imm));
  return v;
}
template <int N> __device__ inline void g8_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
__device__ inline void g8_wait_lgkm0() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}
__device__ inline void g8_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Grouped form (GR; fused-MoE expert GEMMs, fused_moe.py:54-273): the x tile is 2 XH consecutive entries of
// sorted_token_ids (moe_align_block_size with block size 2 XH: one expert per tile, expert_ids[tile]); entry id reads
// activation row id / top_k_div and writes output row id (entries >= num_valid are padding), optionally scaled by
// topk_weights[id]; W = w[expert].
struct G8Group {
  const int32_t* sorted_ids;
  const int32_t* expert_ids;
  const int32_t* num_post_pad;
  const float* topk_weights;
  int num_valid, top_k_div, mul_routed_weight;
  uint32_t inverse;                            // (2^32 - 1) / top_k_div
};

// The MFMAs of the 4-wave kernel as inline asm with the accumulator tile tied to an ACCUMULATION register ("+a"): 256 of the
// wave's 512 registers are accumulators, and left to itself the register allocator moves fragments into the accumulation half
// too, spills accumulators and copies them around (1.2 KB of scratch per lane, ~370 v_accvgpr moves inside the K loop in the
// first build).  With the classes fixed -- accumulators in a[0:255], fragments and addresses in v[0:255] -- nothing spills.
// asm volatile also keeps the issue order of a phase: the fragment reads and the DMA first, then the 32 MFMAs.
template <typename T> struct G4Mfma;
template <> struct G4Mfma<bf16_t> {
  __device__ static inline void mma(g8_f32x4& c, const G8Frag& a, const G8Frag& b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a.b), "v"(b.b));
  }
};
template <> struct G4Mfma<f16_t> {
  __device__ static inline void mma(g8_f32x4& c, const G8Frag& a, const G8Frag& b) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a.f), "v"(b.f));
  }
};

// moe_gemm_rows.h: tiles of up to 320 of a group's entries
constexpr int kMoeRowsTile = 320;
template <typename T> int launch_moe_gemm_rows(T* c, const T* a, const T* w, const G8Group& grp, int64_t max_sorted, int N, int K, int epi, hipStream_t st);

}  // namespace semipd
