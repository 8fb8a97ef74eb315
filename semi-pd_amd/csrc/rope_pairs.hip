// RoPE of q and k, with the pool rows of k and v, for batches of prompts (gfx950); smaller batches and other forms: rope_vec_kernel
// (elementwise.hip), whose bits these are.
//
// Neox pairs of whole heads, a workgroup a token: a lane has two items of it, both in flight at once, with the angles of its pairs read
// once for both (the threads of a workgroup are a multiple of a head's items).  Half the threads a token, so all tokens that a CU has of
// such a batch run at once, where a lane an item took them in two rounds of the chain position -> angles -> rows.  32 + 8 heads of
// 128, rows of 16 bits, whole call: 6000 tokens 39.7 -> 27.4 us (5.4 TB/s), 1595 15.5 -> 14.5 (the host's call), in a prefill of three
// prompts 18 us of 2940 less for four layers; 64 + 8 heads, 2000 tokens 27.0 -> 16.1.
#include "common.h"

namespace semipd {

template <typename T, bool STORE, typename KV = T>
__global__ void __launch_bounds__(512)
rope_pairs_kernel(T* __restrict__ q, T* __restrict__ k, const T* __restrict__ v, KV* __restrict__ k_buf, KV* __restrict__ v_buf,
                  const int64_t* __restrict__ loc, const float* __restrict__ cache, const int64_t* __restrict__ positions, int Hq, int Hk, int head,
                  int vhead, int64_t q_stride, int64_t k_stride, int64_t v_stride, int64_t kbuf_stride, int64_t vbuf_stride) {
  constexpr int V = Elem<T>::kVec;
  const int64_t t = blockIdx.x;
  const int half = head >> 1, per_head = half / V, n_q = Hq * per_head, n_rot = (Hq + Hk) * per_head, total = n_rot + (STORE ? Hk * vhead / V : 0);
  const int i0 = (int)(threadIdx.x % per_head) * V;              // first pair of either item
  int64_t dst = 0;
  if (STORE) dst = loc[t];
  Vec16<T> a[2], b[2];
  T* at[2];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int it = threadIdx.x + u * blockDim.x;
    if (it < n_rot) {
      at[u] = it < n_q ? q + t * q_stride + (it / per_head) * head + i0 : k + t * k_stride + (it / per_head - Hq) * head + i0;
      a[u] = load16(at[u]);
      b[u] = load16(at[u] + half);
    } else if (STORE && it < total) {
      a[u] = load16(v + t * v_stride + (int64_t)(it - n_rot) * V);
    }
  }
  const float* cs = cache + positions[t] * head + i0;
  float c[V], sn[V];
#pragma unroll
  for (int j = 0; j < V; ++j) c[j] = cs[j], sn[j] = cs[half + j];
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int it = threadIdx.x + u * blockDim.x;
    if (it < n_rot) {
      Vec16<T> oa, ob;
#pragma unroll
      for (int j = 0; j < V; ++j) {
        float r1, r2;
        rope_pair(Elem<T>::to_f(a[u].e[j]), Elem<T>::to_f(b[u].e[j]), c[j], sn[j], r1, r2);
        oa.e[j] = Elem<T>::from_f(r1);
        ob.e[j] = Elem<T>::from_f(r2);
      }
      store16(at[u], oa);
      store16(at[u] + half, ob);
      if (STORE && it >= n_q) {
        KV* mirror = k_buf + dst * kbuf_stride + (it / per_head - Hq) * head + i0;
        KVTraits<T, KV>::store8(mirror, oa);
        KVTraits<T, KV>::store8(mirror + half, ob);
      }
    } else if (STORE && it < total) {
      KVTraits<T, KV>::store8(v_buf + dst * vbuf_stride + (int64_t)(it - n_rot) * V, a[u]);
    }
  }
}

template <typename T, bool STORE, typename KV>
void launch_rope_pairs(int threads, T* q, T* k, const T* v, KV* k_buf, KV* v_buf, const int64_t* loc, const float* cache, const int64_t* positions,
                       int64_t num_tokens, int Hq, int Hk, int head, int vhead, int64_t q_stride, int64_t k_stride, int64_t v_stride,
                       int64_t kbuf_stride, int64_t vbuf_stride, hipStream_t st) {
  hipLaunchKernelGGL((rope_pairs_kernel<T, STORE, KV>), dim3((unsigned)num_tokens), dim3((unsigned)threads), 0, st, q, k, v, k_buf, v_buf, loc, cache, positions, Hq,
                     Hk, head, vhead, q_stride, k_stride, v_stride, kbuf_stride, vbuf_stride);
}
#define ROPE_PAIRS(T, STORE, KV)                                                                                                               \
  template void launch_rope_pairs<T, STORE, KV>(int, T*, T*, const T*, KV*, KV*, const int64_t*, const float*, const int64_t*, int64_t, int, int, int, int, \
                                                int64_t, int64_t, int64_t, int64_t, int64_t, hipStream_t);
ROPE_PAIRS(float, false, float)
ROPE_PAIRS(bf16_t, false, bf16_t)
ROPE_PAIRS(f16_t, false, f16_t)
ROPE_PAIRS(float, true, float)
ROPE_PAIRS(bf16_t, true, bf16_t)
ROPE_PAIRS(f16_t, true, f16_t)
ROPE_PAIRS(bf16_t, true, f8e5m2_t)
ROPE_PAIRS(bf16_t, true, f8e4m3_t)
ROPE_PAIRS(f16_t, true, f8e5m2_t)
ROPE_PAIRS(f16_t, true, f8e4m3_t)
#undef ROPE_PAIRS

}  // namespace semipd
