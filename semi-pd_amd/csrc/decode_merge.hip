// replaces _decode_softmax_reducev_fwd for up to 32 kv splits (layers/attention/triton_ops/decode_attention.py:476-531)
#include "common.h"

namespace semipd {

// The merge of a request's kv splits (stage 2 of decode attention, see decode_attention.hip): up to S splits and two elements a thread, everything
// under way at once: the lengths, which say how many splits there are, their log sums and their elements (of a split without rows too: its
// place is there, what stands in it is not used).  One round trip to memory where stage2_merge takes one for the lengths, one for the log sums
// and one for every element a thread; the sums are the same, in the same order.  Bound by that round trip.  Whole call, us: 16 heads of 512,
// 32 requests of 1100 tokens in 8 splits 20.0 -> 18.9, 1 of 3000 in 32 splits 16.8 -> 14.2; 32 / 8 heads of 128, 1 of 3000 13.7 -> 12.2, 32 of 1100
// 35.8 -> 35.0.  More than 32 splits, or four elements a thread, would hold their registers for nothing: as before.
template <typename T, int S>
__global__ void __launch_bounds__(256)
decode_stage2_at_once_kernel(T* __restrict__ out, const float* __restrict__ attn_logits, const int32_t* __restrict__ kv_indptr, int num_q_heads, int Dv,
                             int64_t o_stride, int num_kv_splits) {
  const int b = blockIdx.x, hq = blockIdx.y, lane = threadIdx.x & 63;
  const float* base = attn_logits + ((int64_t)b * num_q_heads + hq) * num_kv_splits * (Dv + 1);
  const int begin = kv_indptr[b], end = kv_indptr[b + 1], last = num_kv_splits - 1;
  const float log_sum = base[(int64_t)min(lane, last) * (Dv + 1) + Dv];
  const bool two = Dv > (int)blockDim.x;
  float v[2][S];
#pragma unroll
  for (int u = 0; u < 2; ++u)
    if (u == 0 || two)
#pragma unroll
      for (int s = 0; s < S; ++s) v[u][s] = base[(int64_t)min(s, last) * (Dv + 1) + min((int)threadIdx.x + u * (int)blockDim.x, Dv - 1)];
  const int seq_len = end - begin, per_split = (seq_len + num_kv_splits - 1) / num_kv_splits;
  const int n_valid = per_split > 0 ? min(num_kv_splits, (seq_len + per_split - 1) / per_split) : 0;
  const float mine = lane < n_valid ? log_sum : -INFINITY;
  float e_max = mine;
#pragma unroll
  for (int off = S <= 8 ? 4 : S <= 16 ? 8 : 16; off > 0; off >>= 1) e_max = fmaxf(e_max, __shfl_xor(e_max, off, 64));
  e_max = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(e_max)));
  const float w = lane < n_valid ? __expf(mine - e_max) : 0.f;
  float e_sum = 0.f, acc[2] = {};
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < n_valid) {
      const float ws = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(w), s));
      e_sum += ws;
      acc[0] = __builtin_fmaf(ws, v[0][s], acc[0]);
      if (two) acc[1] = __builtin_fmaf(ws, v[1][s], acc[1]);
    }
  const float inv = e_sum > 0.f ? 1.f / e_sum : 0.f;
  T* row = out + (int64_t)b * o_stride + (int64_t)hq * Dv;
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int d = (int)threadIdx.x + u * (int)blockDim.x;
    if ((u == 0 || two) && d < Dv) row[d] = Elem<T>::from_f(acc[u] * inv);
  }
}

template <typename T>
bool launch_stage2_at_once(T* out, const float* attn_logits, const int32_t* kv_indptr, int64_t batch, int num_q_heads, int head_dim_v, int64_t o_stride,
                           int num_kv_splits, int threads, hipStream_t st) {
  if (head_dim_v > 2 * threads || num_kv_splits > 32) return false;
  const dim3 grid((unsigned)batch, (unsigned)num_q_heads);
#define SEMIPD_STAGE2(S) \
  hipLaunchKernelGGL((decode_stage2_at_once_kernel<T, S>), grid, dim3(threads), 0, st, out, attn_logits, kv_indptr, num_q_heads, head_dim_v, o_stride, num_kv_splits)
  if (num_kv_splits <= 8) SEMIPD_STAGE2(8);
  else if (num_kv_splits <= 16) SEMIPD_STAGE2(16);
  else SEMIPD_STAGE2(32);
#undef SEMIPD_STAGE2
  return true;
}

template bool launch_stage2_at_once<bf16_t>(bf16_t*, const float*, const int32_t*, int64_t, int, int, int64_t, int, int, hipStream_t);
template bool launch_stage2_at_once<f16_t>(f16_t*, const float*, const int32_t*, int64_t, int, int, int64_t, int, int, hipStream_t);

}  // namespace semipd
