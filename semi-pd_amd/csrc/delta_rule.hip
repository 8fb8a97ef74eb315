// Gated delta rule over a pool of per-request state rows (gfx950, wave64).
//
// Per head, a matrix S [D, E] in fp32 that starts at zero and is carried from token to token:
//     S <- g_t S;   u_t = beta_t (v_t - S^T k_t);   S <- S + k_t u_t^T;   o_t = S^T q_t
// with q, k unit vectors per head (q also times D^-1/2), g_t = exp(-exp(A_log) softplus(a_t + dt_bias)) and
// beta_t = sigmoid(b_t) one number per head and token.  q, k and v first pass a short causal convolution over time per
// channel and silu; the last taps - 1 inputs of every channel are part of the request's state.  Several heads may share a
// q / k head.  Everything behind the projection GEMM is fp32 whatever the activation type.
//
//  * delta_prep_kernel: a workgroup per token, its waves taking the token's q, k and v heads in turn: convolution (inputs in
//    front of the portion come from the state row), silu, unit norms, decay and beta -> an fp32 work row per token.
//  * delta_conv_state: the last taps - 1 inputs of the portion (shifted in behind what the row held) -> state row, by the first workgroups
//    of delta_post_vec_kernel's launch or in delta_conv_state_kernel.
//  * delta_scan_kernel: ONE WAVE per (request, head, block of columns); column j of S lives in the registers of DS adjacent
//    lanes (D / DS rows each), so a step is two dot products over the lanes' rows, a 2-step lane reduction and one update
//    of the column: dk = S^T k, dq = S^T q from the old S, then u = beta (v - g dk), o = g dq + u (k . q), S <- g S + k u
//    (the same values as the sequence above: the read-out sees the current token's write).  k, q, v of kStage tokens come in
//    as 16-byte pieces that are in flight a stage ahead and sit in LDS (k . q, g, beta beside them); o leaves the same way.
//    The state is read when the rows of the launch do not start the sequence and written back after the last row, so a
//    prompt cut into portions, single decode tokens and a slot that another request held all take one path.
//  * Prompt batches: delta_chunk_operands_kernel and delta_chunk_walk_kernel (keys of up to 64: delta_chunk_walk_small_kernel) in place of
//    the three, 32 tokens at a time on the matrix cores, operands of 24 bits and fp32 sums.
//  * delta_post_kernel / delta_post_vec_kernel: o / rms(o) * weight * silu(gate) -> the output projection's input, a workgroup per token.
//  * delta_step_kernel / delta_decode_kernel: all of the above for batches of one token per request, a workgroup per (request, key
//    head) where the state lies on 16-byte boundaries, else per (request, head).
#include <cstring>
#include <type_traits>

#include "common.h"
#include "recurrent_chunks.h"

namespace semipd {

struct DeltaArgs {
  const void* p; int64_t ld;                       // projection rows: q | k | v | gate | a | b at the offsets below
  int64_t q_off, k_off, v_off, gate_off, a_off, b_off;
  const void* conv_q; const void* conv_k; const void* conv_v;    // [channels, taps] of the activation type
  const float* a_log; const float* dt_bias;        // [H] fp32
  const void* norm_w;                              // [E] of the activation type
  float* work; int64_t wld;                        // fp32 [T, wld]: q [G D] | k [G D] | v, later o [H E] | g [H] | beta [H]
  float* state; int64_t state_ld;                  // fp32 [slots, >= H D E]: S[h][d][e]
  float* conv_state; int64_t conv_ld;              // fp32 [slots, >= (taps - 1) C]: [tap][channel], C = 2 G D + H E
  const int64_t* state_indices; const int64_t* seq_lens;
  const int32_t* q_start; const int32_t* q_len;    // [B] or NULL (one row per request)
  int64_t batch, num_tokens;
  int H, G, D, E, taps;
  float eps;
  void* out; int64_t out_ld;                       // [T, H E] of the activation type
  int o_off;                                       // column of o in a work row: 2 G D, in the matrix-core form (rows of o alone) 0
  float* frags;                                    // operands of the chunks (matrix-core form), see delta_chunk_operands_kernel
};

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }
__device__ __forceinline__ float silu_f(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float softplus_f(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// two adjacent elements in one access
template <typename T> __device__ __forceinline__ void load2(const T* p, float& x0, float& x1) {
  if constexpr (sizeof(T) == 2) {
    const uint32_t w = *reinterpret_cast<const uint32_t*>(p);
    T lo, hi;
    lo.v = (uint16_t)(w & 0xffffu);
    hi.v = (uint16_t)(w >> 16);
    x0 = Elem<T>::to_f(lo);
    x1 = Elem<T>::to_f(hi);
  } else {
    const float2 w = *reinterpret_cast<const float2*>(p);
    x0 = w.x;
    x1 = w.y;
  }
}

// the sum over groups of 2 / 4 adjacent lanes, in every lane of the group (data-parallel-primitive moves inside a quad)
template <int DS> __device__ __forceinline__ float quad_sum(float x) {
  if (DS >= 2) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0xB1, 0xF, 0xF, true));   // lane ^ 1
  if (DS >= 4) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x4E, 0xF, 0xF, true));   // lane ^ 2
  return x;
}

// the request that owns row t, the row's index inside the request's portion, the portion's length and its first position
__device__ __forceinline__ bool delta_locate(const DeltaArgs& a, int64_t t, int& b, int64_t& li, int64_t& n, int64_t& first_pos) {
  if (a.q_start == nullptr) {
    b = (int)t;
    li = 0;
    n = 1;
    first_pos = a.seq_lens[b] - 1;
    return first_pos >= 0;
  }
  for (int r = 0; r < (int)a.batch; ++r) {
    const int64_t s = a.q_start[r], m = a.q_len[r];
    if (t >= s && t < s + m) {
      b = r;
      li = t - s;
      n = m;
      first_pos = a.seq_lens[r] - m;
      return true;
    }
  }
  return false;
}

// ---------------------------------------------------------------------------------- convolution, silu, norms, gates
template <typename T>
__global__ void __launch_bounds__(256) delta_prep_kernel(DeltaArgs a) {
  // a workgroup per token; its waves take the token's units (q heads, k heads, v heads) in turn
  const int lane = threadIdx.x & 63;
  const int units = 2 * a.G + a.H;
  const int64_t t = blockIdx.x;
  int b;
  int64_t li, n, first_pos;
  if (!delta_locate(a, t, b, li, n, first_pos)) return;
  const int D = a.D, E = a.E, G = a.G, taps = a.taps;
  const int C = 2 * G * D + a.H * E;
  const T* p = (const T*)a.p;
  const float* cs = a.conv_state + a.state_indices[b] * a.conv_ld;
  const bool fresh = first_pos == 0;
  for (int u = threadIdx.x >> 6; u < units; u += 4) {
  // unit u: q head u, k head u - G, or v head u - 2 G
  const bool is_v = u >= 2 * G;
  const int size = is_v ? E : D;
  const int64_t col0 = is_v ? a.v_off + (int64_t)(u - 2 * G) * E : (u < G ? a.q_off + (int64_t)u * D : a.k_off + (int64_t)(u - G) * D);
  const int ch0 = is_v ? 2 * G * D + (u - 2 * G) * E : u * D;               // channel in the state's order (q | k | v)
  const T* cw = is_v ? (const T*)a.conv_v + (int64_t)(u - 2 * G) * E * taps
                     : (u < G ? (const T*)a.conv_q + (int64_t)u * D * taps : (const T*)a.conv_k + (int64_t)(u - G) * D * taps);
  float* w = a.work + t * a.wld + (is_v ? 2 * G * D + (u - 2 * G) * E : u * D);
  float sq = 0.f;
  // two adjacent channels per lane in one access each when everything is even (the work rows and the state rows are)
  const bool two = ((size | D | E) & 1) == 0 && ((col0 | a.ld | a.conv_ld) & 1) == 0;
  for (int c = 2 * lane; two && c < size; c += 128) {
    float y0 = 0.f, y1 = 0.f;
    for (int i = 0; i < taps; ++i) {
      const int64_t l = li - i;
      float x0 = 0.f, x1 = 0.f;
      if (l >= 0) load2(p + (t - i) * a.ld + col0 + c, x0, x1);
      else if (!fresh) {
        const float2 x = *reinterpret_cast<const float2*>(cs + (int64_t)(taps - 1 + l) * C + ch0 + c);
        x0 = x.x;
        x1 = x.y;
      }
      y0 += Elem<T>::to_f(cw[(int64_t)c * taps + (taps - 1 - i)]) * x0;
      y1 += Elem<T>::to_f(cw[(int64_t)(c + 1) * taps + (taps - 1 - i)]) * x1;
    }
    y0 = silu_f(y0);
    y1 = silu_f(y1);
    sq += y0 * y0 + y1 * y1;
    *reinterpret_cast<float2*>(w + c) = float2{y0, y1};
  }
  for (int c = lane; !two && c < size; c += 64) {
    float y = 0.f;
    for (int i = 0; i < taps; ++i) {
      const int64_t l = li - i;
      float x;
      if (l >= 0) x = Elem<T>::to_f(p[(t - i) * a.ld + col0 + c]);
      else if (fresh) x = 0.f;
      else x = cs[(int64_t)(taps - 1 + l) * C + ch0 + c];
      y += Elem<T>::to_f(cw[(int64_t)c * taps + (taps - 1 - i)]) * x;
    }
    y = silu_f(y);
    sq += y * y;
    w[c] = y;
  }
  if (!is_v) {
    sq = wave_sum(sq);
    const float inv = (u < G ? rsqrtf((float)D) : 1.0f) / sqrtf(sq + 1e-6f);
    for (int c = 2 * lane; two && c < size; c += 128) {      // (each lane rescales what it wrote itself)
      w[c] *= inv;
      w[c + 1] *= inv;
    }
    for (int c = lane; !two && c < size; c += 64) w[c] *= inv;
  } else if (lane == 0) {
    const int h = u - 2 * G;
    const float av = Elem<T>::to_f(p[t * a.ld + a.a_off + h]), bv = Elem<T>::to_f(p[t * a.ld + a.b_off + h]);
    float* gb = a.work + t * a.wld + C;
    gb[h] = expf(-expf(a.a_log[h]) * softplus_f(av + a.dt_bias[h]));
    gb[a.H + h] = sigmoid_f(bv);
  }
  }
}

// ---------------------------------------------------------------------------------- the inputs the next portion looks back at
template <typename T>
__device__ __forceinline__ void delta_conv_state(const DeltaArgs& a, int b, int c) {
  const int C = 2 * a.G * a.D + a.H * a.E;
  if (c >= C) return;
  int64_t t0, n, first_pos;
  if (a.q_start == nullptr) {
    t0 = b; n = 1; first_pos = a.seq_lens[b] - 1;
  } else {
    t0 = a.q_start[b]; n = a.q_len[b]; first_pos = a.seq_lens[b] - n;
  }
  if (n <= 0 || first_pos < 0) return;
  const int GD = a.G * a.D;
  const int64_t col = c < GD ? a.q_off + c : (c < 2 * GD ? a.k_off + (c - GD) : a.v_off + (c - 2 * GD));
  float* cs = a.conv_state + a.state_indices[b] * a.conv_ld;
  const T* p = (const T*)a.p;
  const int keep = a.taps - 1;
  // entry s of the new state is the input at index n - keep + s of the portion; a negative index reaches into the old
  // state (entry s + n > s, read before entry s is written) or, at the start of a sequence, in front of it
  auto input = [&](int s) {
    const int64_t l = n - keep + s;
    if (l >= 0) return Elem<T>::to_f(p[(t0 + l) * a.ld + col]);
    return first_pos == 0 ? 0.f : cs[(int64_t)(keep + l) * C + c];
  };
  if (keep <= kRecHalo) {                                        // (read at once, then written: not a round trip each)
    float x[kRecHalo];
#pragma unroll
    for (int s = 0; s < kRecHalo; ++s) x[s] = s < keep ? input(s) : 0.f;
#pragma unroll
    for (int s = 0; s < kRecHalo; ++s)
      if (s < keep) cs[(int64_t)s * C + c] = x[s];
    return;
  }
  for (int s = 0; s < keep; ++s) cs[(int64_t)s * C + c] = input(s);
}
template <typename T>
__global__ void __launch_bounds__(256) delta_conv_state_kernel(DeltaArgs a) {
  delta_conv_state<T>(a, blockIdx.y, blockIdx.x * 256 + threadIdx.x);
}

// ---------------------------------------------------------------------------------- the recurrence
constexpr int kStage = 16;      // tokens whose k, q and scalars sit in LDS at a time

template <int DPT, int DS>
__global__ void __launch_bounds__(64) delta_scan_kernel(DeltaArgs a) {
  // per staged token: k and q, each as DS slices of DPT elements with 4 elements of padding behind every slice (the DS lanes
  // of a column read 16-byte pieces of different banks), then k . q, g, beta; then the block's columns of v, later o
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int DP = DPT * DS, SL = DPT + 4, KQ = 2 * DS * SL;
  constexpr int COLS = 64 / DS;                                    // columns of S per workgroup (one wave)
  constexpr int NV = (kStage * 2 * DP / 4 + 63) / 64;              // 16-byte pieces of k | q per lane and stage
  constexpr int NO = (kStage * COLS / 4 + 63) / 64;                // ... of v / o
  const int b = blockIdx.x, h = blockIdx.y;
  const int D = a.D, E = a.E, G = a.G, H = a.H;
  const int gk = h / (H / G);
  int64_t t0, n, first_pos;
  if (a.q_start == nullptr) {
    t0 = b; n = 1; first_pos = a.seq_lens[b] - 1;
  } else {
    t0 = a.q_start[b]; n = a.q_len[b]; first_pos = a.seq_lens[b] - n;
  }
  if (n <= 0 || first_pos < 0) return;
  const int tid = threadIdx.x;
  const int s = tid % DS;
  const int C = 2 * G * D + H * E;
  float* kq_l = lds;
  float* sc_l = lds + kStage * KQ;
  float* vo_l = sc_l + kStage * 4;
  float* st = a.state + a.state_indices[b] * a.state_ld + (int64_t)h * D * E;
  const int jc = tid / DS;                                         // this lane's column inside the block
  const int j0 = blockIdx.z * COLS, j = j0 + jc;                   // ... and of S
  const bool on = j < E;
  // 16-byte accesses when every piece is whole and aligned (the work rows are: their width is a multiple of 4)
  const bool vec = (D & 3) == 0 && (E & 3) == 0 && COLS >= 4 && DP >= 4;
  float S[DPT];
#pragma unroll
  for (int r = 0; r < DPT; ++r) {
    const int d = s * DPT + r;
    S[r] = (on && d < D && first_pos > 0) ? st[(int64_t)d * E + j] : 0.f;
  }
  float4 pkq[NV], pvo[NO];
  // the pieces of stage c0 into registers: all loads of a stage are in flight together
  auto fetch = [&](int64_t c0) {
    const int m = (int)(n - c0 < kStage ? n - c0 : kStage);
#pragma unroll
    for (int u = 0; u < NV; ++u) {
      const int f = tid + 64 * u, tok = f / (2 * DP / 4), within = f % (2 * DP / 4), which = within / (DP / 4), d = 4 * (within % (DP / 4));
      pkq[u] = (tok < m && d < D) ? *reinterpret_cast<const float4*>(a.work + (t0 + c0 + tok) * a.wld + (which ? 0 : G * D) + gk * D + d)
                                  : float4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int u = 0; u < NO; ++u) {
      const int f = tid + 64 * u, tok = f / (COLS / 4 > 0 ? COLS / 4 : 1), c = 4 * (f % (COLS / 4 > 0 ? COLS / 4 : 1));
      pvo[u] = (tok < m && j0 + c < E) ? *reinterpret_cast<const float4*>(a.work + (t0 + c0 + tok) * a.wld + 2 * G * D + h * E + j0 + c)
                                       : float4{0.f, 0.f, 0.f, 0.f};
    }
  };
  if (vec) fetch(0);
  for (int64_t c0 = 0; c0 < n; c0 += kStage) {
    const int m = (int)(n - c0 < kStage ? n - c0 : kStage);
    __syncthreads();
    if (vec) {
#pragma unroll
      for (int u = 0; u < NV; ++u) {
        const int f = tid + 64 * u, tok = f / (2 * DP / 4), within = f % (2 * DP / 4), which = within / (DP / 4), d = 4 * (within % (DP / 4));
        if (tok < kStage)
          *reinterpret_cast<float4*>(kq_l + tok * KQ + (which ? DS * SL : 0) + (d / DPT) * SL + d % DPT) = pkq[u];   // k first, then q
      }
#pragma unroll
      for (int u = 0; u < NO; ++u) {
        const int f = tid + 64 * u;
        if (f < kStage * COLS / 4) *reinterpret_cast<float4*>(vo_l + 4 * f) = pvo[u];
      }
    } else {
      for (int i = tid; i < m * 2 * DP; i += 64) {
        const int tok = i / (2 * DP), r = i % (2 * DP), d = r % DP;
        const float* wrow = a.work + (t0 + c0 + tok) * a.wld;
        const float x = d < D ? wrow[(r < DP ? G * D : 0) + gk * D + d] : 0.f;
        kq_l[tok * KQ + (r < DP ? 0 : DS * SL) + (d / DPT) * SL + d % DPT] = x;
      }
      for (int i = tid; i < m * COLS; i += 64) {
        const int tok = i / COLS, c = i % COLS;
        vo_l[i] = j0 + c < E ? a.work[(t0 + c0 + tok) * a.wld + 2 * G * D + h * E + j0 + c] : 0.f;
      }
    }
    __syncthreads();
    if (vec && c0 + kStage < n) fetch(c0 + kStage);                // the next stage's loads fly while this one is walked
    {                                                              // k . q, g, beta per token: four lanes a token
      static_assert(kStage * 4 == 64, "four lanes per staged token");
      const int tok = tid >> 2, part = tid & 3;
      float acc = 0.f;
      if (tok < m)
        for (int d = part; d < DP; d += 4) {
          const int o = (d / DPT) * SL + d % DPT;
          acc += kq_l[tok * KQ + o] * kq_l[tok * KQ + DS * SL + o];
        }
      acc = quad_sum<4>(acc);
      if (part == 0 && tok < m) {
        const float* gb = a.work + (t0 + c0 + tok) * a.wld + C;
        sc_l[tok * 4 + 0] = acc;
        sc_l[tok * 4 + 1] = gb[h];
        sc_l[tok * 4 + 2] = gb[H + h];
      }
    }
    __syncthreads();
#pragma unroll 2
    for (int tok = 0; tok < m; ++tok) {
      const float v = vo_l[tok * COLS + jc];
      const float4* kk4 = reinterpret_cast<const float4*>(kq_l + tok * KQ + s * SL);
      const float4* qq4 = reinterpret_cast<const float4*>(kq_l + tok * KQ + DS * SL + s * SL);
      float kk[DPT];
      float dk0 = 0.f, dq0 = 0.f, dk1 = 0.f, dq1 = 0.f;
#pragma unroll
      for (int r = 0; r < DPT; r += 4) {
        const float4 kv = kk4[r >> 2], qv = qq4[r >> 2];
        kk[r] = kv.x; kk[r + 1] = kv.y; kk[r + 2] = kv.z; kk[r + 3] = kv.w;
        dk0 += S[r] * kv.x;
        dq0 += S[r] * qv.x;
        dk1 += S[r + 1] * kv.y;
        dq1 += S[r + 1] * qv.y;
        dk0 += S[r + 2] * kv.z;
        dq0 += S[r + 2] * qv.z;
        dk1 += S[r + 3] * kv.w;
        dq1 += S[r + 3] * qv.w;
      }
      const float dk = quad_sum<DS>(dk0 + dk1), dq = quad_sum<DS>(dq0 + dq1);
      const float kq = sc_l[tok * 4 + 0], g = sc_l[tok * 4 + 1], beta = sc_l[tok * 4 + 2];
      const float u = beta * (v - g * dk);
#pragma unroll
      for (int r = 0; r < DPT; ++r) S[r] = g * S[r] + kk[r] * u;
      if (s == 0) vo_l[tok * COLS + jc] = g * dq + u * kq;         // (only this lane group reads or writes the element)
    }
    __syncthreads();
    if (vec) {
      for (int f = tid; f < m * COLS / 4; f += 64) {
        const int tok = f / (COLS / 4 > 0 ? COLS / 4 : 1), c = 4 * (f % (COLS / 4 > 0 ? COLS / 4 : 1));
        if (j0 + c < E)
          *reinterpret_cast<float4*>(a.work + (t0 + c0 + tok) * a.wld + 2 * G * D + h * E + j0 + c) = *reinterpret_cast<const float4*>(vo_l + 4 * f);
      }
    } else {
      for (int i = tid; i < m * COLS; i += 64) {
        const int tok = i / COLS, c = i % COLS;
        if (j0 + c < E) a.work[(t0 + c0 + tok) * a.wld + 2 * G * D + h * E + j0 + c] = vo_l[i];
      }
    }
  }
  if (on) {
#pragma unroll
    for (int r = 0; r < DPT; ++r) {
      const int d = s * DPT + r;
      if (d < D) st[(int64_t)d * E + j] = S[r];
    }
  }
}

// ---------------------------------------------------------------------------------- one token per request: everything at once
// A decode batch: a workgroup per (request, head) with all columns of S (DS lanes each) does the convolutions of its q / k head
// and of its value head, the unit norms, the gates, the step of the recurrence and the output norm and gate: one launch in
// place of three, and no work rows.  The same arithmetic as the kernels above (the unit norms multiply in at the use).
template <typename T, int DPT, int DS>
__global__ void __launch_bounds__(1024) delta_decode_kernel(DeltaArgs a) {
  extern __shared__ float lds[];          // k [DP] | q [DP] | scalars
  __shared__ float red[16];
  constexpr int DP = DPT * DS;
  const int b = blockIdx.x, h = blockIdx.y;
  const int D = a.D, E = a.E, G = a.G, H = a.H, taps = a.taps;
  const int gk = h / (H / G);
  const int64_t pos = a.seq_lens[b] - 1;
  if (pos < 0) return;
  const bool fresh = pos == 0;
  const int tid = threadIdx.x, s = tid % DS, j = tid / DS;
  const bool on = j < E;
  const int C = 2 * G * D + H * E;
  const int64_t slot = a.state_indices[b];
  const T* p = (const T*)a.p + (int64_t)b * a.ld;
  const float* cs = a.conv_state + slot * a.conv_ld;
  float* sc = lds + 2 * DP;
  auto conv = [&](const T* cw, int64_t col, int ch) -> float {      // cw: the channel's taps; ch: its place in the state
    float y = Elem<T>::to_f(cw[taps - 1]) * Elem<T>::to_f(p[col]);
    if (!fresh)
      for (int i = 1; i < taps; ++i) y += Elem<T>::to_f(cw[taps - 1 - i]) * cs[(int64_t)(taps - 1 - i) * C + ch];
    return silu_f(y);
  };
  for (int i = tid; i < 2 * DP; i += blockDim.x) {
    const bool is_q = i >= DP;
    const int d = is_q ? i - DP : i;
    float y = 0.f;
    if (d < D)
      y = is_q ? conv((const T*)a.conv_q + (int64_t)(gk * D + d) * taps, a.q_off + gk * D + d, gk * D + d)
               : conv((const T*)a.conv_k + (int64_t)(gk * D + d) * taps, a.k_off + gk * D + d, G * D + gk * D + d);
    lds[i] = y;
  }
  __syncthreads();
  if (tid < 64) {
    float sk = 0.f, sq = 0.f, kq = 0.f;
    for (int d = tid; d < DP; d += 64) {
      const float kv = lds[d], qv = lds[DP + d];
      sk += kv * kv;
      sq += qv * qv;
      kq += kv * qv;
    }
    sk = wave_sum(sk);
    sq = wave_sum(sq);
    kq = wave_sum(kq);
    if (tid == 0) {
      const float ik = 1.0f / sqrtf(sk + 1e-6f), iq = rsqrtf((float)D) / sqrtf(sq + 1e-6f);
      sc[0] = ik;
      sc[1] = iq;
      sc[2] = kq * ik * iq;
    }
  }
  __syncthreads();
  const float ik = sc[0], iq = sc[1], kq = sc[2];
  const float g = expf(-expf(a.a_log[h]) * softplus_f(Elem<T>::to_f(p[a.a_off + h]) + a.dt_bias[h]));
  const float beta = sigmoid_f(Elem<T>::to_f(p[a.b_off + h]));
  const float v = on ? conv((const T*)a.conv_v + (int64_t)(h * E + j) * taps, a.v_off + h * E + j, 2 * G * D + h * E + j) : 0.f;
  float* st = a.state + slot * a.state_ld + (int64_t)h * D * E;
  const float* kk = lds + s * DPT;
  const float* qq = kk + DP;
  float S[DPT];
  float dk = 0.f, dq = 0.f;
#pragma unroll
  for (int r = 0; r < DPT; ++r) {
    const int d = s * DPT + r;
    S[r] = (on && d < D && !fresh) ? st[(int64_t)d * E + j] : 0.f;
    dk += S[r] * (kk[r] * ik);
    dq += S[r] * (qq[r] * iq);
  }
  dk = quad_sum<DS>(dk);
  dq = quad_sum<DS>(dq);
  const float u = beta * (v - g * dk);
  const float o = g * dq + u * kq;
  if (on) {
#pragma unroll
    for (int r = 0; r < DPT; ++r) {
      const int d = s * DPT + r;
      if (d < D) st[(int64_t)d * E + j] = g * S[r] + (kk[r] * ik) * u;
    }
  }
  const float sq_o = block_sum((on && s == 0) ? o * o : 0.f, red);
  if (on && s == 0) {
    const float inv = 1.0f / sqrtf(sq_o / (float)E + a.eps);
    const float gate = Elem<T>::to_f(p[a.gate_off + h * E + j]);
    ((T*)a.out)[(int64_t)b * a.out_ld + h * E + j] = Elem<T>::from_f(o * inv * Elem<T>::to_f(((const T*)a.norm_w)[j]) * silu_f(gate));
  }
}

// The same with S in 16-byte pieces: a workgroup per (key head, request) with a team of four waves per value head (in turn, where there
// are more heads than teams: a piece of the next one is fetched as one of this is stored), so the convolution's channels belong to
// one workgroup, which moves their inputs on itself: ONE launch.  (gridDim.z > 1: the heads of a key head over several.)  A thread of a team has four columns and every 1024 / E-th row
// of S, all of its pieces in flight from the start; the two dot products are summed over lanes and the team's waves.  Bound by HBM, the
// state read and written once: 32 requests, 32 heads of 128 x 128 (134 MB): a column of S by four lanes of four bytes each 57.7 -> 32.3
// us; 3 requests, 32 heads of 64 x 64: 10.6 (two launches) -> 9.8.  With the loads of the convolutions and of the gates in front of the state's (they came one
// behind the other when the state had arrived): 32 heads of 128 x 128, 32 requests, whole call 31.6 -> 28.5, 64 requests 77.7 -> 68.9.
template <typename T, int NIT, int EARLY>
__global__ void __launch_bounds__(NIT > 4 ? 512 : 1024) delta_step_kernel(DeltaArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];       // q [D] | k [D] | v, later o [per E] | sums of every team [4][2][E] | scalars
  const int g = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63, team = tid >> 8, tt = tid & 255, teams = blockDim.x >> 8;
  const int64_t pos = a.seq_lens[b] - 1;
  if (pos < 0) return;
  const bool fresh = pos == 0;
  const int D = a.D, E = a.E, G = a.G, H = a.H, taps = a.taps, per = H / G, C = 2 * G * D + H * E;
  const int quads = E / 4, rows = 256 / quads, n0 = tt / quads, e = tt % quads * 4;
  const int64_t slot = a.state_indices[b];
  const T* p = (const T*)a.p + (int64_t)b * a.ld;
  float* q_l = lds;
  float* k_l = lds + D;
  float* v_l = lds + 2 * D;
  float* sums = v_l + per * E + team * 8 * E;
  float* sc = v_l + per * E + teams * 8 * E;
  float4 S[NIT];
  auto piece = [&](int hh, int n) {
    return !fresh && hh < per && n < D ? *reinterpret_cast<const float4*>(a.state + slot * a.state_ld + ((int64_t)(g * per + hh) * D + n) * E + e) : float4{0.f, 0.f, 0.f, 0.f};
  };
  // Memory answers in order: what the convolutions are made of is asked for in front of the state, and with it what the team's first head needs
  // behind the sums; their arithmetic goes on while the state is on its way, and nothing is a round trip of its own.  Up to EARLY
  // taps, the workgroup's first two channels a thread; others (EARLY 0: more than four taps) one by one.
  const int channels = 2 * D + per * E;
  struct Channel {
    const T *p, *cw;
    int ch;                                                       // its place in the kept inputs
  };
  auto channel = [&](int i) {
    const bool is_v = i >= 2 * D;
    const int d = is_v ? g * per * E + i - 2 * D : g * D + (i < D ? i : i - D);                              // channel within q, k or v
    return Channel{p + (is_v ? a.v_off : (i < D ? a.q_off : a.k_off)) + d, (const T*)(is_v ? a.conv_v : (i < D ? a.conv_q : a.conv_k)) + (int64_t)d * taps,
                   is_v ? 2 * G * D + d : (i < D ? d : G * D + d)};
  };
  auto mine = [&](int i) { return i < channels && (i < 2 * D || gridDim.z == 1 || ((i - 2 * D) / E / teams) % gridDim.z == blockIdx.z); };      // (or a head of another workgroup)
  float* cs = a.conv_state + slot * a.conv_ld;
  struct Inputs {
    T cur, w[EARLY + 1];
    float x[EARLY + 1];                                           // (of k tokens back)
  } in[2];
  if constexpr (EARLY > 0)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const Channel c = channel(min(tid + (int)blockDim.x * u, channels - 1));
      in[u].cur = *c.p;
#pragma unroll
      for (int k = 0; k < EARLY; ++k) {
        in[u].w[k] = c.cw[max(taps - 1 - k, 0)];
        in[u].x[k] = k > 0 && k < taps && !fresh ? cs[(int64_t)(taps - 1 - k) * C + c.ch] : 0.f;
      }
    }
  float gate_log, gate_bias, weight[4];
  T gate_a, gate_b, gate[4];
  auto fetch_gates = [&](int hh) {
    const int h = g * per + (hh < per ? hh : per - 1);
    gate_log = a.a_log[h], gate_bias = a.dt_bias[h];
    gate_a = p[a.a_off + h], gate_b = p[a.b_off + h];
    if (n0 == 0)
#pragma unroll
      for (int c = 0; c < 4; ++c) gate[c] = p[a.gate_off + h * E + e + c];
  };
  fetch_gates((int)blockIdx.z * teams + team);
  if (n0 == 0)
#pragma unroll
    for (int c = 0; c < 4; ++c) weight[c] = Elem<T>::to_f(((const T*)a.norm_w)[e + c]);
#pragma unroll
  for (int i = 0; i < NIT; ++i) S[i] = piece((int)blockIdx.z * teams + team, n0 + i * rows);
  // state entry s is the input s - (taps - 1) tokens back; every entry moves one place down and the token comes in last (where several
  // workgroups read the old inputs of q and k, in a launch of its own)
  if constexpr (EARLY > 0)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = tid + (int)blockDim.x * u;
      if (!mine(i)) continue;
      const float cur = Elem<T>::to_f(in[u].cur);
      float y = Elem<T>::to_f(in[u].w[0]) * cur;
#pragma unroll
      for (int k = 1; k < EARLY; ++k)
        if (k < taps && !fresh) y += Elem<T>::to_f(in[u].w[k]) * in[u].x[k];
      lds[i] = silu_f(y);
      if (gridDim.z > 1) continue;
      const int ch = channel(i).ch;
#pragma unroll
      for (int k = 1; k < EARLY - 1; ++k)
        if (k < taps - 1) cs[(int64_t)(taps - 2 - k) * C + ch] = in[u].x[k];
      if (taps > 1) cs[(int64_t)(taps - 2) * C + ch] = cur;
    }
  for (int i = EARLY > 0 ? tid + 2 * (int)blockDim.x : tid; i < channels; i += blockDim.x) {
    if (!mine(i)) continue;
    const Channel c = channel(i);
    const float cur = Elem<T>::to_f(*c.p);
    float y = Elem<T>::to_f(c.cw[taps - 1]) * cur;
    for (int k = 1; k < taps; ++k) {
      const int s = taps - 1 - k;
      const float x = fresh ? 0.f : cs[(int64_t)s * C + c.ch];
      if (!fresh) y += Elem<T>::to_f(c.cw[s]) * x;
    }
    lds[i] = silu_f(y);
    if (gridDim.z > 1) continue;
    for (int s = 1; s < taps - 1; ++s) cs[(int64_t)(s - 1) * C + c.ch] = fresh ? 0.f : cs[(int64_t)s * C + c.ch];
    if (taps > 1) cs[(int64_t)(taps - 2) * C + c.ch] = cur;
  }
  __syncthreads();
  if (tid < 64) {
    float sk = 0.f, sq = 0.f, kq = 0.f;
    for (int d = lane; d < D; d += 64) {
      sk += k_l[d] * k_l[d];
      sq += q_l[d] * q_l[d];
      kq += k_l[d] * q_l[d];
    }
    sk = wave_sum(sk);
    sq = wave_sum(sq);
    kq = wave_sum(kq);
    if (lane == 0) {
      const float ik = 1.0f / sqrtf(sk + 1e-6f), iq = rsqrtf((float)D) / sqrtf(sq + 1e-6f);
      sc[0] = ik;
      sc[1] = iq;
      sc[2] = kq * ik * iq;
    }
  }
  __syncthreads();
  const float ik = sc[0], iq = sc[1], kq = sc[2];
  for (int h0 = blockIdx.z * teams; h0 < per; h0 += teams * gridDim.z) {       // (every team goes round as often: there are barriers inside)
    const int hh = h0 + team, h = g * per + (hh < per ? hh : per - 1);
    const bool on = hh < per;
    float4 dk = {0.f, 0.f, 0.f, 0.f}, dq = {0.f, 0.f, 0.f, 0.f};
    if (on)
#pragma unroll
      for (int i = 0; i < NIT; ++i) {
        const int n = n0 + i * rows;
        if (n < D) {
          const float kv = k_l[n] * ik, qv = q_l[n] * iq;
          dk = float4{dk.x + S[i].x * kv, dk.y + S[i].y * kv, dk.z + S[i].z * kv, dk.w + S[i].w * kv};
          dq = float4{dq.x + S[i].x * qv, dq.y + S[i].y * qv, dq.z + S[i].z * qv, dq.w + S[i].w * qv};
        }
      }
    for (int o = quads; o < 64; o <<= 1) {
      dk.x += __shfl_xor(dk.x, o, 64); dk.y += __shfl_xor(dk.y, o, 64); dk.z += __shfl_xor(dk.z, o, 64); dk.w += __shfl_xor(dk.w, o, 64);
      dq.x += __shfl_xor(dq.x, o, 64); dq.y += __shfl_xor(dq.y, o, 64); dq.z += __shfl_xor(dq.z, o, 64); dq.w += __shfl_xor(dq.w, o, 64);
    }
    if (lane < quads) {
      *reinterpret_cast<float4*>(sums + (tt >> 6) * 2 * E + e) = dk;
      *reinterpret_cast<float4*>(sums + (tt >> 6) * 2 * E + E + e) = dq;
    }
    __syncthreads();
    const float gt = expf(-expf(gate_log) * softplus_f(Elem<T>::to_f(gate_a) + gate_bias)), beta = sigmoid_f(Elem<T>::to_f(gate_b));
    float u[4], o4[4], sq_o = 0.f;
    const float* vh = v_l + (on ? hh : 0) * E + e;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float* sk = sums + e + c;
      const float dkc = (sk[0] + sk[2 * E]) + (sk[4 * E] + sk[6 * E]), dqc = (sk[E] + sk[3 * E]) + (sk[5 * E] + sk[7 * E]);
      u[c] = beta * (vh[c] - gt * dkc);
      o4[c] = gt * dqc + u[c] * kq;
      sq_o += o4[c] * o4[c];
    }
    if (on) {
      float* st = a.state + slot * a.state_ld + (int64_t)h * D * E;
#pragma unroll
      for (int i = 0; i < NIT; ++i) {
        const int n = n0 + i * rows;
        if (n < D) {
          const float kv = k_l[n] * ik;
          *reinterpret_cast<float4*>(st + n * E + e) = float4{gt * S[i].x + kv * u[0], gt * S[i].y + kv * u[1], gt * S[i].z + kv * u[2], gt * S[i].w + kv * u[3]};
        }
        S[i] = piece(hh + teams * (int)gridDim.z, n);                // (the team's next head)
      }
    }
    for (int o = 1; o < quads; o <<= 1) sq_o += __shfl_xor(sq_o, o, 64);       // (a row of S is `quads` neighbouring lanes, all columns)
    if (on && n0 == 0) {
      const float inv = 1.0f / sqrtf(sq_o / (float)E + a.eps);
      T* out = (T*)a.out + (int64_t)b * a.out_ld + h * E + e;
#pragma unroll
      for (int c = 0; c < 4; ++c) out[c] = Elem<T>::from_f(o4[c] * inv * weight[c] * silu_f(Elem<T>::to_f(gate[c])));
    }
    if (h0 + teams * (int)gridDim.z < per) fetch_gates(hh + teams * (int)gridDim.z);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------- unit RMS, weight, gate
template <typename T>
__global__ void __launch_bounds__(256) delta_post_kernel(DeltaArgs a) {
  // a workgroup per token; its waves take the token's heads in turn
  const int lane = threadIdx.x & 63;
  const int64_t t = blockIdx.x;
  const int E = a.E;
  for (int h = threadIdx.x >> 6; h < a.H; h += 4) {
  const float* o = a.work + t * a.wld + a.o_off + h * E;
  float sq = 0.f;
  for (int e = lane; e < E; e += 64) sq += o[e] * o[e];
  sq = wave_sum(sq);
  const float inv = 1.0f / sqrtf(sq / (float)E + a.eps);
  const T* gate = (const T*)a.p + t * a.ld + a.gate_off + (int64_t)h * E;
  const T* nw = (const T*)a.norm_w;
  T* out = (T*)a.out + t * a.out_ld + (int64_t)h * E;
  for (int e = lane; e < E; e += 64)
    out[e] = Elem<T>::from_f(o[e] * inv * Elem<T>::to_f(nw[e]) * silu_f(Elem<T>::to_f(gate[e])));
  }
}

// ---------------------------------------------------------------------------------- prompt batches: 32 tokens at a time
// With b_t the running sum of the log decays inside a chunk of 32 tokens and S the state in front of it:
//     u_t = beta_t (v_t - e^(b_t) S^T k_t - sum_(s < t) e^(b_t - b_s) (k_t . k_s) u_s)
//     o_t = e^(b_t) S^T q_t + sum_(s <= t) e^(b_t - b_s) (q_t . k_s) u_s
//     S  <- e^(b_last) S + sum_s k_s (e^(b_last - b_s) u_s)^T
// The sums over s < t are a unit lower triangular matrix A, so U = (I + A)^-1 diag(beta) (V - diag(e^b) K S); everything in
// front of V and S is independent of the chunks before it and is computed for all chunks at once.  Every exponent is at most 0, b is
// summed, and its differences are taken, in 64 bits.  All products are of fp32 operands (v_mfma_f32_16x16x4_f32), those with S of keys of
// more than 64 on the bf16 matrix cores, three pieces a value (see rec_mma; state behind 4 requests of 1900 tokens 3.37e-8 from the 64-bit
// one, in either form), sums fp32.
// Bound: token by token a step is a chain of two dot products, a lane sum and an update (0.8 us; 7262 tokens of 4 requests, 32 heads of
// 128 x 128: 1861 us + 317 of preparation).  In chunks with all products in fp32, a wave all rows of 16 columns: a chain of 216 products of
// 32 cycles a chunk, one wave a SIMD at 4 requests: 385 us.  In pieces, two waves a column block with half the rows each: 345, two waves a
// SIMD, each with 72 products of 16 cycles, 16 or 20 of 32, 450 vector instructions and 50 LDS reads of 1 KB a chunk, which cover each other
// in part (10 k cycles a chunk against 7 k one behind the other).  Operands 60.
// Elements of the operands of one (chunk, key head), counted in fp32: keys of more than 64: K, Q and K^T in three planes of bf16 each,
// left-hand operands of 16 x 16 x 32 products in the order in which they are held, [tile][lane][8] (see rec_split8; tiles of K and Q: 16
// tokens x 32 rows of S, of K^T: 16 rows x the tokens); else in fp32, of 16 x 16 x 16 products, [tile][lane][4], lane (r16, kq) element s =
// row r16, column 4 kq + s of the tile; a flag in a piece of 4.  Of one (chunk, head), fp32, [tile][lane][4]: tiles 00, 10, 11 of
// (I + A)^-1 diag(beta) and of the weighted Q K^T, then e^(b_t) | e^(b_last - b_t) | decay | beta.
constexpr int kDeltaSmall = 64;
__host__ __device__ constexpr int64_t delta_frag_elems(int np) { return (np <= kDeltaSmall ? 3 : 4.5) * kRecChunk * np + 4; }
constexpr int kDeltaHead = 6 * 256 + 4 * kRecChunk;

// A workgroup per (chunk, key head): convolution, silu and unit norm of its q and k (a channel per thread), K K^T and Q K^T, then
// half a wave per head of the group: gates; weights, A and its inverse in blocks of 16 by whole waves.  Bound by what it lays down where the chip is
// full of it (1848 workgroups, 185 MB) and by the chain of one workgroup where it is not: 42 k cycles, now 27 k (search 2.9, rows 3.5,
// convolution 4.6, norms 2.1, pieces 4, products 2.7, gates 3.3, weights 1.3 (7.6 a column at a time, its exponentials one behind the other and
// stores of 4 bytes), inverse 2.4 (7.5 as one chain of 32 rows)).  32 heads of 128 x 128 over 8, whole call: 1 request of 100 rows 44 -> 37.5
// us, 5 of 155 81 -> 75, 4 of 1900 426 -> 414.
template <typename T, int NP>
__global__ void __launch_bounds__(256, 4) delta_chunk_operands_kernel(DeltaArgs a) {
  constexpr int L = kRecChunk, CS = NP + 4, PS = L + 4, AL = 16 * 16 + 16 * 36, LATER = 8 * AL + 2 * L * PS;
  // K [32][CS] | Q; later A, one per half wave (rows of 16, from row 16 on of 36: it is strictly lower triangular) | K K^T | Q K^T.  39 KB and
  // 128 registers: four workgroups a CU (45 KB and three before: 1824 workgroups took three rounds of 20 us)
  __shared__ __attribute__((aligned(16))) float kq_l[2 * L * CS > LATER ? 2 * L * CS : LATER];
  float *const kk_l = kq_l + 8 * AL, *const qk_l = kk_l + L * PS;
  __shared__ __attribute__((aligned(16))) double cum_l[8 * L];
  __shared__ __attribute__((aligned(16))) float beta_l[8 * L];
  __shared__ int bad_l;
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, kq = lane >> 4, g = blockIdx.y;
  RecChunk at;
  if (!rec_find_chunk(a.q_len, a.seq_lens, a.q_start, (int)a.batch, blockIdx.x, at) || at.first_pos < 0) return;
  const int64_t l0 = at.c * L, t0 = at.q_start + l0;
  const int cnt = (int)(at.n - l0 < L ? at.n - l0 : L);
  const int D = a.D, taps = a.taps, C = 2 * a.G * D + a.H * a.E, per = a.H / a.G;
  float* frag = a.frags + ((int64_t)blockIdx.x * a.G + g) * delta_frag_elems(NP);
  const float* kept = l0 == 0 && at.first_pos > 0 && taps > 1 ? a.conv_state + a.state_indices[at.b] * a.conv_ld : nullptr;
  bool bad = false;
  // up to eight heads at a time, half wave `half` of wave w has w + 4 half: its decays and the diagonal blocks of its inverse; the weights
  // and the rest of the inverse of a wave's heads by the whole wave, one head after the other (each for its own: with four heads half of the
  // chip's waves have none, 7.3 us of a workgroup's 30).  What the first heads' gates are made of is fetched here.
  const int half = lane >> 5, ln = tid & 31;
  T gate_a, gate_b;
  float gate_log, gate_bias;
  auto fetch_gates = [&](int h0) {                               // (of rows and heads that there are; raw, so that nothing waits for them here)
    const int h = g * per + min(h0 + w + 4 * half, per - 1);
    const T* pr = (const T*)a.p + (t0 + min(ln, cnt - 1)) * a.ld;
    gate_a = pr[a.a_off + h];
    gate_b = pr[a.b_off + h];
    gate_log = a.a_log[h];
    gate_bias = a.dt_bias[h];
  };
  fetch_gates(blockIdx.z * 8);
  if (tid == 0) bad_l = 0;
  for (int ch = tid; ch < 2 * NP; ch += 256) {
    const bool is_q = ch >= NP;
    const int d = is_q ? ch - NP : ch;
    float* dst = kq_l + (is_q ? L * CS : 0) + d;
    if (d < D) {
      const int cc = (is_q ? 0 : a.G * D) + g * D + d;                                      // channel in the state's order (q | k | v)
      const T* p = (const T*)a.p + t0 * a.ld + (is_q ? a.q_off : a.k_off) + g * D + d;
      const T* cw = (const T*)(is_q ? a.conv_q : a.conv_k) + (int64_t)(g * D + d) * taps;
      float wt[kRecTaps], in[kRecTaps], x[L];
      rec_channel<T>(p, a.ld, cnt, cw, taps, l0 > 0, kept != nullptr ? kept + cc : nullptr, C, wt, in, x);
      rec_conv_silu(wt, in, x, 0.f, taps, cnt, dst, CS);
    } else {
      for (int t = 0; t < L; ++t) dst[t * CS] = 0.f;
    }
  }
  __syncthreads();
  // unit norms: four lanes a row, a quarter of it each (in turns that keep the sixteen lanes of an access in banks of their own)
  {
    const int row = tid >> 2, part = tid & 3;                    // rows 0 .. 31: k, 32 .. 63: q
    float* x = kq_l + (row >= L ? L * CS : 0) + (row % L) * CS + part * (NP / 4);
    constexpr int Q = NP / 16;                                   // 16-byte pieces of a quarter
    f32x4 v[Q];
    float sq = 0.f;
#pragma unroll
    for (int i = 0; i < Q; ++i) v[i] = *reinterpret_cast<const f32x4*>(x + 4 * ((i + Q / 2 * (part >> 1)) % Q));
#pragma unroll
    for (int i = 0; i < Q; ++i) sq += (v[i][0] * v[i][0] + v[i][1] * v[i][1]) + (v[i][2] * v[i][2] + v[i][3] * v[i][3]);
    sq = quad_sum<4>(sq);
    const float inv = (row >= L ? rsqrtf((float)D) : 1.0f) / sqrtf(sq + 1e-6f);
#pragma unroll
    for (int i = 0; i < Q; ++i) {
      v[i] *= inv;
      *reinterpret_cast<f32x4*>(x + 4 * ((i + Q / 2 * (part >> 1)) % Q)) = v[i];
      bad |= !rec_finite(v[i][0]) || !rec_finite(v[i][1]) || !rec_finite(v[i][2]) || !rec_finite(v[i][3]);
    }
    if (__any(bad) && lane == 0) bad_l = 1;
  }
  __syncthreads();
  // the operands in the order in which they are held
  const bool lays = blockIdx.z == 0;                             // (the workgroups of a group's heads all have the operands, one lays them down)
  if (lays && tid == 0) frag[delta_frag_elems(NP) - 4] = bad_l ? 1.f : 0.f;
  if constexpr (NP <= kDeltaSmall) {
    for (int i = lays ? tid : 2 * L * NP; i < 2 * L * NP / 4; i += 256) {              // K | Q: tile (row tile, column tile)
      const int half = i / (L * NP / 4), it = i % (L * NP / 4), tile = it >> 6, ln = it & 63, rt = tile / (NP / 16), ct = tile % (NP / 16);
      *reinterpret_cast<float4*>(frag + 4 * i) = *reinterpret_cast<const float4*>(kq_l + half * L * CS + (16 * rt + (ln & 15)) * CS + 16 * ct + 4 * (ln >> 4));
    }
    for (int i = lays ? tid : L * NP; i < L * NP / 4; i += 256) {                  // K^T: tile (row of S, tokens)
      const int tile = i >> 6, ln = i & 63, rt = tile >> 1, ct = tile & 1;
      const float* s = kq_l + (16 * ct + 4 * (ln >> 4)) * CS + 16 * rt + (ln & 15);
      *reinterpret_cast<float4*>(frag + 2 * L * NP + 4 * i) = float4{s[0], s[CS], s[2 * CS], s[3 * CS]};
    }
  } else {
    // pieces of three planes: K and Q, tiles (16 tokens, 32 rows of S), and K^T, tiles (16 rows of S, the tokens)
    for (int i = lays ? tid : L * NP; i < 3 * (L * NP / 8); i += 256) {
      const int part = i / (L * NP / 8), it = i % (L * NP / 8), tile = it >> 6, ln = it & 63, r = ln & 15, q4 = 4 * (ln >> 4);
      f32x4 x0, x1;
      if (part < 2) {
        const float* s = kq_l + part * L * CS + (16 * (tile / (NP / 32)) + r) * CS + 32 * (tile % (NP / 32)) + q4;
        x0 = *reinterpret_cast<const f32x4*>(s);
        x1 = *reinterpret_cast<const f32x4*>(s + 16);
      } else {
        const float* s = kq_l + q4 * CS + 16 * tile + r;
        x0 = f32x4{s[0], s[CS], s[2 * CS], s[3 * CS]};
        x1 = f32x4{s[16 * CS], s[17 * CS], s[18 * CS], s[19 * CS]};
      }
      // (unit vectors: what is larger is not a number or infinite)
      float z = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) z = fmaf(x1[q], 0.f, fmaf(x0[q], 0.f, z));
      Split3 s3;
      if (__any(z != 0.f)) s3 = rec_split8_any(x0, x1);
      else s3 = rec_split8(x0, x1);
      uint4* dst = reinterpret_cast<uint4*>(frag + part * (3 * L * NP / 2)) + it;
  #pragma unroll
      for (int p = 0; p < 3; ++p) dst[p * (L * NP / 8)] = s3.p[p].u;
    }
  }
  {
    const int i0 = (w >> 1) * 16, j0 = (w & 1) * 16;
    f32x4 kk = {}, qk = {};
#pragma unroll 4
    for (int k = 0; k < NP; k += 16) {
      const f32x4 ak = *reinterpret_cast<const f32x4*>(kq_l + (i0 + r16) * CS + k + 4 * kq);
      const f32x4 aq = *reinterpret_cast<const f32x4*>(kq_l + L * CS + (i0 + r16) * CS + k + 4 * kq);
      const f32x4 bv = *reinterpret_cast<const f32x4*>(kq_l + (j0 + r16) * CS + k + 4 * kq);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        kk = __builtin_amdgcn_mfma_f32_16x16x4f32(ak[s], bv[s], kk, 0, 0, 0);
        qk = __builtin_amdgcn_mfma_f32_16x16x4f32(aq[s], bv[s], qk, 0, 0, 0);
      }
    }
    __syncthreads();                                              // (K and Q have been read)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      kk_l[(i0 + 4 * kq + r) * PS + j0 + r16] = kk[r];
      qk_l[(i0 + 4 * kq + r) * PS + j0 + r16] = qk[r];
    }
  }
  __syncthreads();
  double* cum = cum_l + (2 * w + half) * L;
  for (int h0 = blockIdx.z * 8; h0 < per; h0 += 8 * gridDim.z) {
    if (h0 + w >= per) break;
    const int heads = h0 + w + 4 < per ? 2 : 1;                  // of this wave
    const bool mine = half < heads;
    const int h = g * per + h0 + w + (mine ? 4 * half : 0);      // (a half wave without a head of its own goes along with the other, and lays nothing down)
    const bool on = ln < cnt && mine;
    if (h0 != (int)blockIdx.z * 8) fetch_gates(h0);
    const float la = on ? -expf(gate_log) * softplus_f(Elem<T>::to_f(gate_a) + gate_bias) : 0.f;
    const float beta = on ? sigmoid_f(Elem<T>::to_f(gate_b)) : 0.f;
    double c = (double)la * 1.4426950408889634;
#pragma unroll
    for (int o = 1; o < L; o <<= 1) {
      const double v = __shfl_up(c, o, L);
      if (ln >= o) c += v;
    }
    const double last = __shfl(c, L - 1, L);
    cum[ln] = c;
    beta_l[(2 * w + half) * L + ln] = beta;
    float* hp = a.frags + (int64_t)gridDim.x * a.G * delta_frag_elems(NP) + ((int64_t)blockIdx.x * a.H + h) * kDeltaHead;
    const float eb = rec_exp2(c), wt = rec_exp2(last - c), dec = expf(la);
    const bool no = !rec_finite(eb) || !rec_finite(wt) || !rec_finite(dec) || !rec_finite(beta) || !rec_moderate_decay(la);
    const float flagged = rec_flagged(eb, no);
    if (mine) {
      hp[1536 + ln] = flagged;
      hp[1536 + L + ln] = wt;
      hp[1536 + 2 * L + ln] = dec;
      hp[1536 + 3 * L + ln] = beta;
    }
    __builtin_amdgcn_wave_barrier();
    // A and the weighted Q K^T, four columns of a row a lane, tiles 00, 10, 11
    for (int v = 0; v < heads; ++v) {
      const double* cv = cum_l + (2 * w + v) * L;
      float* av = kq_l + (2 * w + v) * AL;
      float* hv = a.frags + (int64_t)gridDim.x * a.G * delta_frag_elems(NP) + ((int64_t)blockIdx.x * a.H + g * per + h0 + w + 4 * v) * kDeltaHead;
#pragma unroll
      for (int tile = 0; tile < 3; ++tile) {
        const int row = (tile ? 16 : 0) + r16, col = (tile == 2 ? 16 : 0) + 4 * kq;
        const double ct = cv[row];
        const float bt = beta_l[(2 * w + v) * L + row];
        const f32x4 kk = *reinterpret_cast<const f32x4*>(kk_l + row * PS + col), qk = *reinterpret_cast<const f32x4*>(qk_l + row * PS + col);
        f32x4 am, qm;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const float x = rec_exp2(ct - cv[col + s]);
          am[s] = col + s < row ? bt * (x * kk[s]) : 0.f;
          qm[s] = col + s <= row ? x * qk[s] : 0.f;
        }
        *reinterpret_cast<f32x4*>(av + (tile ? 256 + r16 * 36 + col : r16 * 16 + col)) = am;
        *reinterpret_cast<f32x4*>(hv + 768 + 256 * tile + 4 * lane) = qm;
      }
    }
    __builtin_amdgcn_wave_barrier();
    // T = (I + A)^-1 in blocks of 16: the diagonal ones column by column, a lane each (four terms of a row at a time), into the place of A's,
    // then T10 = -T11 A10 T00, as its transpose, so that it leaves as it stands.  (All 32 rows column by column were a chain of 496 terms.)
    if (mine) {
      const int st = ln >> 4, c = ln & 15, ald = st ? 36 : 16;
      float* a_l = kq_l + (2 * w + half) * AL + (st ? 256 + 16 : 0);
      float x[16];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        float acc = t == c ? 1.f : 0.f;
#pragma unroll
        for (int s = 0; s < t; s += 4) {
          const float4 av = *reinterpret_cast<const float4*>(a_l + t * ald + s);
          acc -= av.x * x[s];
          if (s + 1 < t) acc -= av.y * x[s + 1];
          if (s + 2 < t) acc -= av.z * x[s + 2];
          if (s + 3 < t) acc -= av.w * x[s + 3];
        }
        x[t] = acc;
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t = 0; t < 16; ++t) a_l[t * ald + c] = x[t];
    }
    __builtin_amdgcn_wave_barrier();
    for (int v = 0; v < heads; ++v) {
      const float *tl = kq_l + (2 * w + v) * AL, *bv = beta_l + (2 * w + v) * L;
      float* hv = a.frags + (int64_t)gridDim.x * a.G * delta_frag_elems(NP) + ((int64_t)blockIdx.x * a.H + g * per + h0 + w + 4 * v) * kDeltaHead;
      const f32x4 t00 = *reinterpret_cast<const f32x4*>(tl + r16 * 16 + 4 * kq), a10 = *reinterpret_cast<const f32x4*>(tl + 256 + r16 * 36 + 4 * kq);
      const f32x4 t11 = *reinterpret_cast<const f32x4*>(tl + 256 + r16 * 36 + 16 + 4 * kq);
      const f32x4 b0 = *reinterpret_cast<const f32x4*>(bv + 4 * kq), b1 = *reinterpret_cast<const f32x4*>(bv + 16 + 4 * kq);
      f32x4 y = {}, z = {};
#pragma unroll
      for (int s = 0; s < 4; ++s) y = __builtin_amdgcn_mfma_f32_16x16x4f32(a10[s], tl[(4 * kq + s) * 16 + r16], y, 0, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; ++s) z = __builtin_amdgcn_mfma_f32_16x16x4f32(y[s], t11[s], z, 0, 0, 0);
      *reinterpret_cast<f32x4*>(hv + 4 * lane) = t00 * b0;
      *reinterpret_cast<f32x4*>(hv + 256 + 4 * lane) = -z * b0;
      *reinterpret_cast<f32x4*>(hv + 512 + 4 * lane) = t11 * b1;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// The chunks of a request in turn, a workgroup of eight waves per (request, head, 16 CB columns of S), two or four waves per 16 columns.  A wave
// has its part of the rows of S in accumulators: lane (r16, kq) holds rows 16 t + 4 kq + r of column r16, two tiles of which are the
// right-hand operand of a product over 32 rows (split on the way), so S goes from one chunk's sum into the next one's product without leaving
// its registers.  The parts of K S go to the other waves of the columns through LDS and all make U; of Q S, v and the results a wave finishes
// 16 of the tokens.
// Four waves per 16 columns halve what a wave does for a chunk and leave U to be made twice as often: for launches that leave CUs without
// work at 64 columns a workgroup.  Their chunk was 4.2 us of 10 k cycles, now 7.8 k, about 500 vector instructions and 56 products of either
// wave of a SIMD; half the work a wave left the waits for the operands, so everything is fetched a whole chunk ahead there (3.5 -> 3.2 us; the form
// of two waves is 5 % slower so).  32 heads of 128 x 128 over 8, whole call: 1 request of 5083 rows 741 -> 583 us, of 1000 168 -> 139.
// Of a chunk's 10.3 k cycles (4 requests of 1900 rows) the products with S take 4.6 k and what is behind them 5.7 k; a SIMD's two waves take turns
// rather than overlap.  K S and Q S as four sums side by side, the state's update in front of the results' products, one sum for all pieces, the
// silus of a lane's tokens side by side, and one of the two waves through its convolution while the other multiplies: whole call 417 -> 406 us,
// 1 request of 5000 rows 566 -> 548.  No gain: the higher priority for the waves with more products (424), everything a chunk ahead (422).
template <typename T, int NP, int CB>
__global__ void __launch_bounds__(512, 2) delta_chunk_walk_kernel(DeltaArgs a, int64_t max_chunks) {
  constexpr int PARTS = 8 / CB;                                 // waves that share 16 columns
  constexpr int L = kRecChunk, NT = NP / 16, HT = NT / PARTS, HALO = kRecHalo;  // HT: 16-row tiles of S a wave
  constexpr int EX = PARTS == 2 ? 3 : 2;
  constexpr bool AHEAD = PARTS > 2;                             // everything is fetched a whole chunk ahead, not half of one
  static_assert(HT % 2 == 0, "two tiles are an operand");
  constexpr int PB = L * NP * 2, ALL = 3 * PB / 16, PIECES = (ALL + 511) / 512;  // bytes of a plane; 16-byte pieces of three, a thread's
  using Tile = RowTile<T, 16>;
  static_assert(Tile::kElems * sizeof(T) <= EX * 1024 && 16 * kOutStride * 4 <= EX * 1024, "a wave's part of ex_l");
  __shared__ __attribute__((aligned(16))) uint8_t k_l[3 * PB], q_l[3 * PB], kt_l[3 * PB];    // K, Q and K^T of the chunk, as laid down
  __shared__ __attribute__((aligned(16))) float head_l[kDeltaHead];             // the head's weights
  // by turns half sums for a wave from the other one of its columns, its raw inputs, its results on their way out (token by token: v)
  __shared__ __attribute__((aligned(16))) uint8_t ex_l[8][EX][1024];
  __shared__ __attribute__((aligned(16))) uint8_t sum_l[PARTS == 2 ? 1 : 8][4][PARTS == 2 ? 16 : 1024];     // four waves: their parts of K S and Q S
  __shared__ __attribute__((aligned(16))) uint8_t v_l[CB][2][1024];             // v of the chunk: [columns][token tile][lane][16]
  __shared__ int serial_l[2];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, kq = lane >> 4;
  // of four waves the first two make v, the others finish the results, either of 16 tokens; of two each does both
  const int cw = w % CB, part = w / CB, half = part & 1;
  const bool makes_v = PARTS == 2 || part < 2, ends = PARTS == 2 || part >= 2;
  const bool conv_first = PARTS == 2 && part == 1;              // (the other wave of the SIMD goes through its products meanwhile)
  // workgroups of one (request, key head) read the same operands: they go to one XCD (workgroup ids go round the 8 XCDs)
  const int H = a.H, G = a.G, D = a.D, E = a.E, taps = a.taps, per = H / G;
  const int eblocks = (E + 16 * CB - 1) / (16 * CB), members = per * eblocks;
  const RecPlace at = rec_place((int)a.batch * G, members);
  if (at.unit < 0) return;
  const int member = at.member, g = at.unit % G, b = rec_by_length(a.q_len, (int)a.batch, at.unit / G, (int)a.batch);      // (113 KB of LDS: one a CU)
  const int64_t first_pos = a.seq_lens[b] - a.q_len[b], t0 = a.q_start[b];
  const int n = a.q_len[b];
  if (n <= 0 || first_pos < 0) return;
  const int64_t chunk0 = __builtin_amdgcn_readfirstlane((int)rec_chunks_before(a.q_len, b));
  if (chunk0 + (n + L - 1) / L > max_chunks) return;            // (requests that share rows: more rows than the launch has)
  const int h = g * per + member / eblocks;
  const int e0 = member % eblocks * (16 * CB) + 16 * cw, e = e0 + r16;
  const bool on = e0 < E;                                        // (waves without columns take their part of the staging)
  const bool e_ok = e < E, wide = e0 + 16 <= E;
  const int C = 2 * G * D + H * E;
  const int64_t slot = a.state_indices[b];
  float* st = a.state + slot * a.state_ld + (int64_t)h * D * E + e;
  const int row0 = part * (NP / PARTS) + 4 * kq;                 // this lane's rows of S: row0 + 16 t + r
  f32x4 S[HT];
#pragma unroll
  for (int t = 0; t < HT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[t][r] = (first_pos > 0 && e_ok && row0 + 16 * t + r < D) ? st[(row0 + 16 * t + r) * E] : 0.f;
  float wt[kRecTaps];
#pragma unroll
  for (int i = 0; i < kRecTaps; ++i) wt[i] = (i < taps && e_ok) ? Elem<T>::to_f(((const T*)a.conv_v)[(int64_t)(h * E + e) * taps + taps - 1 - i]) : 0.f;
  const int64_t frag_ld = (int64_t)G * delta_frag_elems(NP), head_ld = (int64_t)H * kDeltaHead;
  const float* f = a.frags + chunk0 * frag_ld + g * delta_frag_elems(NP);
  const float* fh = a.frags + max_chunks * frag_ld + (chunk0 * H + h) * kDeltaHead;
  const T* p = (const T*)a.p + t0 * a.ld + a.v_off + h * E + e0;
  float* yo = a.work + t0 * a.wld + h * E + e0;
  // 16-byte pieces of the projection's and of the result's rows: everything starts on one
  const bool vec = wide && ((reinterpret_cast<uintptr_t>(p) | (uintptr_t)(a.ld * sizeof(T))) & 15) == 0 &&
                   ((reinterpret_cast<uintptr_t>(yo) | (uintptr_t)(a.wld * 4)) & 15) == 0 && a.ld < (1 << 24) && a.wld < (1 << 24);

  // raw inputs of the convolution, tokens 16 half - HALO .. 16 half + 15 of the chunk at l0 > 0
  Tile tile;
  auto fetch_v = [&](int l0) {
    int ln = lane;
    asm volatile("" : "+v"(ln));                                 // (addresses made where they are used, not held over the loop)
    if (vec && makes_v) tile.fetch_clamped(p, a.ld, l0 + 16 * half, n, ln);
  };
  // v of this lane's tokens 16 half + 4 kq + s, zero behind the portion; taps that the layer does not have see zeros
  auto convolve = [&](const float (&raw)[HALO + 4], int cnt, f32x4& v, bool& bad) {
    f32x4 y;
#pragma unroll
    for (int s = 0; s < 4; ++s) y[s] = wt[0] * raw[s + HALO];
    if (taps == kRecTaps) {
#pragma unroll
      for (int i = 1; i < kRecTaps; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) y[s] += wt[i] * raw[s + HALO - i];
    } else {
#pragma unroll
      for (int i = 1; i < kRecTaps - 1; ++i)
#pragma unroll
        for (int s = 0; s < 4; ++s) y[s] += wt[i] * __int_as_float(__float_as_int(raw[s + HALO - i]) & (i < taps ? -1 : 0));
    }
    float z[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) z[s] = rec_silu(y[s]);
    asm volatile("" : "+v"(z[0]), "+v"(z[1]), "+v"(z[2]), "+v"(z[3]));         // (all four, side by side, also of rows that there are not: see rec_conv_silu)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bool in = 16 * half + 4 * kq + s < cnt, large = !rec_moderate(y[s]);
      v[s] = in ? (large ? y[s] : z[s]) : 0.f;                    // (one that is not moderate: see `serial`)
      bad |= in & large;
    }
  };
  // ... of the chunk at l0 into this lane's place, by way of the wave's LDS
  float in[HALO + 4];
  auto place_v = [&](int l0) {
    if (!makes_v) return;
    T* raw = reinterpret_cast<T*>(ex_l[w][0]);
    int ln = lane;
    asm volatile("" : "+v"(ln));
    __builtin_amdgcn_wave_barrier();
    if (vec) {
      tile.place(raw, ln);
    } else {                                                     // (rows or columns that start off a 16-byte boundary: not fetched ahead)
      const int first = l0 + 16 * half - HALO, r16 = ln & 15;
      const bool e_ok = e0 + r16 < E;
      for (int r = ln >> 4; r < 16 + HALO; r += 4) raw[r * Tile::kStride + r16] = e_ok && first + r < n ? p[(int64_t)(first + r) * a.ld + r16] : Elem<T>::from_f(0.f);
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < HALO + 4; ++i) in[i] = Elem<T>::to_f(raw[(4 * (ln >> 4) + i) * Tile::kStride + (ln & 15)]);
  };
  u32x4 stage[2 * PIECES], stage_kt[AHEAD ? PIECES : 1], head;
  auto fetch_head = [&](const float* src) {
    if (tid < kDeltaHead / 4) head = reinterpret_cast<const u32x4*>(src)[tid];
  };
  auto fetch = [&](const float* src, u32x4* to) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PIECES; ++u)
      if (ALL % 512 == 0 || u * 512 + tid < ALL) to[u] = reinterpret_cast<const u32x4*>(src)[u * 512 + tid];
  };
  auto place = [&](uint8_t* dst, const u32x4* from) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < PIECES; ++u)
      if (ALL % 512 == 0 || u * 512 + tid < ALL) reinterpret_cast<u32x4*>(dst)[u * 512 + tid] = from[u];
  };
  // a wave's part of a sum and the others' (in pairs, so that all of them have the same)
  auto summed = [&](const f32x4& mine, int i) __attribute__((always_inline)) {
    if constexpr (PARTS == 2) return mine + *reinterpret_cast<const f32x4*>(&ex_l[w][i][16 * lane]);
    else return (mine + *reinterpret_cast<const f32x4*>(&sum_l[w ^ CB][i][16 * lane])) +
                (*reinterpret_cast<const f32x4*>(&sum_l[w ^ (2 * CB)][i][16 * lane]) + *reinterpret_cast<const f32x4*>(&sum_l[w ^ (3 * CB)][i][16 * lane]));
  };
  bool bad = false;
  fetch(f, stage);
  fetch(f + 3 * L * NP / 2, stage + PIECES);
  float flag_next = 0.f, keep_next = 0.f;
  if constexpr (AHEAD) {
    fetch_head(fh);
    fetch(f + 3 * L * NP, stage_kt);
    flag_next = f[9 * L * NP / 2], keep_next = fh[1536 + L - 1];
  }
  if (L < n) fetch_v(L);
  if (makes_v) {
#pragma unroll
    for (int i = 0; i < HALO + 4; ++i) {
      const int l = 16 * half + 4 * kq + i - HALO;
      in[i] = 0.f;
      if (e_ok && l < n) {
        if (l >= 0) in[i] = Elem<T>::to_f(p[(int64_t)l * a.ld + r16]);
        else if (first_pos > 0 && taps - 1 + l >= 0) in[i] = a.conv_state[slot * a.conv_ld + (int64_t)(taps - 1 + l) * C + 2 * G * D + h * E + e];
      }
    }
    f32x4 v;
    convolve(in, n, v, bad);
    *reinterpret_cast<f32x4*>(&v_l[cw][half][16 * lane]) = v;
  }
  place(k_l, stage);
  place(q_l, stage + PIECES);
  if (tid < 2) serial_l[tid] = 0;
  if (L < n) place_v(L);
  __syncthreads();

  // Two steps a chunk, what the next one needs on its way into registers during each: K S and Q S while K^T comes, then U, the products
  // inside the chunk and the new S while the next chunk's K and Q come.
  for (int l0 = 0; l0 < n; l0 += L) {
    const int cnt = n - l0 < L ? n - l0 : L, turn = (l0 / L) & 1;
    const bool more = l0 + L < n;
    const float* fn = f + (more ? frag_ld : 0);                 // (the last chunk fetches itself again)
    const float* fhn = fh + (more ? head_ld : 0);
    float* yr = yo + (int64_t)(l0 + 16 * half) * a.wld;
    const float flag = AHEAD ? flag_next : f[9 * L * NP / 2], keep = AHEAD ? keep_next : fh[1536 + L - 1];
    if constexpr (AHEAD) {
      fetch(fn, stage);
      fetch(fn + 3 * L * NP / 2, stage + PIECES);
      flag_next = fn[9 * L * NP / 2], keep_next = fhn[1536 + L - 1];
    } else {
      fetch_head(fh);
      fetch(f + 3 * L * NP, stage);
    }
    f32x4 O = {}, P[2] = {}, v[2] = {}, vn;
    bool serial = false, bad_next = false;
    if (on) {
      f32x4 Q[2];
      {
        if (conv_first) convolve(in, n - l0 - L, vn, bad_next);  // (the next chunk's; there is none: zeros)
        f32x4 PQ[4] = {};
        Split3 s[HT / 2];
        Frag16 c[HT / 2][4][3];
#pragma unroll
        for (int u = 0; u < HT / 2; ++u) {
          s[u] = rec_split8(S[2 * u], S[2 * u + 1]);
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int q = 0; q < 3; ++q)
              c[u][i][q].u = *reinterpret_cast<const uint4*>((i < 2 ? k_l : q_l) + q * PB + ((i & 1) * (NT / 2) + part * (HT / 2) + u) * 1024 + lane * 16);
          rec_mma_small<4>(c[u], s[u], PQ);
        }
#pragma unroll
        for (int u = 0; u < HT / 2; ++u) rec_mma_big<4>(c[u], s[u], PQ);
        if (makes_v && !conv_first) convolve(in, n - l0 - L, vn, bad_next);
#pragma unroll
        for (int i = 0; i < 2; ++i) P[i] = PQ[i], Q[i] = PQ[2 + i];
      }
      // the others of these columns get all of K S and the tokens of Q S that they finish
      if constexpr (PARTS == 2) {
        *reinterpret_cast<f32x4*>(&ex_l[w ^ 4][0][16 * lane]) = P[0];
        *reinterpret_cast<f32x4*>(&ex_l[w ^ 4][1][16 * lane]) = P[1];
        *reinterpret_cast<f32x4*>(&ex_l[w ^ 4][2][16 * lane]) = half ? Q[0] : Q[1];
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          *reinterpret_cast<f32x4*>(&sum_l[w][i][16 * lane]) = P[i];
          *reinterpret_cast<f32x4*>(&sum_l[w][2 + i][16 * lane]) = Q[i];
        }
      }
      O = half ? Q[1] : Q[0];
      float z = 0.f, top = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          z = fmaf(P[i][r], 0.f, z);
          top = fmaxf(top, fabsf(P[i][r]));
        }
      // An infinity or a NaN in the chunk, or one that sums of large values end in, would reach the tokens in front of it through a product
      // with a weight of zero, and so would a product of a large S with rows behind a step that resets it: the workgroup takes such a
      // chunk token by token, from S in the state row and v in LDS (a rare path: it must not set the kernel's registers).  Up to 2^90 what
      // U grows to, 2^31 at most, and the sums of it stay within 32 bits; |q| = D^-1/2: its products stay below the largest of S.
      const bool off = z != 0.f || top > 0x1p90f;
      if (__any(bad || flag != 0.f || keep != keep || off)) {    // (keep: see rec_flagged)
        float c = 0.f, most = 0.f;                               // (a column of S that has a NaN and no infinity stays so in either form)
#pragma unroll
        for (int t = 0; t < HT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            c = fmaf(S[t][r], 0.f, c);
            most = fmaxf(most, fabsf(S[t][r]));
          }
        c += __shfl_xor(c, 16, 64);
        c += __shfl_xor(c, 32, 64);
        serial = __any(bad || flag != 0.f || keep != keep || (off && (c == 0.f || !rec_finite(most))));
      }
      if (serial && lane == 0) serial_l[turn] = 1;
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i] = *reinterpret_cast<const f32x4*>(&v_l[cw][i][16 * lane]);
    }
    place(kt_l, AHEAD ? stage_kt : stage);
    if (tid < kDeltaHead / 4) reinterpret_cast<u32x4*>(head_l)[tid] = head;
    if (l0 + 2 * L < n) fetch_v(l0 + 2 * L);
    __syncthreads();
    if constexpr (AHEAD) {
      fetch_head(fhn);
      fetch(fn + 3 * L * NP, stage_kt);
    } else {
      fetch(fn, stage);
      fetch(fn + 3 * L * NP / 2, stage + PIECES);
    }
    serial = __builtin_amdgcn_readfirstlane(serial_l[turn]) != 0;
    if (tid == 0) serial_l[turn ^ 1] = 0;
    if (!serial) {
      if (on) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const f32x4 eb = *reinterpret_cast<const f32x4*>(head_l + 1536 + 16 * i + 4 * kq);
          P[i] = summed(P[i], i);
          v[i] -= eb * P[i];
        }
        if (ends) O = summed(O, PARTS == 2 ? 2 : 2 + half) * *reinterpret_cast<const f32x4*>(head_l + 1536 + 16 * half + 4 * kq);
        f32x4 Ti[3], M[2], wv[2];
#pragma unroll
        for (int i = 0; i < 3; ++i) Ti[i] = *reinterpret_cast<const f32x4*>(head_l + 256 * i + 4 * lane);
#pragma unroll
        for (int i = 0; i < 2; ++i) wv[i] = *reinterpret_cast<const f32x4*>(head_l + 1536 + L + 16 * i + 4 * kq);
        M[0] = *reinterpret_cast<const f32x4*>(head_l + 768 + 256 * half + 4 * lane);       // row tile `half` of the weighted Q K^T
        M[1] = *reinterpret_cast<const f32x4*>(head_l + 768 + 512 * half + 4 * lane);
        // (products of 16 or 32 columns: as they are, in fp32; both waves of these columns make U)
        f32x4 U[2] = {}, U1 = {};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          U[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ti[0][s], v[0][s], U[0], 0, 0, 0);
          U[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ti[1][s], v[0][s], U[1], 0, 0, 0);
          U1 = __builtin_amdgcn_mfma_f32_16x16x4f32(Ti[2][s], v[1][s], U1, 0, 0, 0);
        }
        U[1] += U1;
        const Split3 us = rec_split8(U[0] * wv[0], U[1] * wv[1]);
        {
          Frag16 kt[HT][3];
#pragma unroll
          for (int t = 0; t < HT; ++t)
#pragma unroll
            for (int q = 0; q < 3; ++q) kt[t][q].u = *reinterpret_cast<const uint4*>(kt_l + q * PB + (part * HT + t) * 1024 + lane * 16);
          f32x4 A[HT] = {};
          rec_mma_small<HT>(kt, us, A);
          rec_mma_big<HT>(kt, us, A);
#pragma unroll
          for (int t = 0; t < HT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[t][r] = fmaf(S[t][r], keep, A[t][r]);
        }
        f32x4 O1 = {};
        if (ends) {
#pragma unroll
          for (int s = 0; s < 4; ++s) O = __builtin_amdgcn_mfma_f32_16x16x4f32(M[0][s], U[0][s], O, 0, 0, 0);
          if (half) {
#pragma unroll
            for (int s = 0; s < 4; ++s) O1 = __builtin_amdgcn_mfma_f32_16x16x4f32(M[1][s], U[1][s], O1, 0, 0, 0);
          }
          O += O1;
        }
      }
    } else {
      int rows = D, step = E, ln = lane;
      asm volatile("" : "+s"(rows), "+s"(step), "+v"(ln));       // (no addresses held over the loop)
      const int r16 = ln & 15, kq = ln >> 4, row0 = part * (NP / PARTS) + 4 * kq, e = e0 + r16;
      const bool e_ok = e < E;
      float* st = a.state + slot * a.state_ld + (int64_t)h * D * E + e;
      float* vs = reinterpret_cast<float*>(ex_l[0][0]) + 16 * cw + r16;          // v [32][16 CB]
      if (makes_v)
#pragma unroll
        for (int s = 0; s < 4; ++s) vs[(16 * half + 4 * kq + s) * (16 * CB)] = rec_silu_if_large(half ? v[1][s] : v[0][s]);
      if (e_ok)
#pragma unroll
        for (int t = 0; t < HT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (row0 + 16 * t + r < rows) st[(row0 + 16 * t + r) * step] = S[t][r];
      __syncthreads();
      if (part == 0 && on) {
#pragma unroll 1
        for (int t = 0; t < cnt; ++t) {
          // row t of K: this lane group's four of every 16
          const uint16_t* kr = reinterpret_cast<const uint16_t*>(f) + (t >> 4) * (NT / 2) * 512 + 8 * (16 * kq + (t & 15));
          float dk = 0.f, dq = 0.f, kd = 0.f;
#pragma unroll 1
          for (int u = 0; u < 4 * NT; ++u) {
            const int row = 16 * (u >> 2) + 4 * kq + (u & 3), at = (u >> 3) * 512 + (u & 3) + (u & 4);
            if (row < rows) {
              const float kv = rec_joined(kr + at, L * NP), qv = rec_joined(kr + 3 * L * NP + at, L * NP), sv = e_ok ? st[row * step] : 0.f;
              dk += sv * kv;
              dq += sv * qv;
              kd += kv * qv;
            }
          }
          dk += __shfl_xor(dk, 16, 64);
          dk += __shfl_xor(dk, 32, 64);
          dq += __shfl_xor(dq, 16, 64);
          dq += __shfl_xor(dq, 32, 64);
          kd += __shfl_xor(kd, 16, 64);
          kd += __shfl_xor(kd, 32, 64);
          const float gt = fh[1536 + 2 * L + t], bt = fh[1536 + 3 * L + t];
          const float u1 = bt * (vs[t * (16 * CB)] - gt * dk);
#pragma unroll 1
          for (int u = 0; u < 4 * NT; ++u) {
            const int row = 16 * (u >> 2) + 4 * kq + (u & 3);
            if (row < rows && e_ok) st[row * step] = gt * st[row * step] + rec_joined(kr + (u >> 3) * 512 + (u & 3) + (u & 4), L * NP) * u1;
          }
          if (kq == 0 && e_ok) yr[(int64_t)t * a.wld + r16] = gt * dq + u1 * kd;
        }
      }
      __syncthreads();
#pragma unroll
      for (int t = 0; t < HT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[t][r] = e_ok && row0 + 16 * t + r < rows ? st[(row0 + 16 * t + r) * step] : 0.f;
      __builtin_amdgcn_s_waitcnt(0x0f70);                        // (vmcnt(0) here, or the other path waits for what it has in flight where they join)
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more && on && makes_v) *reinterpret_cast<f32x4*>(&v_l[cw][half][16 * lane]) = vn;
    bad = bad_next;
    place(k_l, stage);
    place(q_l, stage + PIECES);
    // behind the wait for the pieces (memory answers in order), so that it is the next one's
    if (!serial && ends) {
      __builtin_amdgcn_wave_barrier();
      float* ol = reinterpret_cast<float*>(ex_l[w][0]);
      int ln = lane;
      asm volatile("" : "+v"(ln));
#pragma unroll
      for (int r = 0; r < 4; ++r) ol[(4 * kq + r) * kOutStride + r16] = O[r];
      __builtin_amdgcn_wave_barrier();
      if (vec) {
        const int row = ln >> 2;
        if (16 * half + row < cnt)
          *reinterpret_cast<f32x4*>(reinterpret_cast<char*>(yr) + ((uint32_t)row * (uint32_t)(a.wld * 4) + 16u * (ln & 3))) = *reinterpret_cast<const f32x4*>(ol + row * kOutStride + 4 * (ln & 3));
      } else if (e_ok) {
        const int r16 = ln & 15;
#pragma unroll 1
        for (int row = ln >> 4; row < 16 && 16 * half + row < cnt; row += 4) yr[(int64_t)row * a.wld + r16] = ol[row * kOutStride + r16];
      }
    }
    if (l0 + 2 * L < n) place_v(l0 + 2 * L);
    f = fn;
    fh = fhn;
    __syncthreads();
  }
  int rows = D, step = E;
  asm volatile("" : "+s"(rows), "+s"(step));                     // (no addresses of 16 rows held over the loop)
  if (e_ok)
#pragma unroll
    for (int t = 0; t < HT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (row0 + 16 * t + r < rows) st[(row0 + 16 * t + r) * step] = S[t][r];
}

// Keys of up to 64, operands of fp32: the chunks of a request in turn, a wave per (request, head, 16 columns of S) with nothing shared: four waves a workgroup for the
// sake of their common loads.  S [NP x 16] stays in accumulators: lane (r16, kq) holds rows 16 t + 4 kq + r of column r16, which is
// also how the right-hand operand of a product over the rows is held, so S, R = V - e^b K S and U go from sums into products
// without moving; v is convolved in its place by the lane that needs it, from raw inputs in the wave's own LDS.  Left-hand operands
// come straight into registers in the order they are used, not through LDS, the next chunk's into the registers that this chunk has
// just read.  Results leave by way of the wave's LDS; nothing is shared between waves, so there are no barriers.  Half the
// products of keys of 128 leave the two barriers and the exchange of delta_chunk_walk_kernel nothing to cover them with: 32 heads of 64 x 64,
// 1 request of 1000 rows 144 us, there 160; 1 of 4000 rows 456 / 531; 8 of 900 rows 212 / 236; 32 of 40 rows 95 / 97.
template <typename T, int W>
__global__ void __launch_bounds__(256, W) delta_chunk_walk_small_kernel(DeltaArgs a, int64_t max_chunks) {
  constexpr int NP = kDeltaSmall, L = kRecChunk, NT = NP / 16, HALO = kRecHalo;
  __shared__ __attribute__((aligned(16))) T in_l[4][RowTile<T>::kElems];       // a wave's own: raw inputs of its convolution
  __shared__ __attribute__((aligned(16))) float o_l[4][L * kOutStride];         // ... results on their way out (token by token: its v)
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, kq = lane >> 4;
  // workgroups of one (request, key head) read the same operands: they go to one XCD (workgroup ids go round the 8 XCDs)
  const int H = a.H, G = a.G, D = a.D, E = a.E, taps = a.taps, per = H / G;
  const int eblocks = (E + 63) / 64, members = per * eblocks;
  const RecPlace at = rec_place((int)a.batch * G, members);
  if (at.unit < 0) return;
  const int member = at.member, b = at.unit / G, g = at.unit % G;
  const int64_t first_pos = a.seq_lens[b] - a.q_len[b], t0 = a.q_start[b];
  const int n = a.q_len[b];
  if (n <= 0 || first_pos < 0) return;
  const int64_t chunk0 = rec_chunks_before(a.q_len, b);
  if (chunk0 + (n + L - 1) / L > max_chunks) return;            // (requests that share rows: more rows than the launch has)
  const int h = g * per + member / eblocks;
  const int e0 = member % eblocks * 64 + 16 * w, e = e0 + r16;
  if (e0 >= E) return;
  const bool e_ok = e < E, wide = e0 + 16 <= E;
  const int C = 2 * G * D + H * E;
  const int64_t slot = a.state_indices[b];
  float* st = a.state + slot * a.state_ld + (int64_t)h * D * E + e;
  f32x4 S[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * t + 4 * kq + r;
      S[t][r] = (first_pos > 0 && e_ok && row < D) ? st[row * E] : 0.f;
    }
  float wt[kRecTaps];
#pragma unroll
  for (int i = 0; i < kRecTaps; ++i)
    wt[i] = (i < taps && e_ok) ? Elem<T>::to_f(((const T*)a.conv_v)[(int64_t)(h * E + e) * taps + taps - 1 - i]) : 0.f;
  const int64_t frag_ld = (int64_t)G * delta_frag_elems(NP), head_ld = (int64_t)H * kDeltaHead;
  const float* f = a.frags + chunk0 * frag_ld + g * delta_frag_elems(NP) + 4 * lane;
  const float* fh = a.frags + max_chunks * frag_ld + (chunk0 * H + h) * kDeltaHead;
  const T* p = (const T*)a.p + t0 * a.ld + a.v_off + h * E + e0;
  float* yo = a.work + t0 * a.wld + h * E + e0;
  // 16-byte pieces of the projection's and of the result's rows: everything starts on one
  const bool vec = wide && ((reinterpret_cast<uintptr_t>(p) | (uintptr_t)(a.ld * sizeof(T))) & 15) == 0 &&
                   ((reinterpret_cast<uintptr_t>(yo) | (uintptr_t)(a.wld * 4)) & 15) == 0;

  // raw inputs of the convolution, tokens 16 j + 4 kq - HALO + i of the chunk at l0 > 0
  RowTile<T> tile;
  auto fetch_v = [&](int l0) { if (vec) tile.fetch(p, a.ld, l0, n, lane); };
  // v of this lane's tokens, zero behind the portion; taps that the layer does not have see zeros
  auto convolve = [&](const float (&x)[2][HALO + 4], int cnt, f32x4 (&v)[2], bool& bad) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        float y = wt[0] * x[j][s + HALO];
#pragma unroll
        for (int i = 1; i < kRecTaps; ++i) y += wt[i] * __int_as_float(__float_as_int(x[j][s + HALO - i]) & (i < taps ? -1 : 0));
        float z = rec_silu(y);
        asm volatile("" : "+v"(z));                              // (straight-line code: it goes between the products)
        const bool in = 16 * j + 4 * kq + s < cnt;
        v[j][s] = in ? (rec_moderate(y) ? z : y) : 0.f;       // (one that is not: see `serial`)
        bad |= in && !rec_moderate(y);
      }
  };
  f32x4 v[2];
  bool bad = false;
  {
    float x[2][HALO + 4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < HALO + 4; ++i) {
        const int l = 16 * j + 4 * kq + i - HALO;
        x[j][i] = 0.f;
        if (e_ok && l < n) {
          if (l >= 0) x[j][i] = Elem<T>::to_f(p[(int64_t)l * a.ld + r16]);
          else if (first_pos > 0 && taps - 1 + l >= 0) x[j][i] = a.conv_state[slot * a.conv_ld + (int64_t)(taps - 1 + l) * C + 2 * G * D + h * E + e];
        }
      }
    convolve(x, n, v, bad);
  }
  f32x4 K[2 * NT], Q[2 * NT], KT[2 * NT], Ti[3], M[3], eb[2], wv[2];
  float flag;
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) K[i] = *reinterpret_cast<const f32x4*>(f + 256 * i);
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) Q[i] = *reinterpret_cast<const f32x4*>(f + L * NP + 256 * i);
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    Ti[i] = *reinterpret_cast<const f32x4*>(fh + 256 * i + 4 * lane);
    M[i] = *reinterpret_cast<const f32x4*>(fh + 768 + 256 * i + 4 * lane);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    eb[i] = *reinterpret_cast<const f32x4*>(fh + 1536 + 16 * i + 4 * kq);
    wv[i] = *reinterpret_cast<const f32x4*>(fh + 1536 + L + 16 * i + 4 * kq);
  }
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) KT[i] = *reinterpret_cast<const f32x4*>(f + 2 * L * NP + 256 * i);
  flag = f[3 * L * NP - 4 * lane];
  if (L < n) fetch_v(L);

  for (int l0 = 0; l0 < n; l0 += L) {
    const int cnt = n - l0 < L ? n - l0 : L;
    const bool more = l0 + L < n;
    const float* fn = f + (more ? frag_ld : 0);                 // (the last chunk fetches itself again)
    const float* fhn = fh + (more ? head_ld : 0);
    float* yr = yo + (int64_t)l0 * a.wld;
    // An infinity or a NaN in the chunk, or one that sums of large values end in, would reach the tokens in front of it through a product
    // with a weight of zero, and so would a product of a large S with rows behind a step that resets it: the wave takes such a chunk
    // token by token behind the products, which then count for nothing, from S in the state row and v in LDS (a rare path: it must
    // not set the kernel's registers)
    const bool flagged = bad || flag != 0.f;
    int rows = D, step = E;
    asm volatile("" : "+s"(rows), "+s"(step));
    bool serial;
    {
      const float keep = __shfl(eb[1][3], 63, 64);
      f32x4 P[2] = {}, O[2] = {};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i) P[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(K[i * NT + t][s], S[t][s], P[i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 2 * NT; ++i) K[i] = *reinterpret_cast<const f32x4*>(fn + 256 * i);
      flag = fn[3 * L * NP - 4 * lane];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i) O[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(Q[i * NT + t][s], S[t][s], O[i], 0, 0, 0);
      // the next chunk's v between the products: a product keeps the matrix pipe for 32 cycles, in which a few of these fit
      f32x4 vn[2];
      bad = false;
      {
        float x[2][HALO + 4];
        if (vec) {
          tile.place(in_l[w], lane);
        } else {                                                 // (rows or columns that start off a 16-byte boundary: not fetched ahead)
          for (int r = kq; r < L + HALO; r += 4)
            in_l[w][r * RowTile<T>::kStride + r16] = e_ok && l0 + L - HALO + r < n ? p[(int64_t)(l0 + L - HALO + r) * a.ld + r16] : Elem<T>::from_f(0.f);
        }
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int i = 0; i < HALO + 4; ++i) x[j][i] = Elem<T>::to_f(in_l[w][(16 * j + 4 * kq + i) * RowTile<T>::kStride + r16]);
        convolve(x, n - l0 - L, vn, bad);
      }
#pragma unroll
      for (int i = 0; i < 8 * NT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
      }
#pragma unroll
      for (int i = 0; i < 2 * NT; ++i) Q[i] = *reinterpret_cast<const f32x4*>(fn + L * NP + 256 * i);
      if (l0 + 2 * L < n) fetch_v(l0 + 2 * L);
      {
        float z = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) z = fmaf(P[i / 4][i % 4], 0.f, z);      // (|q| = D^-1/2: its products stay below the largest of S)
        serial = __any(flagged || keep != keep);                 // (keep: see rec_flagged)
        if (__any(z != 0.f)) {                                   // (a column of S that is not finite stays so in either form)
          float c = 0.f;
#pragma unroll
          for (int t = 0; t < NT; ++t) c = fmaf(S[t][0], 0.f, fmaf(S[t][1], 0.f, fmaf(S[t][2], 0.f, fmaf(S[t][3], 0.f, c))));
          c += __shfl_xor(c, 16, 64);
          c += __shfl_xor(c, 32, 64);
          serial |= __any(z != 0.f && c == 0.f);
        }
      }
      if (serial) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int s = 0; s < 4; ++s) o_l[w][(16 * j + 4 * kq + s) * kOutStride + r16] = rec_silu_if_large(v[j][s]);
        if (e_ok)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (16 * t + 4 * kq + r < rows) st[(16 * t + 4 * kq + r) * step] = S[t][r];
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        v[i] -= eb[i] * P[i];
        O[i] *= eb[i];
      }
      f32x4 U[2] = {};
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i) U[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ti[i][s], v[0][s], U[i], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; ++s) U[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ti[2][s], v[1][s], U[1], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i) O[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(M[i][s], U[0][s], O[i], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; ++s) O[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(M[2][s], U[1][s], O[1], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 2; ++i) U[i] *= wv[i];
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        Ti[i] = *reinterpret_cast<const f32x4*>(fhn + 256 * i + 4 * lane);
        M[i] = *reinterpret_cast<const f32x4*>(fhn + 768 + 256 * i + 4 * lane);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        eb[i] = *reinterpret_cast<const f32x4*>(fhn + 1536 + 16 * i + 4 * kq);
        wv[i] = *reinterpret_cast<const f32x4*>(fhn + 1536 + L + 16 * i + 4 * kq);
      }
      if (serial) {
      } else if (cnt == L && vec) {
        rec_store_tile(O, o_l[w], yr, a.wld, lane);
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (16 * i + 4 * kq + r < cnt && e_ok) yr[(int64_t)(16 * i + 4 * kq + r) * a.wld + r16] = O[i][r];
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) S[t] *= keep;
#pragma unroll
      for (int t = 0; t < NT; t += 2)
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < 2; ++i) S[t + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(KT[2 * (t + i) + k][s], U[k][s], S[t + i], 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 2 * NT; ++i) KT[i] = *reinterpret_cast<const f32x4*>(fn + 2 * L * NP + 256 * i);
      v[0] = vn[0];
      v[1] = vn[1];
    }
    if (serial) {
#pragma unroll 1
      for (int t = 0; t < cnt; ++t) {
        // row t of K (tile row t / 16, lane r16 = t % 16): this lane group's four of every 16
        const float* kr = f - 4 * lane + (t >> 4) * NT * 256 + 4 * (16 * kq + (t & 15));
        float dk = 0.f, dq = 0.f, kd = 0.f;
#pragma unroll 1
        for (int u = 0; u < 4 * NT; ++u) {
          const int row = 16 * (u >> 2) + 4 * kq + (u & 3);
          if (row < rows) {
            const float kv = kr[(u >> 2) * 256 + (u & 3)], qv = kr[L * NP + (u >> 2) * 256 + (u & 3)], sv = e_ok ? st[row * step] : 0.f;
            dk += sv * kv;
            dq += sv * qv;
            kd += kv * qv;
          }
        }
        dk += __shfl_xor(dk, 16, 64);
        dk += __shfl_xor(dk, 32, 64);
        dq += __shfl_xor(dq, 16, 64);
        dq += __shfl_xor(dq, 32, 64);
        kd += __shfl_xor(kd, 16, 64);
        kd += __shfl_xor(kd, 32, 64);
        const float gt = fh[1536 + 2 * L + t], bt = fh[1536 + 3 * L + t];
        const float u1 = bt * (o_l[w][t * kOutStride + r16] - gt * dk);
#pragma unroll 1
        for (int u = 0; u < 4 * NT; ++u) {
          const int row = 16 * (u >> 2) + 4 * kq + (u & 3);
          if (row < rows && e_ok) st[row * step] = gt * st[row * step] + kr[(u >> 2) * 256 + (u & 3)] * u1;
        }
        if (kq == 0 && e_ok) yr[(int64_t)t * a.wld + r16] = gt * dq + u1 * kd;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[t][r] = e_ok && 16 * t + 4 * kq + r < rows ? st[(16 * t + 4 * kq + r) * step] : 0.f;
      __builtin_amdgcn_sched_barrier(0);
    }
    f = fn;
    fh = fhn;
  }
  int rows = D, step = E;
  asm volatile("" : "+s"(rows), "+s"(step));                     // (no addresses of 32 rows held over the loop)
  if (e_ok)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (16 * t + 4 * kq + r < rows) st[(16 * t + 4 * kq + r) * step] = S[t][r];
}

// The same with 16-byte accesses: a head is taken by LP = E / 8 lanes (a power of two), 64 / LP heads per wave.  Bound by HBM: 7262
// tokens of 32 heads of 128, 238 MB: 84 us -> 46.
template <typename T, int LP>
__global__ void __launch_bounds__(256) delta_post_vec_kernel(DeltaArgs a, int conv_blocks) {
  // the first workgroups move the convolutions' inputs on, 256 channels of a request each: the others neither read nor write them (a
  // launch of its own is 2.5 us)
  if ((int)blockIdx.x < conv_blocks) {
    const int per = (2 * a.G * a.D + a.H * a.E + 255) / 256;
    delta_conv_state<T>(a, blockIdx.x / per, blockIdx.x % per * 256 + threadIdx.x);
    return;
  }
  const int lane = threadIdx.x & 63, sl = lane % LP, E = a.E;
  const int64_t item = ((int64_t)(blockIdx.x - conv_blocks) * 4 + (threadIdx.x >> 6)) * (64 / LP) + lane / LP;
  const bool on = item < a.num_tokens * a.H;
  const int64_t t = on ? item / a.H : 0;
  const int h = on ? (int)(item % a.H) : 0;
  const float* o = a.work + t * a.wld + a.o_off + (int64_t)h * E + sl * 8;
  const float4 o0 = *reinterpret_cast<const float4*>(o), o1 = *reinterpret_cast<const float4*>(o + 4);
  const Vec16<T> gate = load16((const T*)a.p + t * a.ld + a.gate_off + (int64_t)h * E + sl * 8), nw = load16((const T*)a.norm_w + sl * 8);
  const float x[8] = {o0.x, o0.y, o0.z, o0.w, o1.x, o1.y, o1.z, o1.w};
  float sq = 0.f;
#pragma unroll
  for (int i = 0; i < 8; ++i) sq += x[i] * x[i];
#pragma unroll
  for (int m = LP / 2; m > 0; m >>= 1) sq += __shfl_xor(sq, m, 64);
  if (!on) return;
  const float inv = 1.0f / sqrtf(sq / (float)E + a.eps);
  Vec16<T> r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r.e[i] = Elem<T>::from_f(x[i] * inv * Elem<T>::to_f(nw.e[i]) * silu_f(Elem<T>::to_f(gate.e[i])));
  store16((T*)a.out + t * a.out_ld + (int64_t)h * E + sl * 8, r);
}

}  // namespace semipd

using namespace semipd;

extern "C" int64_t semipd_delta_rule_work_width(int num_heads, int num_k_heads, int k_dim, int v_dim) {
  const int64_t w = 2 * (int64_t)num_k_heads * k_dim + (int64_t)num_heads * v_dim + 2 * (int64_t)num_heads;
  return (w + 3) / 4 * 4;
}

// The rows per request from which a prompt batch goes in chunks: on average, since the lengths are on the device.  (The time token by token
// is the longest request's: an uneven batch gains from chunks at a lower average than these.)  A chunk costs the same however few its rows
// and heads; token by token a token's heads are prepared one behind another, so that form is ahead where there are few. Token by token
// against chunks, whole call, 32 heads over 8 of 128 x 128: 1 request of 2 rows 47 / 34 us, 48 rows 82 / 38; 16 requests of 2 rows 79 / 68;
// 32 of 2 rows 114 / 115, 16 rows 198 / 123; 64 of 4 rows 207 / 237, 8 rows 259 / 240.  16 over 2 of 128 x 128: 1 request of 8 rows 33 / 36,
// 12 rows 37 / 36; 16 of 12 rows 52 / 50.  8 over 1: 1 request of 16 rows 31 / 35, 24 rows 39 / 36; 32 of 12 rows 50 / 50.  Keys of up to
// 64: 32 over 8 of 64 x 64, 4 requests of 2 rows 46 / 32, 32 of 8 rows 59 / 64, 16 rows 73 / 66; 16 over 4 of 64 x 128, 16 of 24 rows 43 /
// 46, 32 rows 49 / 46; 8 over 1 of 64 x 64, 8 of 32 rows 30 / 35, 32 of 48 rows 49 / 42.  (Some would be ahead in chunks earlier, 8 of 12
// rows 45 / 33, but a state of theirs is then 1.1 times as far from the 64-bit one.)
// 9 to 16 requests of 1 row: 24 heads over 4 of 128 x 128, 16 requests 51 / 57, of 2 rows 54 / 57; 32 over 2 65 / 65; 32 over 32 95 / 69.  One key
// head for all: a request is a unit of the walk, and one past 8 (16) of them costs what the next 8 would: 30 over 1, 8 requests of 1 row
// 53 / 56, 9 of 3 rows 73 / 78, 12 of 3 rows 69 / 79, 16 of 2 rows 80 / 80, 17 of 6 rows 95 / 101, 24 of 6 rows 117 / 104; 14 over 1, 1
// request of 12 rows 39 / 41, 14 rows 41 / 41, 2 of 13 rows 45 / 42.
static int64_t delta_chunk_min_rows(int64_t batch, int num_heads, int num_k_heads, int k_dim) {
  const int heads = num_heads + 2 * num_k_heads;
  if (k_dim <= 64) return heads >= 32 ? (batch <= 4 ? 0 : 16) : heads >= 16 ? 32 : 48;
  if (heads >= 32 && num_k_heads == 1) return batch <= 4 ? 0 : batch <= 8 ? 2 : batch <= 16 ? 18 - batch : 6 + (7 - (batch - 1) % 8) / 3;
  if (heads >= 32) return batch <= 8 ? 0 : batch <= 16 ? (heads < 36 ? 2 : 0) : 6;
  if (heads >= 16) return num_k_heads == 1 && batch == 1 ? 14 : 12;
  return batch < 32 ? 22 : 14;
}

extern "C" int64_t semipd_delta_rule_chunk_elems(int64_t num_tokens, int64_t batch, int num_heads, int num_k_heads, int k_dim, int taps) {
  if (batch <= 0 || num_heads <= 0 || num_k_heads <= 0 || k_dim > 128 || taps > kRecTaps) return 0;
  if (num_tokens < delta_chunk_min_rows(batch, num_heads, num_k_heads, k_dim) * batch) return 0;
  const int64_t elems = rec_max_chunks(num_tokens, batch) * (num_k_heads * delta_frag_elems(k_dim <= 64 ? 64 : 128) + (int64_t)num_heads * kDeltaHead);
  return rec_short_and_large(num_tokens, batch, elems) ? 0 : elems;
}

template <typename T, int NP>
static void launch_delta_chunks(const DeltaArgs& a, hipStream_t s) {
  const int64_t chunks = rec_max_chunks(a.num_tokens, a.batch);
  hipLaunchKernelGGL((delta_chunk_operands_kernel<T, NP>), dim3((unsigned)chunks, (unsigned)a.G, rec_head_splits(chunks * a.G, a.H / a.G)), dim3(256), 0, s, a);
  const int64_t members = (int64_t)(a.H / a.G) * ((a.E + 63) / 64);
  const dim3 grid(rec_walk_blocks(a.batch * a.G, members));
  if constexpr (NP > kDeltaSmall) {
    // 32 columns a workgroup as long as every one of them has a CU of the launch's share (rec_walk_blocks: of the XCD with the most)
    const unsigned narrow = rec_walk_blocks(a.batch * a.G, (int64_t)(a.H / a.G) * ((a.E + 31) / 32));
    if (narrow <= launch_cus()) hipLaunchKernelGGL((delta_chunk_walk_kernel<T, NP, 2>), dim3(narrow), dim3(512), 0, s, a, chunks);
    else hipLaunchKernelGGL((delta_chunk_walk_kernel<T, NP, 4>), grid, dim3(512), 0, s, a, chunks);
  } else if (a.batch * a.G * members > 256) {
    // more workgroups than CUs: two a CU, at the price of 40 spilled registers (32 heads of 64 x 64, one / two a CU, whole call: 64 requests
    // of 64 rows 226 / 202 us; 4 requests of 96 rows, 128 workgroups: 52 / 58)
    hipLaunchKernelGGL((delta_chunk_walk_small_kernel<T, 2>), grid, dim3(256), 0, s, a, chunks);
  } else {
    hipLaunchKernelGGL((delta_chunk_walk_small_kernel<T, 1>), grid, dim3(256), 0, s, a, chunks);
  }
}

// gate and norm, and the convolutions' inputs moved on, both behind everything that reads them; in one launch unless the result may be
// written over the inputs; 16-byte accesses where a head is a power of two of pieces and everything starts on one
static int launch_delta_post(const DeltaArgs& a, int dtype, hipStream_t s) {
  const int lp = a.E / 8;
  const bool vec = dtype != SEMIPD_F32 && a.E % 8 == 0 && lp <= 64 && (lp & (lp - 1)) == 0 && a.gate_off % 8 == 0 && a.ld % 8 == 0 &&
                   a.out_ld % 8 == 0 && a.wld % 4 == 0 && a.o_off % 4 == 0 && aligned16(a.p) && aligned16(a.out) && aligned16(a.work) &&
                   aligned16(a.norm_w);
  const int64_t gd = (int64_t)a.G * a.D, he = (int64_t)a.H * a.E, blocks = a.taps > 1 ? (2 * gd + he + 255) / 256 : 0;
  auto apart = [&](int64_t off, int64_t n) { return rec_apart(a.p, off, n, a.ld, a.out, he, a.out_ld, a.num_tokens); };
  const bool one = vec && apart(a.q_off, gd) && apart(a.k_off, gd) && apart(a.v_off, he);
  if (blocks && !one)
    SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((delta_conv_state_kernel<T>), dim3((unsigned)blocks, (unsigned)a.batch), dim3(256), 0, s, a));
  if (!vec) {
    SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((delta_post_kernel<T>), dim3((unsigned)a.num_tokens), dim3(256), 0, s, a));
    return 0;
  }
  const int64_t items = a.num_tokens * a.H, per = 4 * (64 / lp);
  const int cb = (int)(one ? blocks * a.batch : 0);
  const dim3 grid((unsigned)((items + per - 1) / per + cb));
  SEMIPD_DISPATCH_HALF(dtype, T, {
    switch (lp) {
      case 1: hipLaunchKernelGGL((delta_post_vec_kernel<T, 1>), grid, dim3(256), 0, s, a, cb); break;
      case 2: hipLaunchKernelGGL((delta_post_vec_kernel<T, 2>), grid, dim3(256), 0, s, a, cb); break;
      case 4: hipLaunchKernelGGL((delta_post_vec_kernel<T, 4>), grid, dim3(256), 0, s, a, cb); break;
      case 8: hipLaunchKernelGGL((delta_post_vec_kernel<T, 8>), grid, dim3(256), 0, s, a, cb); break;
      case 16: hipLaunchKernelGGL((delta_post_vec_kernel<T, 16>), grid, dim3(256), 0, s, a, cb); break;
      case 32: hipLaunchKernelGGL((delta_post_vec_kernel<T, 32>), grid, dim3(256), 0, s, a, cb); break;
      default: hipLaunchKernelGGL((delta_post_vec_kernel<T, 64>), grid, dim3(256), 0, s, a, cb); break;
    }
  });
  return 0;
}

static int delta_rule(const void* proj, int64_t ld, int64_t q_off, int64_t k_off, int64_t v_off, int64_t gate_off,
                                 int64_t a_off, int64_t b_off, const void* conv_q, const void* conv_k, const void* conv_v,
                                 const float* a_log, const float* dt_bias, const void* norm_weight, float eps, float* work,
                                 int64_t work_ld, float* state, int64_t state_ld, float* conv_state, int64_t conv_ld,
                                 const int64_t* state_indices, const int64_t* seq_lens, const int32_t* q_start,
                                 const int32_t* q_len, int64_t batch, int64_t num_tokens, int num_heads, int num_k_heads,
                                 int k_dim, int v_dim, int taps, void* out, int64_t out_ld, float* chunk_work, int64_t chunk_elems,
                      int dtype, void* stream) {
  SEMIPD_CHECK_ARG(batch >= 0 && num_tokens >= 0, SEMIPD_EINVAL, "delta_rule: bad sizes");
  if (batch == 0 || num_tokens == 0) return 0;
  SEMIPD_CHECK_ARG(num_heads > 0 && num_k_heads > 0 && num_heads % num_k_heads == 0, SEMIPD_ESHAPE,
                   "delta_rule: %d heads over %d q / k heads", num_heads, num_k_heads);
  SEMIPD_CHECK_ARG(k_dim > 0 && k_dim <= 256 && v_dim > 0 && taps >= 1 && taps <= 64, SEMIPD_ESHAPE,
                   "delta_rule: key size %d (at most 256), value size %d, %d taps (1 .. 64)", k_dim, v_dim, taps);
  const bool in_one = q_start == nullptr && (k_dim >= 32 ? 4 : 1) * (int64_t)v_dim <= 1024;       // (decode batches that need no work rows)
  SEMIPD_CHECK_ARG(proj && conv_q && conv_k && conv_v && a_log && dt_bias && norm_weight && (work || in_one) && state && state_indices &&
                       seq_lens && out && (conv_state || taps == 1),
                   SEMIPD_EINVAL, "delta_rule: null pointer");
  SEMIPD_CHECK_ARG((q_start == nullptr) == (q_len == nullptr), SEMIPD_EINVAL, "delta_rule: q_start and q_len come together");
  SEMIPD_CHECK_ARG(q_start != nullptr || num_tokens == batch, SEMIPD_EINVAL, "delta_rule: one row per request without q_start");
  const int64_t C = 2 * (int64_t)num_k_heads * k_dim + (int64_t)num_heads * v_dim;
  const int64_t want = q_start ? semipd_delta_rule_chunk_elems(num_tokens, batch, num_heads, num_k_heads, k_dim, taps) : 0;
  const bool chunks = want > 0 && chunk_work && chunk_elems >= want && aligned16(chunk_work);
  SEMIPD_CHECK_ARG((in_one || work_ld >= (chunks ? (int64_t)num_heads * v_dim : C + 2 * num_heads)) && state_ld >= (int64_t)num_heads * k_dim * v_dim &&
                       (taps == 1 || conv_ld >= (taps - 1) * C) && out_ld >= (int64_t)num_heads * v_dim,
                   SEMIPD_EINVAL, "delta_rule: a row of the work buffer, the state or the output is too short");
  DeltaArgs a{proj, ld, q_off, k_off, v_off, gate_off, a_off, b_off, conv_q, conv_k, conv_v, a_log, dt_bias, norm_weight,
              work, work_ld, state, state_ld, conv_state, conv_ld, state_indices, seq_lens, q_start, q_len, batch, num_tokens,
              num_heads, num_k_heads, k_dim, v_dim, taps, eps, out, out_ld, chunks ? 0 : 2 * num_k_heads * k_dim, chunk_work};
  hipStream_t st = as_stream(stream);
  // lanes per column and rows of S per lane: four lanes share a column from 32 rows up
  const int ds = k_dim >= 32 ? 4 : 1;
  const int per = (k_dim + ds - 1) / ds;
  const int dpt = per <= 4 ? 4 : (per <= 8 ? 8 : (per <= 16 ? 16 : (per <= 32 ? 32 : 64)));
  // a decode batch whose state rows lie on 16-byte boundaries: up to 16 pieces of four columns a thread.  Four teams a workgroup while
  // the chip takes all workgroups at once, two where a CU goes through several, so that one loads while another computes (32 heads
  // of 64 x 64, 8 key heads, four teams / two, us: 3 requests 9.8 / 12.1, 32 13.2 / 15.3, 48 22.9 / 18.3, 128 47.7 / 37.7)
  const int per_group = num_heads / num_k_heads, most = k_dim * v_dim > 4 * 1024 || batch * num_k_heads > 256 ? 2 : 4, teams = per_group < most ? per_group : most;
  // A key head with more value heads than teams goes round (shared out over several workgroups as long as the CUs have none, 256 in
  // all; the convolutions' inputs then move on in a second launch).  The kernel below is ahead where these rounds are short (k_dim up to
  // 64: from 128 workgroups on they are as long as its own; up to 1024 elements of state a head a team has idle threads).  Below / here,
  // shared out / in turn, us: 32 heads over 1 of 128 x 128, 1 request 17.8 / 16.7 / 107, 32 requests 57 / 36 / 121; 8 over 1 of 64 x 64,
  // 1 request 10.3 / 11.8 / 14.0, 128 requests 17.4 / 16.5 / 18.1; 64 over 2 of 32 x 32, 32 requests 12.8 / - / 43.
  const int rounds = (per_group + teams - 1) / teams;
  const bool step_pays = rounds == 1 || ((k_dim > 64 || batch * num_k_heads >= 128) && (k_dim * v_dim > 1024 || rounds <= 2));
  const size_t step_lds = ((size_t)2 * k_dim + (size_t)per_group * v_dim + (size_t)teams * 8 * v_dim + 4) * sizeof(float);
  if (q_start == nullptr && batch <= 65535 && v_dim >= 16 && v_dim <= 256 && (v_dim & (v_dim - 1)) == 0 && k_dim % 2 == 0 && k_dim * v_dim <= 16 * 1024 &&
      aligned16(state) && state_ld % 4 == 0 && step_lds <= 65536 && step_pays) {
    const int nit = (k_dim * v_dim + 1023) / 1024;
    const int64_t room = 256 / (batch * num_k_heads), splits = rounds < room ? rounds : (room < 1 ? 1 : room);
    const dim3 sgrid((unsigned)num_k_heads, (unsigned)batch, (unsigned)splits);
    SEMIPD_DISPATCH_DTYPE(dtype, T, {
      const auto go = [&](auto early) {
        constexpr int EARLY = decltype(early)::value;
        if (nit <= 4) hipLaunchKernelGGL((delta_step_kernel<T, 4, EARLY>), sgrid, dim3(256 * teams), step_lds, st, a);
        else if (nit <= 8) hipLaunchKernelGGL((delta_step_kernel<T, 8, EARLY>), sgrid, dim3(256 * teams), step_lds, st, a);
        else hipLaunchKernelGGL((delta_step_kernel<T, 16, EARLY>), sgrid, dim3(256 * teams), step_lds, st, a);
      };
      // (instances of their own: what is asked for early holds its registers where it is not used, five taps and more 1 to 5 % faster without;
      // two taps with the loads of four 3 % slower in batches of a few requests)
      if (taps <= 2) go(std::integral_constant<int, 2>{});
      else if (taps <= kRecTaps) go(std::integral_constant<int, kRecTaps>{});
      else go(std::integral_constant<int, 0>{});
    });
    if (splits > 1 && taps > 1)
      SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((delta_conv_state_kernel<T>), dim3((unsigned)((C + 255) / 256), (unsigned)batch),
                                                         dim3(256), 0, st, a));
    return launch_status("delta_rule(step)");
  }
  if (q_start == nullptr && (int64_t)ds * v_dim <= 1024) {
    // a decode batch: one launch, then the convolutions' inputs move on (the launch above has read the old ones)
    const int threads = (ds * v_dim + 63) / 64 * 64;
    const size_t lds = (size_t)(2 * dpt * ds + 4) * sizeof(float);
    const dim3 grid((unsigned)batch, (unsigned)num_heads);
#define SEMIPD_DELTA_DEC(DPT, DS) \
  SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((delta_decode_kernel<T, DPT, DS>), grid, dim3(threads), lds, st, a))
    if (ds == 1) {
      switch (dpt) {
        case 4: SEMIPD_DELTA_DEC(4, 1); break;
        case 8: SEMIPD_DELTA_DEC(8, 1); break;
        case 16: SEMIPD_DELTA_DEC(16, 1); break;
        default: SEMIPD_DELTA_DEC(32, 1); break;
      }
    } else {
      switch (dpt) {
        case 8: SEMIPD_DELTA_DEC(8, 4); break;
        case 16: SEMIPD_DELTA_DEC(16, 4); break;
        case 32: SEMIPD_DELTA_DEC(32, 4); break;
        default: SEMIPD_DELTA_DEC(64, 4); break;
      }
    }
#undef SEMIPD_DELTA_DEC
    if (taps > 1)
      SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((delta_conv_state_kernel<T>), dim3((unsigned)((C + 255) / 256), (unsigned)batch),
                                                         dim3(256), 0, st, a));
    return launch_status("delta_rule(decode)");
  }
  if (chunks) {
    SEMIPD_DISPATCH_DTYPE(dtype, T, if (k_dim <= 64) launch_delta_chunks<T, 64>(a, st); else launch_delta_chunks<T, 128>(a, st));
    if (launch_delta_post(a, dtype, st)) return SEMIPD_EDTYPE;
    return launch_status("delta_rule(chunks)");
  }
  SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((delta_prep_kernel<T>), dim3((unsigned)num_tokens), dim3(256), 0, st, a));
  // one wave per workgroup: the workgroups of a CU stage and walk their tokens independently, so the loads of one overlap
  // the arithmetic of the others
  const int threads = 64;
  const int cols = threads / ds;
  const size_t lds = (size_t)kStage * (2 * ds * (dpt + 4) + 4 + cols) * sizeof(float);
  const dim3 grid((unsigned)batch, (unsigned)num_heads, (unsigned)((v_dim + cols - 1) / cols));
#define SEMIPD_DELTA_SCAN(DPT, DS) hipLaunchKernelGGL((delta_scan_kernel<DPT, DS>), grid, dim3(threads), lds, st, a)
  if (ds == 1) {
    switch (dpt) {
      case 4: SEMIPD_DELTA_SCAN(4, 1); break;
      case 8: SEMIPD_DELTA_SCAN(8, 1); break;
      case 16: SEMIPD_DELTA_SCAN(16, 1); break;
      default: SEMIPD_DELTA_SCAN(32, 1); break;
    }
  } else {
    switch (dpt) {
      case 8: SEMIPD_DELTA_SCAN(8, 4); break;
      case 16: SEMIPD_DELTA_SCAN(16, 4); break;
      case 32: SEMIPD_DELTA_SCAN(32, 4); break;
      default: SEMIPD_DELTA_SCAN(64, 4); break;
    }
  }
#undef SEMIPD_DELTA_SCAN
  if (launch_delta_post(a, dtype, st)) return SEMIPD_EDTYPE;
  return launch_status("delta_rule");
}

extern "C" int semipd_delta_rule(const void* proj, int64_t ld, int64_t q_off, int64_t k_off, int64_t v_off, int64_t gate_off,
                                 int64_t a_off, int64_t b_off, const void* conv_q, const void* conv_k, const void* conv_v,
                                 const float* a_log, const float* dt_bias, const void* norm_weight, float eps, float* work,
                                 int64_t work_ld, float* state, int64_t state_ld, float* conv_state, int64_t conv_ld,
                                 const int64_t* state_indices, const int64_t* seq_lens, const int32_t* q_start,
                                 const int32_t* q_len, int64_t batch, int64_t num_tokens, int num_heads, int num_k_heads,
                                 int k_dim, int v_dim, int taps, void* out, int64_t out_ld, int dtype, void* stream) {
  return delta_rule(proj, ld, q_off, k_off, v_off, gate_off, a_off, b_off, conv_q, conv_k, conv_v, a_log, dt_bias, norm_weight, eps, work, work_ld,
                    state, state_ld, conv_state, conv_ld, state_indices, seq_lens, q_start, q_len, batch, num_tokens, num_heads, num_k_heads, k_dim,
                    v_dim, taps, out, out_ld, nullptr, 0, dtype, stream);
}

extern "C" int semipd_delta_rule_record(const void* record) {
  SEMIPD_CHECK_ARG(record != nullptr, SEMIPD_EINVAL, "delta_rule: null record");
  int64_t r[36];
  double eps;
  memcpy(r, record, sizeof(r));
  memcpy(&eps, &r[14], sizeof(eps));
  auto at = [&](int i) { return reinterpret_cast<void*>(r[i]); };
  return semipd_delta_rule(at(0), r[1], r[2], r[3], r[4], r[5], r[6], r[7], at(8), at(9), at(10), (const float*)at(11), (const float*)at(12), at(13), (float)eps,
                           (float*)at(15), r[16], (float*)at(17), r[18], (float*)at(19), r[20], (const int64_t*)at(21), (const int64_t*)at(22),
                           (const int32_t*)at(23), (const int32_t*)at(24), r[25], r[26], (int)r[27], (int)r[28], (int)r[29], (int)r[30], (int)r[31], at(32), r[33],
                           (int)r[34], at(35));
}

extern "C" int semipd_delta_rule_prompt(const void* proj, int64_t ld, int64_t q_off, int64_t k_off, int64_t v_off, int64_t gate_off,
                                 int64_t a_off, int64_t b_off, const void* conv_q, const void* conv_k, const void* conv_v,
                                 const float* a_log, const float* dt_bias, const void* norm_weight, float eps, float* work,
                                 int64_t work_ld, float* state, int64_t state_ld, float* conv_state, int64_t conv_ld,
                                 const int64_t* state_indices, const int64_t* seq_lens, const int32_t* q_start,
                                 const int32_t* q_len, int64_t batch, int64_t num_tokens, int num_heads, int num_k_heads,
                                 int k_dim, int v_dim, int taps, void* out, int64_t out_ld, float* chunk_work, int64_t chunk_elems, int dtype, void* stream) {
  return delta_rule(proj, ld, q_off, k_off, v_off, gate_off, a_off, b_off, conv_q, conv_k, conv_v, a_log, dt_bias, norm_weight, eps, work, work_ld,
                    state, state_ld, conv_state, conv_ld, state_indices, seq_lens, q_start, q_len, batch, num_tokens, num_heads, num_k_heads, k_dim,
                    v_dim, taps, out, out_ld, chunk_work, chunk_elems, dtype, stream);
}
