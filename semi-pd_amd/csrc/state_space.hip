// Selective state-space recurrence (the scalar-decay form with a matrix state per head) over a pool of per-request state
// rows (gfx950, wave64).
//
// Rows of the projection hold [z: H E | x: H E | B: G N | C: G N | dt: H].  x, B and C pass a causal convolution over time
// per channel (taps weights and a bias per channel, zeros in front of the sequence) and silu; the last taps - 1 inputs of
// every channel are part of the request's state.  Per head h (group g = h / (H / G)), with S [N, E] in fp32 from zero:
//     dt_t = softplus(dt_t + dt_bias_h);   S <- exp(-exp(A_log_h) dt_t) S + dt_t B_t x_t^T;   y_t = S^T C_t + D_h x_t
// then y * silu(z), an RMS norm over each of `norm_groups` equal parts of the row, times a weight.  Everything behind the
// projection GEMM is fp32 whatever the activation type.
//
//  * ssm_prep_kernel: a workgroup per (tile of 32 tokens -- one token in small batches --, 1024 channels), four channels per
//    thread with their taps in registers where alignment allows: convolution + bias + silu of the token's x | B | C channels (inputs in front
//    of the portion come from the state row), dt and the decay -> an fp32 work row per token.
//  * ssm_conv_state: the last taps - 1 inputs of the portion (shifted in behind what the row held) -> state row, by the first workgroups of
//    ssm_post_vec_kernel's launch or in ssm_conv_state_kernel.
//  * ssm_scan_kernel: ONE WAVE per (request, head, block of 64 / NS columns of S); a column of S lives in the registers of NS
//    adjacent lanes, NPT rows each, so a step is one multiply-add per register for the update, one for the read-out, and a
//    log2(NS)-step lane reduction.  B, C, x, dt and the decay of kStage tokens sit in LDS; the next stage's 16-byte pieces are
//    fetched into registers while a stage is multiplied and go into the other half of the LDS buffer behind it.  The state is read when the rows
//    of the launch do not start the sequence and written back after the last row, so a prompt cut into portions, single
//    decode tokens and a slot that another request held all take one path.
//  * Prompt batches: ssm_chunk_operands_kernel and ssm_chunk_walk_kernel (states of up to 64 rows, up to a workgroup a CU:
//    ssm_chunk_walk_small_kernel) in place of the three, 32 tokens at a time on the matrix cores, operands of 24 bits and fp32 sums.
//  * ssm_post_kernel / ssm_post_vec_kernel: gate, grouped norm, weight -> the output projection's input, a workgroup per token.
//  * ssm_step_kernel: batches of one token per request in place of preparation and recurrence, a workgroup per (head, request).
//  * ssm_decode_kernel: all of the above for batches of one token per request whose state is small, a workgroup per request.
#include <cstring>
#include <type_traits>

#include "common.h"
#include "recurrent_chunks.h"

namespace semipd {

struct SsmArgs {
  const void* p; int64_t ld;                       // projection rows
  int64_t z_off, x_off, dt_off;                    // columns of z, of x | B | C (one range, the convolution's channels), of dt
  const void* conv_w; const void* conv_b;          // [C, taps], [C] of the activation type, C = H E + 2 G N
  const float* dt_bias; const float* a_log; const float* d_skip;      // [H] fp32
  const void* norm_w; int norm_groups; float eps;  // [H E] of the activation type
  float* work; int64_t wld;                        // fp32 [T, wld]: x (later y) [H E] | B [G N] | C [G N] | dt [H] | decay [H]
  float* state; int64_t state_ld;                  // fp32 [slots, >= H N E]: S[h][n][e]
  float* conv_state; int64_t conv_ld;              // fp32 [slots, >= (taps - 1) C]: [tap][channel]
  const int64_t* state_indices; const int64_t* seq_lens;
  const int32_t* q_start; const int32_t* q_len;    // [B] or NULL (one row per request)
  int64_t batch, num_tokens;
  int H, G, N, E, taps;
  void* out; int64_t out_ld;                       // [T, H E] of the activation type
  float* frags;                                    // operands of the chunks (matrix-core form), see ssm_chunk_operands_kernel
};

__device__ __forceinline__ float ssm_silu(float x) { return x / (1.0f + expf(-x)); }
__device__ __forceinline__ float ssm_softplus(float x) { return x > 20.f ? x : log1pf(expf(x)); }

// the request that owns row t, the row's index inside the request's portion, the portion's length and its first position
__device__ __forceinline__ bool ssm_locate(const SsmArgs& a, int64_t t, int& b, int64_t& li, int64_t& n, int64_t& first_pos) {
  if (a.q_start == nullptr) {
    b = (int)t; li = 0; n = 1; first_pos = a.seq_lens[b] - 1;
    return first_pos >= 0;
  }
  for (int r = 0; r < (int)a.batch; ++r) {
    const int64_t s = a.q_start[r], m = a.q_len[r];
    if (t >= s && t < s + m) {
      b = r; li = t - s; n = m; first_pos = a.seq_lens[r] - m;
      return true;
    }
  }
  return false;
}

// one channel of the convolution for row t (index li of its portion): bias + sum of taps, then silu
template <typename T>
__device__ __forceinline__ float ssm_conv_channel(const SsmArgs& a, const T* p, const float* cs, bool fresh, int64_t t, int64_t li,
                                                  int c, int C) {
  const T* cw = (const T*)a.conv_w + (int64_t)c * a.taps;
  float y = a.conv_b ? Elem<T>::to_f(((const T*)a.conv_b)[c]) : 0.f;
  for (int i = 0; i < a.taps; ++i) {
    const int64_t l = li - i;
    float x;
    if (l >= 0) x = Elem<T>::to_f(p[(t - i) * a.ld + a.x_off + c]);
    else if (fresh) x = 0.f;
    else x = cs[(int64_t)(a.taps - 1 + l) * C + c];
    y += Elem<T>::to_f(cw[a.taps - 1 - i]) * x;
  }
  return ssm_silu(y);
}

// ---------------------------------------------------------------------------------- convolution, silu, step sizes, decays
constexpr int kPrepChannels = 1024;      // channels per workgroup (blockIdx.y walks a token's channels)

// four adjacent elements of the activation type in one access
template <typename T> __device__ __forceinline__ void load4(const T* p, float (&x)[4]) {
  if constexpr (sizeof(T) == 2) {
    const uint2 w = *reinterpret_cast<const uint2*>(p);
    T e;
    e.v = (uint16_t)(w.x & 0xffffu); x[0] = Elem<T>::to_f(e);
    e.v = (uint16_t)(w.x >> 16);     x[1] = Elem<T>::to_f(e);
    e.v = (uint16_t)(w.y & 0xffffu); x[2] = Elem<T>::to_f(e);
    e.v = (uint16_t)(w.y >> 16);     x[3] = Elem<T>::to_f(e);
  } else {
    const float4 w = *reinterpret_cast<const float4*>(p);
    x[0] = w.x; x[1] = w.y; x[2] = w.z; x[3] = w.w;
  }
}

constexpr int kPrepMaxTaps = 8;          // taps whose weights the four-channel form keeps in registers
constexpr int kPrepTileBlocks = 512;
constexpr int kPrepTile = 32;            // tokens a workgroup of a prompt batch walks with them

template <typename T, bool VEC4>
__global__ void __launch_bounds__(256) ssm_prep_kernel(SsmArgs a, int tile) {
  const int C = a.H * a.E + 2 * a.G * a.N;
  const T* p = (const T*)a.p;
  const int c_lo = blockIdx.y * kPrepChannels;
  const int c_hi = c_lo + kPrepChannels < C ? c_lo + kPrepChannels : C;
  const int taps = a.taps;
  // four channels per thread (8- / 16-byte reads of the inputs and of the state's rows, one 16-byte write), their taps and
  // bias in registers for all tokens of the tile
  const int c4 = c_lo + 4 * threadIdx.x;
  const bool mine = VEC4 && c4 < c_hi;
  float wt[kPrepMaxTaps][4], bias[4] = {0.f, 0.f, 0.f, 0.f};
  if (mine) {
    const T* cw = (const T*)a.conv_w + (int64_t)c4 * taps;
#pragma unroll
    for (int i = 0; i < kPrepMaxTaps; ++i)
#pragma unroll
      for (int u = 0; u < 4; ++u) wt[i][u] = i < taps ? Elem<T>::to_f(cw[u * taps + taps - 1 - i]) : 0.f;      // i tokens back
    if (a.conv_b)
#pragma unroll
      for (int u = 0; u < 4; ++u) bias[u] = Elem<T>::to_f(((const T*)a.conv_b)[c4 + u]);
  }
  for (int tt = 0; tt < tile; ++tt) {
    const int64_t t = (int64_t)blockIdx.x * tile + tt;
    if (t >= a.num_tokens) break;
    int b;
    int64_t li, n, first_pos;
    if (!ssm_locate(a, t, b, li, n, first_pos)) continue;
    const float* cs = a.conv_state + a.state_indices[b] * a.conv_ld;
    float* w = a.work + t * a.wld;
    const bool fresh = first_pos == 0;
    if constexpr (VEC4) {
      if (mine) {
        float y[4] = {bias[0], bias[1], bias[2], bias[3]};
#pragma unroll
        for (int i = 0; i < kPrepMaxTaps; ++i) {
          if (i >= taps) break;
          const int64_t l = li - i;
          float x[4] = {0.f, 0.f, 0.f, 0.f};
          if (l >= 0) load4(p + (t - i) * a.ld + a.x_off + c4, x);
          else if (!fresh) {
            const float4 v = *reinterpret_cast<const float4*>(cs + (int64_t)(taps - 1 + l) * C + c4);
            x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) y[u] += wt[i][u] * x[u];
        }
        *reinterpret_cast<float4*>(w + c4) = float4{ssm_silu(y[0]), ssm_silu(y[1]), ssm_silu(y[2]), ssm_silu(y[3])};
      }
    } else {
      for (int c = c_lo + threadIdx.x; c < c_hi; c += 256) w[c] = ssm_conv_channel<T>(a, p, cs, fresh, t, li, c, C);
    }
    if (blockIdx.y == 0)
      for (int h = threadIdx.x; h < a.H; h += 256) {
        const float dt = ssm_softplus(Elem<T>::to_f(p[t * a.ld + a.dt_off + h]) + a.dt_bias[h]);
        w[C + h] = dt;
        w[C + a.H + h] = expf(-expf(a.a_log[h]) * dt);
      }
  }
}

// ---------------------------------------------------------------------------------- the inputs the next portion looks back at
template <typename T>
__device__ __forceinline__ void ssm_conv_state(const SsmArgs& a, int b, int c) {
  const int C = a.H * a.E + 2 * a.G * a.N;
  if (c >= C) return;
  int64_t t0, n, first_pos;
  if (a.q_start == nullptr) {
    t0 = b; n = 1; first_pos = a.seq_lens[b] - 1;
  } else {
    t0 = a.q_start[b]; n = a.q_len[b]; first_pos = a.seq_lens[b] - n;
  }
  if (n <= 0 || first_pos < 0) return;
  float* cs = a.conv_state + a.state_indices[b] * a.conv_ld;
  const T* p = (const T*)a.p;
  const int keep = a.taps - 1;
  // entry s of the new state is the input at index n - keep + s of the portion; a negative index reaches into the old
  // state (entry s + n > s, read before entry s is written) or, at the start of a sequence, in front of it
  auto input = [&](int s) {
    const int64_t l = n - keep + s;
    if (l >= 0) return Elem<T>::to_f(p[(t0 + l) * a.ld + a.x_off + c]);
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
__global__ void __launch_bounds__(256) ssm_conv_state_kernel(SsmArgs a) {
  ssm_conv_state<T>(a, blockIdx.y, blockIdx.x * 256 + threadIdx.x);
}

// ---------------------------------------------------------------------------------- the recurrence
constexpr int kSsmStage = 8;       // tokens of a stage: their B, C, x, dt and decay sit in LDS, the next stage's in registers

template <int NPT, int NS, bool VEC4>
__global__ void __launch_bounds__(64) ssm_scan_kernel(SsmArgs a) {
  // per staged token: B [NP] | C [NP] | x of the block's columns [COLS] | dt | decay | 2 unused.  B and C are cut into the NS
  // slices that the lanes of a column read, each slice followed by 4 unused floats: the 16-byte reads of the NS lanes then
  // fall into different banks (slices of 32 floats alone would put lanes 0 and 2 on the same ones)
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr int SEG = NS > 1 ? NPT + 4 : NPT, NP = SEG * NS, COLS = 64 / NS, TOK = 2 * NP + COLS + 4, TOKU = TOK / 4;
  constexpr int U = (kSsmStage * TOKU + 63) / 64;          // 16-byte pieces of a stage per lane
  const int lane = threadIdx.x;
  const int H = a.H, G = a.G, N = a.N, E = a.E;
  const int eblocks = (E + COLS - 1) / COLS;
  int64_t id = blockIdx.x;
  const int eb = (int)(id % eblocks); id /= eblocks;
  const int h = (int)(id % H);
  const int b = (int)(id / H);
  int64_t t0, n, first_pos;
  if (a.q_start == nullptr) {
    t0 = b; n = 1; first_pos = a.seq_lens[b] - 1;
  } else {
    t0 = a.q_start[b]; n = a.q_len[b]; first_pos = a.seq_lens[b] - n;
  }
  if (n <= 0 || first_pos < 0) return;
  const int g = h / (H / G);
  const int col = lane / NS, ns = lane % NS;
  const int e = eb * COLS + col;
  const bool e_ok = e < E;
  const int n0 = ns * NPT;
  const int C = H * E + 2 * G * N;
  float* st = a.state + a.state_indices[b] * a.state_ld + (int64_t)h * N * E;
  float S[NPT];
#pragma unroll
  for (int i = 0; i < NPT; ++i) S[i] = (first_pos > 0 && e_ok && n0 + i < N) ? st[(int64_t)(n0 + i) * E + e] : 0.f;
  const float dskip = a.d_skip ? a.d_skip[h] : 0.f;
  // piece u of a staged token: four of B, of C, of the block's x, or (dt, decay, -, -); rows shorter than NP are zero-filled
  auto piece = [&](const float* w, int u) -> float4 {
    const float* src;
    int have;                     // elements of the piece that exist
    if (u < NP / 2) {
      const int pos = 4 * (u < NP / 4 ? u : u - NP / 4), off = pos % SEG;
      if (off >= NPT) return float4{0.f, 0.f, 0.f, 0.f};                 // the gap behind a slice
      const int i = (pos / SEG) * NPT + off;                               // row of the state
      src = w + H * E + (u < NP / 4 ? 0 : G * N) + g * N + i;
      have = N - i;
    } else if (u < NP / 2 + COLS / 4) {
      src = w + h * E + eb * COLS + 4 * (u - NP / 2);
      have = E - eb * COLS - 4 * (u - NP / 2);
    } else {
      return float4{w[C + h], w[C + H + h], 0.f, 0.f};
    }
    if (have <= 0) return float4{0.f, 0.f, 0.f, 0.f};
    if (VEC4 && have >= 4) return *reinterpret_cast<const float4*>(src);
    return float4{src[0], have > 1 ? src[1] : 0.f, have > 2 ? src[2] : 0.f, have > 3 ? src[3] : 0.f};
  };
  // A stage's pieces are fetched into registers while the stage in front of it is multiplied, and put into the other half
  // of the LDS buffer behind it: the loads of HBM rows are in flight during the arithmetic.
  float4 v[U];
  auto fetch = [&](int64_t s0) {
    const int cnt = (int)((n - s0) < kSsmStage ? (n - s0) : kSsmStage);
    const int total = cnt * TOKU;
    const float* w0 = a.work + (t0 + s0) * a.wld;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = u * 64 + lane;
      v[u] = it < total ? piece(w0 + (int64_t)(it / TOKU) * a.wld, it % TOKU) : float4{0.f, 0.f, 0.f, 0.f};
    }
  };
  auto stash = [&](float* buf) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int it = u * 64 + lane;
      if (it < kSsmStage * TOKU) *reinterpret_cast<float4*>(buf + 4 * it) = v[u];
    }
  };
  fetch(0);
  stash(lds);
  __syncthreads();
  int half = 0;
  for (int64_t s0 = 0; s0 < n; s0 += kSsmStage) {
    const int cnt = (int)((n - s0) < kSsmStage ? (n - s0) : kSsmStage);
    const bool more = s0 + kSsmStage < n;
    if (more) fetch(s0 + kSsmStage);
    const float* stage = lds + half * (kSsmStage * TOK);
    for (int k = 0; k < cnt; ++k) {
      const float* l = stage + k * TOK;
      const float xv = l[2 * NP + col], dtv = l[2 * NP + COLS], dec = l[2 * NP + COLS + 1];
      const float dx = dtv * xv;
      float y = 0.f;
#pragma unroll
      for (int i = 0; i < NPT; i += 4) {
        const float4 bv = *reinterpret_cast<const float4*>(l + ns * SEG + i);
        const float4 cv = *reinterpret_cast<const float4*>(l + NP + ns * SEG + i);
        S[i] = dec * S[i] + bv.x * dx;         y += S[i] * cv.x;
        S[i + 1] = dec * S[i + 1] + bv.y * dx; y += S[i + 1] * cv.y;
        S[i + 2] = dec * S[i + 2] + bv.z * dx; y += S[i + 2] * cv.z;
        S[i + 3] = dec * S[i + 3] + bv.w * dx; y += S[i + 3] * cv.w;
      }
      if (NS >= 2) y += __shfl_xor(y, 1, 64);
      if (NS >= 4) y += __shfl_xor(y, 2, 64);
      if (NS >= 8) y += __shfl_xor(y, 4, 64);
      if (ns == 0 && e_ok) a.work[(t0 + s0 + k) * a.wld + h * E + e] = y + dskip * xv;
    }
    half ^= 1;
    if (more) stash(lds + half * (kSsmStage * TOK));
    __syncthreads();
  }
  if (e_ok) {
#pragma unroll
    for (int i = 0; i < NPT; ++i)
      if (n0 + i < N) st[(int64_t)(n0 + i) * E + e] = S[i];
  }
}

// ---------------------------------------------------------------------------------- prompt batches: 32 tokens at a time
// With la_t = log of the decay, b_t its running sum inside a chunk of 32 tokens and S the state in front of the chunk:
//     y_t = e^(b_t) S^T C_t + sum_(s <= t) (C_t . B_s) e^(b_t - b_s) dt_s x_s + D x_t
//     S  <- e^(b_last) S + sum_s B_s (e^(b_last - b_s) dt_s x_s)^T
// Every exponent is at most 0.  The products with S are products of fp32 values on the bf16 matrix cores, three pieces a value (see
// rec_mma), their sums fp32; the others are v_mfma_f32_16x16x4_f32.  The state behind 4 requests of 1900 tokens is 8.5e-8 from the 64-bit
// one (2-norm; all products of fp32 operands: 9.6e-8; with the six products added to S one by one: 1.24e-7).  b is summed, and its
// differences are taken, in 64 bits, so a weight near 1 behind a strong decay is as good as the product of the decays themselves.
// Bound: token by token a step is a chain of LDS reads, 64 multiply-adds and lane sums (1.0 us of a wave's time; 7262 tokens of 4
// requests, 128 heads of 128 x 64: 2394 us + 322 of preparation through fp32 work rows).  In chunks on the fp32 matrix pipe, a wave all
// rows of 16 columns: 560 us (140 products of 32 cycles a wave and chunk, 38 % of the SIMD cycles, waiting for its operands in between).
// Here 325: per wave and chunk 48 products of 16 cycles, 6 of 32 and 340 vector instructions (pieces of S 88, convolution 110), of which
// a SIMD takes one in 4 cycles from two waves or more but only one in 8 from one; LDS reads 22 % of its cycles.  What that took: C and B^T
// once a workgroup through LDS (24 KB each; straight into registers every wave reads them again), two waves a column block with half the
// rows each (four a SIMD instead of two: one request of 2303 rows 265 -> 235), requests placed by length (412 -> 345), and the waits of a rare path kept in
// it (345 -> 325).  Operands 58.
// Chunks of 32 and not 64: the same products with S, half the ones inside a chunk, half the LDS.
// Elements of the operands of one (chunk, group), counted in fp32: C and B^T in three planes of bf16 each, left-hand operands of 16 x 16 x 32
// products in the order in which they are held, [tile][lane][8] (see rec_split8; tiles of C: 16 tokens x 32 rows of S, of B^T: 16 rows x
// the tokens; for ssm_chunk_walk_small_kernel in fp32, of 16 x 16 x 16 products, as the head's), and a flag in a piece of 4.  Of one (chunk, head), fp32: tiles 00, 10, 11 of the weighted C B^T, left-hand operands of 16 x
// 16 x 16 products, [tile][lane][4], lane (r16, kq) element s = row r16, column 4 kq + s, then e^(b_t) | e^(b_last - b_t) dt_t | dt | decay.
__host__ __device__ constexpr int64_t ssm_frag_elems(int np) { return 3 * (int64_t)kRecChunk * np + 4; }
constexpr int kSsmHead = 3 * 256 + 4 * kRecChunk;

// What the heads of a group share, a workgroup per (chunk, group): convolution + bias + silu of the group's B and C channels (a
// channel per thread, its taps and the last inputs in registers), laid down as operands; the 32 x 32 products C B^T and, half a wave
// per head in turn (lane = token), step sizes, running log decays and the weighted C B^T.  NP: N up to a multiple of 64, zeros behind
// N and behind the portion.  The first heads' gates are fetched in front of the convolution, and nothing waits for what is written: 128 heads of 128
// x 64 over 8, 1 request of 100 rows, whole call, 37.3 -> 35.8 us, 6 of 28 51.2 -> 49.2; a chip full of it lays down 197 MB and is
// bound by these (4 of 1900 within the noise).
template <typename T, int NP, bool PIECES>
__global__ void __launch_bounds__(256, 4) ssm_chunk_operands_kernel(SsmArgs a) {
  constexpr int L = kRecChunk, CS = NP + 4, PS = L + 4;
  __shared__ __attribute__((aligned(16))) float c_l[L * CS];
  __shared__ __attribute__((aligned(16))) float b_l[L * CS];
  float* const cb_l = c_l;                                      // (C B^T, behind the products)
  __shared__ __attribute__((aligned(16))) double cum_l[8 * L];
  __shared__ __attribute__((aligned(16))) float dt_l[8 * L];
  const int tid = threadIdx.x, g = blockIdx.y;
  RecChunk at;
  if (!rec_find_chunk(a.q_len, a.seq_lens, a.q_start, (int)a.batch, blockIdx.x, at) || at.first_pos < 0) return;
  const int64_t l0 = at.c * L, t0 = at.q_start + l0;
  const int cnt = (int)(at.n - l0 < L ? at.n - l0 : L);
  const int N = a.N, taps = a.taps, per = a.H / a.G;
  const int C = a.H * a.E + 2 * a.G * N;
  float* frag = a.frags + ((int64_t)blockIdx.x * a.G + g) * ssm_frag_elems(NP);
  const float* kept = l0 == 0 && at.first_pos > 0 && taps > 1 ? a.conv_state + a.state_indices[at.b] * a.conv_ld : nullptr;
  bool bad = false;
  // what the first heads' step sizes are made of: raw, so that nothing waits for it here
  const int hw = tid >> 5, t = tid & 31;
  T gate_dt;
  float gate_bias, gate_log;
  auto fetch_gates = [&](int hh) {                               // (of rows and heads that there are)
    const int h = g * per + min(hh, per - 1);
    gate_dt = ((const T*)a.p)[(t0 + min(t, cnt - 1)) * a.ld + a.dt_off + h];
    gate_bias = a.dt_bias[h];
    gate_log = a.a_log[h];
  };
  fetch_gates(blockIdx.z * 8 + hw);
  for (int ch = tid; ch < 2 * NP; ch += 256) {
    const bool is_c = ch >= NP;
    const int r = is_c ? ch - NP : ch;
    float* dst = (is_c ? c_l : b_l) + r;
    if (r < N) {
      const int col = a.H * a.E + (is_c ? a.G * N : 0) + g * N + r;               // among the convolution's channels
      const T* p = (const T*)a.p + t0 * a.ld + a.x_off + col;
      const T* cw = (const T*)a.conv_w + (int64_t)col * taps;
      const T shift = *(a.conv_b ? (const T*)a.conv_b + col : cw);
      float wt[kRecTaps], in[kRecTaps], x[L];
      rec_channel<T>(p, a.ld, cnt, cw, taps, l0 > 0, kept != nullptr ? kept + col : nullptr, C, wt, in, x);
      const float bias = a.conv_b ? Elem<T>::to_f(shift) : 0.f;
      bad |= rec_conv_silu(wt, in, x, bias, taps, cnt, dst, CS);
    } else {
      for (int t = 0; t < L; ++t) dst[t * CS] = 0.f;
    }
  }
  const int any_bad = __syncthreads_or(bad);
  const bool lays = blockIdx.z == 0;                             // (the workgroups of a group's heads all have the operands, one lays them down)
  if (lays && tid == 0) frag[ssm_frag_elems(NP) - 4] = any_bad ? 1.f : 0.f;      // (at the end that would wait for what is written)
  if constexpr (PIECES) {
    // pieces of three planes: C, tiles (16 tokens, 32 rows of S), and B^T, tiles (16 rows of S, the tokens)
    for (int i = lays ? tid : L * NP; i < 2 * (L * NP / 8); i += 256) {
      const bool is_c = i < L * NP / 8;
      const int it = is_c ? i : i - L * NP / 8, tile = it >> 6, ln = it & 63, r = ln & 15, q4 = 4 * (ln >> 4);
      f32x4 x0, x1;
      if (is_c) {
        const float* s = c_l + (16 * (tile / (NP / 32)) + r) * CS + 32 * (tile % (NP / 32)) + q4;
        x0 = *reinterpret_cast<const f32x4*>(s);
        x1 = *reinterpret_cast<const f32x4*>(s + 16);
      } else {
        const float* s = b_l + q4 * CS + 16 * tile + r;
        x0 = f32x4{s[0], s[CS], s[2 * CS], s[3 * CS]};
        x1 = f32x4{s[16 * CS], s[17 * CS], s[18 * CS], s[19 * CS]};
      }
      float most = 0.f, z = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        z = fmaf(x1[q], 0.f, fmaf(x0[q], 0.f, z));
        most = fmaxf(most, fmaxf(fabsf(x0[q]), fabsf(x1[q])));
      }
      Split3 s3;
      if (__any(z != 0.f || most > 0x1p126f)) s3 = rec_split8_any(x0, x1);
      else s3 = rec_split8(x0, x1);
      uint4* dst = reinterpret_cast<uint4*>(frag + (is_c ? 0 : 3 * L * NP / 2)) + it;
#pragma unroll
      for (int p = 0; p < 3; ++p) dst[p * (L * NP / 8)] = s3.p[p].u;
    }
  } else {
    for (int i = lays ? tid : L * NP; i < L * NP / 4; i += 256) {  // C: tile (tokens, rows of S)
      const int tile = i >> 6, ln = i & 63, rt = tile / (NP / 16), ct = tile % (NP / 16);
      *reinterpret_cast<float4*>(frag + 4 * i) = *reinterpret_cast<const float4*>(c_l + (16 * rt + (ln & 15)) * CS + 16 * ct + 4 * (ln >> 4));
    }
    for (int i = lays ? tid : L * NP; i < L * NP / 4; i += 256) {  // B^T: tile (rows of S, tokens)
      const int tile = i >> 6, ln = i & 63, rt = tile >> 1, ct = tile & 1;
      const float* s = b_l + (16 * ct + 4 * (ln >> 4)) * CS + 16 * rt + (ln & 15);
      *reinterpret_cast<float4*>(frag + L * NP + 4 * i) = float4{s[0], s[CS], s[2 * CS], s[3 * CS]};
    }
  }
  // C B^T, a 16 x 16 tile a wave; k runs 16 at a time, lane group kq takes k = 4 kq .. 4 kq + 3 in four steps (both operands alike)
  {
    const int lane = tid & 63, r16 = lane & 15, kq = lane >> 4, i0 = (tid >> 7) * 16, j0 = ((tid >> 6) & 1) * 16;
    f32x4 acc = {};
#pragma unroll 4
    for (int k = 0; k < NP; k += 16) {
      const f32x4 av = *reinterpret_cast<const f32x4*>(c_l + (i0 + r16) * CS + k + 4 * kq);
      const f32x4 bv = *reinterpret_cast<const f32x4*>(b_l + (j0 + r16) * CS + k + 4 * kq);
#pragma unroll
      for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[s], bv[s], acc, 0, 0, 0);
    }
    __syncthreads();                                              // (C and B have been read)
#pragma unroll
    for (int r = 0; r < 4; ++r) cb_l[(i0 + 4 * kq + r) * PS + j0 + r16] = acc[r];
  }
  __syncthreads();
  double* cum = cum_l + hw * L;
  for (int hh = blockIdx.z * 8 + hw; hh < per; hh += 8 * gridDim.z) {
    const int h = g * per + hh;
    if (hh != (int)blockIdx.z * 8 + hw) fetch_gates(hh);
    const float dt = t < cnt ? ssm_softplus(Elem<T>::to_f(gate_dt) + gate_bias) : 0.f;
    const float la = t < cnt ? -expf(gate_log) * dt : 0.f;
    double c = (double)la * 1.4426950408889634;
#pragma unroll
    for (int o = 1; o < L; o <<= 1) {
      const double v = __shfl_up(c, o, L);
      if (t >= o) c += v;
    }
    const double last = __shfl(c, L - 1, L);
    cum[t] = c;
    dt_l[hw * L + t] = dt;
    float* hp = a.frags + (int64_t)gridDim.x * a.G * ssm_frag_elems(NP) + ((int64_t)blockIdx.x * a.H + h) * kSsmHead;
    const float eb = rec_exp2(c), wt = rec_exp2(last - c) * dt, dec = expf(la);
    // (a weight beyond 2^8 with B and x of up to 2^59: the pieces of a sum that leaves 32 bits would leave it with either sign)
    bool no = !rec_finite(dt) || !rec_moderate_decay(la) || !(wt <= 0x1p8f) || !rec_finite(eb) || !rec_finite(dec);
    hp[768 + L + t] = wt;
    hp[768 + 2 * L + t] = dt;
    hp[768 + 3 * L + t] = dec;
    __builtin_amdgcn_wave_barrier();
    // the weighted C B^T, 16 bytes a lane: piece i of 192 is lane i % 64 of tile i / 64
#pragma unroll
    for (int u = 0; u < 6; ++u) {
      const int i = u * 32 + t, tile = i >> 6, ln = i & 63, row = (tile ? 16 : 0) + (ln & 15), col = (tile == 2 ? 16 : 0) + 4 * (ln >> 4);
      const double bt = cum[row];
      const f32x4 cb = *reinterpret_cast<const f32x4*>(cb_l + row * PS + col), ds = *reinterpret_cast<const f32x4*>(dt_l + hw * L + col);
      f32x4 m;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float x = cb[v] * (rec_exp2(bt - cum[col + v]) * ds[v]);
        m[v] = col + v <= row ? x : 0.f;
        no |= !rec_finite(m[v]);
      }
      *reinterpret_cast<f32x4*>(hp + 4 * i) = m;
    }
    hp[768 + t] = rec_flagged(eb, no);
    __builtin_amdgcn_wave_barrier();
  }
}

// The chunks of a request in turn, a workgroup of eight waves per (request, head, 16 CB columns of S), two or four waves per 16 columns.  A wave
// has its part of the rows of S in accumulators: lane (r16, kq) holds rows 16 t + 4 kq + r of column r16, two tiles of which are the
// right-hand operand of a product over 32 rows (split on the way), so S goes from one chunk's sum into the next one's product without leaving
// its registers.  The parts of C S are added across these waves in LDS, two of which finish 16 of the tokens each; two also convolve these
// tokens' x from raw inputs in LDS of their own and hand x and the pieces of U = e^(b_last - b_t) dt_t x over: x is not written to memory.
// Four waves per 16 columns halve what a wave does for a chunk: for launches that leave CUs without work at 64 columns a workgroup (a CU
// holds one of theirs, not two: everything is fetched a whole chunk ahead, 2.9 -> 2.6 us a chunk, 3.3 at 64 columns).  128 heads of 128 x 64
// over 8, whole call: 1 request of 5083 rows 611 -> 456 us, of 1000 137 -> 106; with the silus of a lane's four tokens side by side and D in one sum 434
// (4 of 1900 rows, 64 columns a workgroup: within 1 %).
template <typename T, int NP, int CB>
__global__ void __launch_bounds__(512, CB == 4 ? 4 : 2) ssm_chunk_walk_kernel(SsmArgs a, int64_t max_chunks) {
  constexpr int PARTS = 8 / CB;                                 // waves that share 16 columns
  constexpr bool AHEAD = PARTS > 2;                             // everything is fetched a whole chunk ahead (half of one: two workgroups a CU cover each other's waits)
  constexpr int L = kRecChunk, NT = NP / 16, HT = NT / PARTS, HALO = kRecHalo;  // HT: 16-row tiles of S a wave
  static_assert(HT % 2 == 0, "two tiles are an operand");
  constexpr int PB = L * NP * 2, ALL = 3 * PB / 16, PIECES = (ALL + 511) / 512;  // bytes of a plane; 16-byte pieces of three, a thread's
  using Tile = RowTile<T, 16>;
  constexpr int OWN = Tile::kElems * (int)sizeof(T) > 16 * kOutStride * 4 ? Tile::kElems * (int)sizeof(T) : 16 * kOutStride * 4;
  __shared__ __attribute__((aligned(16))) uint8_t c_l[3 * PB], b_l[3 * PB];     // C and B^T of the chunk, as laid down
  __shared__ __attribute__((aligned(16))) uint8_t u_l[CB][3][1024];             // U of the chunk: [columns][piece][lane][16]; token by token x
  __shared__ __attribute__((aligned(16))) uint8_t x_l[CB][PARTS / 2][1024];             // x of its tokens 0 .. 15, for the waves of 16 .. 31 (four waves: of all tokens)
  __shared__ __attribute__((aligned(16))) uint8_t own_l[8][OWN];                // by turns a wave's half sum of C S, raw inputs, results on their way out
  __shared__ __attribute__((aligned(16))) uint8_t sum_l[PARTS == 2 ? 1 : 8][2][PARTS == 2 ? 16 : 1024];     // four waves: their parts of C S
  __shared__ int serial_l[2];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, kq = lane >> 4;
  // of four waves the first two make x and U, the others finish the results, either of 16 tokens; of two each does both
  const int cw = w % CB, part = w / CB, half = part & 1;
  const bool makes_x = PARTS == 2 || part < 2, ends = PARTS == 2 || part >= 2;
  // workgroups of one (request, group) read the same operands: they go to one XCD (workgroup ids go round the 8 XCDs)
  const int H = a.H, G = a.G, N = a.N, E = a.E, taps = a.taps, per = H / G;
  const int eblocks = (E + 16 * CB - 1) / (16 * CB), members = per * eblocks;
  const RecPlace at = rec_place((int)a.batch * G, members);
  if (at.unit < 0) return;
  const int member = at.member, g = at.unit % G, b = rec_by_length(a.q_len, (int)a.batch, at.unit / G, rec_first_requests((int)a.batch, G * members));
  const int64_t first_pos = a.seq_lens[b] - a.q_len[b], t0 = a.q_start[b];
  const int n = a.q_len[b];
  if (n <= 0 || first_pos < 0) return;
  const int64_t chunk0 = __builtin_amdgcn_readfirstlane((int)rec_chunks_before(a.q_len, b));
  if (chunk0 + (n + L - 1) / L > max_chunks) return;          // (requests that share rows: more rows than the launch has)
  const int h = g * per + member / eblocks;
  const int e0 = member % eblocks * (16 * CB) + 16 * cw, e = e0 + r16;
  const bool on = e0 < E;                                        // (waves without columns take their part of the staging)
  const bool e_ok = e < E, wide = e0 + 16 <= E;
  const int C = H * E + 2 * G * N;
  const int64_t slot = a.state_indices[b];
  float* st = a.state + slot * a.state_ld + (int64_t)h * N * E + e;
  const int row0 = part * (NP / PARTS) + 4 * kq;                 // this lane's rows of S: row0 + 16 t + r
  f32x4 S[HT];
#pragma unroll
  for (int t = 0; t < HT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) S[t][r] = (first_pos > 0 && e_ok && row0 + 16 * t + r < N) ? st[(row0 + 16 * t + r) * E] : 0.f;
  float wt[kRecTaps];
#pragma unroll
  for (int i = 0; i < kRecTaps; ++i) wt[i] = (i < taps && e_ok) ? Elem<T>::to_f(((const T*)a.conv_w)[(int64_t)(h * E + e) * taps + taps - 1 - i]) : 0.f;
  const float bias = (a.conv_b && e_ok) ? Elem<T>::to_f(((const T*)a.conv_b)[h * E + e]) : 0.f;
  const float dskip = a.d_skip ? a.d_skip[h] : 0.f;
  const int64_t frag_ld = (int64_t)G * ssm_frag_elems(NP), head_ld = (int64_t)H * kSsmHead;
  const float* f = a.frags + chunk0 * frag_ld + g * ssm_frag_elems(NP);
  const float* fh = a.frags + max_chunks * frag_ld + (chunk0 * H + h) * kSsmHead;
  const T* p = (const T*)a.p + t0 * a.ld + a.x_off + h * E + e0;
  float* yo = a.work + t0 * a.wld + h * E + e0;
  // 16-byte pieces of the projection's and of the result's rows: everything starts on one
  const bool vec = wide && ((reinterpret_cast<uintptr_t>(p) | (uintptr_t)(a.ld * sizeof(T))) & 15) == 0 &&
                   ((reinterpret_cast<uintptr_t>(yo) | (uintptr_t)(a.wld * 4)) & 15) == 0 && a.ld < (1 << 24) && a.wld < (1 << 24);

  // raw inputs of the convolution, tokens 16 half - HALO .. 16 half + 15 of the chunk at l0 > 0
  Tile tile;
  auto fetch_x = [&](int l0) {
    int ln = lane;
    asm volatile("" : "+v"(ln));                                 // (addresses made where they are used, not held over the loop)
    if (vec && makes_x) tile.fetch_clamped(p, a.ld, l0 + 16 * half, n, ln);
  };
  // x of this lane's tokens 16 half + 4 kq + s, zero behind the portion; taps that the layer does not have see zeros
  auto convolve = [&](const float (&raw)[HALO + 4], int cnt, f32x4& x, bool& bad) {
    f32x4 y;
#pragma unroll
    for (int s = 0; s < 4; ++s) y[s] = bias + wt[0] * raw[s + HALO];
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
    if constexpr (PARTS > 2) {
      // side by side, also of rows that there are not: behind a branch each, as they are left alone, every token waits for its own exponential
      // and quotient (two workgroups a CU have each other for that, and no registers for it: the walk of 4 of 1900 rows 345 -> 385 us)
      float z[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) z[s] = rec_silu(y[s]);
      asm volatile("" : "+v"(z[0]), "+v"(z[1]), "+v"(z[2]), "+v"(z[3]));
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const bool in = 16 * half + 4 * kq + s < cnt, large = !rec_moderate(y[s]);
        x[s] = in ? (large ? y[s] : z[s]) : 0.f;                 // (one that is not moderate: see `serial`)
        bad |= in & large;
      }
    } else {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const float z = rec_silu(y[s]);
        const bool in = 16 * half + 4 * kq + s < cnt;
        x[s] = in ? (rec_moderate(y[s]) ? z : y[s]) : 0.f;
        bad |= in && !rec_moderate(y[s]);
      }
    }
  };
  // x and U = e^(b_last - b_t) dt_t x to where both waves of these columns find them
  auto hand_over = [&](const f32x4& x, const f32x4& wv) {
    if (PARTS > 2 || half == 0) *reinterpret_cast<f32x4*>(&x_l[cw][PARTS > 2 ? half : 0][16 * lane]) = x;
    uint2 u[3];
    rec_split2(x[0] * wv[0], x[1] * wv[1], u[0].x, u[1].x, u[2].x);
    rec_split2(x[2] * wv[2], x[3] * wv[3], u[0].y, u[1].y, u[2].y);
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<uint2*>(&u_l[cw][i][16 * lane + 8 * half]) = u[i];
  };
  u32x4 stage[PIECES], stage_b[AHEAD ? PIECES : 1];
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
  f32x4 x = {};
  bool bad = false;
  fetch(f, stage);
  if constexpr (AHEAD) fetch(f + 3 * L * NP / 2, stage_b);
  f32x4 head[3];
  float flag_next = 0.f, keep_next = 0.f;
  auto fetch_head = [&](const float* fh, f32x4* to) __attribute__((always_inline)) {      // row tile `half` of the weighted C B^T, weights of this lane's tokens
    to[0] = *reinterpret_cast<const f32x4*>(fh + 256 * half + 4 * lane);
    to[1] = *reinterpret_cast<const f32x4*>(fh + 512 * half + 4 * lane);
    to[2] = *reinterpret_cast<const f32x4*>(fh + 768 + 16 * half + 4 * kq);
  };
  if constexpr (AHEAD) {
    fetch_head(fh, head);
    flag_next = f[3 * L * NP], keep_next = fh[768 + L - 1];
  }
  if (makes_x) {
    float in[HALO + 4];
#pragma unroll
    for (int i = 0; i < HALO + 4; ++i) {
      const int l = 16 * half + 4 * kq + i - HALO;
      in[i] = 0.f;
      if (e_ok && l < n) {
        if (l >= 0) in[i] = Elem<T>::to_f(p[(int64_t)l * a.ld + r16]);
        else if (first_pos > 0 && taps - 1 + l >= 0) in[i] = a.conv_state[slot * a.conv_ld + (int64_t)(taps - 1 + l) * C + h * E + e];
      }
    }
    convolve(in, n, x, bad);
    hand_over(x, *reinterpret_cast<const f32x4*>(fh + 768 + L + 16 * half + 4 * kq));
  }
  place(c_l, stage);
  if (tid < 2) serial_l[tid] = 0;
  if (L < n) fetch_x(L);
  __syncthreads();

  // Two steps a chunk, what the next one needs on its way into registers during each: C S while B^T comes, then the products inside the
  // chunk and the new S while the next chunk's C comes.
  for (int l0 = 0; l0 < n; l0 += L) {
    const int cnt = n - l0 < L ? n - l0 : L, turn = (l0 / L) & 1;
    const bool more = l0 + L < n;
    const float* fn = f + (more ? frag_ld : 0);                 // (the last chunk fetches itself again)
    const float* fhn = fh + (more ? head_ld : 0);
    float* yr = yo + (int64_t)(l0 + 16 * half) * a.wld;
    fetch(AHEAD ? fn : f + 3 * L * NP / 2, stage);
    const float flag = AHEAD ? flag_next : f[3 * L * NP], keep = AHEAD ? keep_next : fh[768 + L - 1];
    if constexpr (AHEAD) flag_next = fn[3 * L * NP], keep_next = fhn[768 + L - 1];
    f32x4 M[2] = {}, eb = {}, wv = {};
    if constexpr (AHEAD) M[0] = head[0], M[1] = head[1], eb = head[2];
    f32x4 O = {};
    bool serial = false;
    if (on) {
      f32x4 P[2] = {}, Ps[2] = {};
#pragma unroll
      for (int u = 0; u < HT / 2; ++u) {
        const Split3 s = rec_split8(S[2 * u], S[2 * u + 1]);
        Frag16 c[2][3];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int q = 0; q < 3; ++q) c[i][q].u = *reinterpret_cast<const uint4*>(c_l + q * PB + (i * (NT / 2) + part * (HT / 2) + u) * 1024 + lane * 16);
        rec_mma<2>(c, s, P, Ps);
      }
      if constexpr (!AHEAD) {
        f32x4 of[3];
        fetch_head(fh, of);
        M[0] = of[0], M[1] = of[1], eb = of[2];
      }
      wv = *reinterpret_cast<const f32x4*>(fhn + 768 + L + 16 * half + 4 * kq);
      float z = 0.f, top = 0.f;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        P[i] += Ps[i];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          z = fmaf(P[i][r], 0.f, z);
          top = fmaxf(top, fabsf(P[i][r]));
        }
      }
      O = half ? P[1] : P[0];
      if constexpr (PARTS == 2) {
        *reinterpret_cast<f32x4*>(&own_l[w ^ 4][16 * lane]) = half ? P[0] : P[1];
      } else {
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (!ends || half != i) *reinterpret_cast<f32x4*>(&sum_l[w][i][16 * lane]) = P[i];
      }
      // An infinity or a NaN in the chunk, or one that sums of large values end in, would reach the tokens in front of it through a product
      // with a weight of zero, and so would a product of a large S with rows behind a step that resets it: the workgroup takes such a
      // chunk token by token, from S in the state row and x in LDS (a rare path: it must not set the kernel's registers)
      const bool off = z != 0.f || top > 0x1p126f;
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
    }
    place(b_l, AHEAD ? stage_b : stage);
    Split3 U;
#pragma unroll
    for (int i = 0; i < 3; ++i) U.p[i].u = *reinterpret_cast<const uint4*>(&u_l[cw][i][16 * lane]);
    const f32x4 x0 = *reinterpret_cast<const f32x4*>(&x_l[cw][0][16 * lane]);
    if constexpr (PARTS > 2) {
      if (ends) x = half ? *reinterpret_cast<const f32x4*>(&x_l[cw][PARTS / 2 - 1][16 * lane]) : x0;
    }
    __syncthreads();
    if constexpr (AHEAD) fetch(fn + 3 * L * NP / 2, stage_b);
    else fetch(fn, stage);
    serial = __builtin_amdgcn_readfirstlane(serial_l[turn]) != 0;
    if (tid == 0) serial_l[turn ^ 1] = 0;
    if (!serial) {
      if (on) {
        if (ends) {
          if constexpr (PARTS == 2) O += *reinterpret_cast<const f32x4*>(&own_l[w][16 * lane]);
          else O = (O + *reinterpret_cast<const f32x4*>(&sum_l[w ^ CB][half][16 * lane])) +
                   (*reinterpret_cast<const f32x4*>(&sum_l[w ^ (2 * CB)][half][16 * lane]) + *reinterpret_cast<const f32x4*>(&sum_l[w ^ (3 * CB)][half][16 * lane]));
          O *= eb;
          // (a row tile of the weights is at most two products of four columns for each of its rows: as they are, in fp32)
          if (half == 0) {
#pragma unroll
            for (int s = 0; s < 4; ++s) O = __builtin_amdgcn_mfma_f32_16x16x4f32(M[0][s], x[s], O, 0, 0, 0);
          } else {
            f32x4 O1 = {};
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              O = __builtin_amdgcn_mfma_f32_16x16x4f32(M[0][s], x0[s], O, 0, 0, 0);
              O1 = __builtin_amdgcn_mfma_f32_16x16x4f32(M[1][s], x[s], O1, 0, 0, 0);
            }
            O += O1;
          }
        }
#pragma unroll
        for (int t = 0; t < HT; t += 2) {
          Frag16 bt[2][3];
#pragma unroll
          for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int q = 0; q < 3; ++q) bt[i][q].u = *reinterpret_cast<const uint4*>(b_l + q * PB + (part * HT + t + i) * 1024 + lane * 16);
          }
          f32x4 D[2] = {};
          rec_mma_small<2>(bt, U, D);
          rec_mma_big<2>(bt, U, D);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[t + i][r] = fmaf(S[t + i][r], keep, D[i][r]);
        }
        O += dskip * x;
      }
    } else {
      int rows = N, step = E;
      asm volatile("" : "+s"(rows), "+s"(step));                 // (no addresses of 16 rows held over the loop)
      int ln = lane;
      asm volatile("" : "+v"(ln));
      const int r16 = ln & 15, kq = ln >> 4, row0 = part * (NP / PARTS) + 4 * kq, e = e0 + r16;
      const bool e_ok = e < E;
      float* st = a.state + slot * a.state_ld + (int64_t)h * N * E + e;
      float* xs = reinterpret_cast<float*>(u_l[0][0]) + 16 * cw + r16;           // x [32][16 CB]
      if (makes_x)
#pragma unroll
        for (int s = 0; s < 4; ++s) xs[(16 * half + 4 * kq + s) * (16 * CB)] = rec_silu_if_large(x[s]);
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
          const float xv = xs[t * (16 * CB)], dt = fh[768 + 2 * L + t], dec = fh[768 + 3 * L + t], dx = dt * xv;
          // row t of C: this lane group's four of every 16; column t of B^T
          const uint16_t* cr = reinterpret_cast<const uint16_t*>(f) + (t >> 4) * (NT / 2) * 512 + 8 * (16 * kq + (t & 15));
          const uint16_t* br = reinterpret_cast<const uint16_t*>(f) + 3 * L * NP + 8 * (16 * ((t & 15) >> 2) + 4 * kq) + (t & 3) + 4 * (t >> 4);
          float y = 0.f;
#pragma unroll 1
          for (int u = 0; u < 4 * NT; ++u) {
            const int row = 16 * (u >> 2) + 4 * kq + (u & 3);
            if (row < rows && e_ok) {
              const float v = dec * st[row * step] + rec_joined(br + (u >> 2) * 512 + 8 * (u & 3), L * NP) * dx;
              st[row * step] = v;
              y += v * rec_joined(cr + (u >> 3) * 512 + (u & 3) + (u & 4), L * NP);
            }
          }
          y += __shfl_xor(y, 16, 64);
          y += __shfl_xor(y, 32, 64);
          if (kq == 0 && e_ok) yr[(int64_t)t * a.wld + r16] = y + dskip * xv;
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
    // the next chunk's x
    f32x4 xn = {};
    bad = false;
    if (more && makes_x) {
      T* raw = reinterpret_cast<T*>(own_l[w]);
      if (vec) {
        int ln = lane;
        asm volatile("" : "+v"(ln));
        tile.place(raw, ln);
      } else {                                                   // (rows or columns that start off a 16-byte boundary: not fetched ahead)
        const int first = l0 + L + 16 * half - HALO;
        int ln = lane;
        asm volatile("" : "+v"(ln));
        const int r16 = ln & 15, kq = ln >> 4;
        const bool e_ok = e0 + r16 < E;
        for (int r = kq; r < 16 + HALO; r += 4) raw[r * Tile::kStride + r16] = e_ok && first + r < n ? p[(int64_t)(first + r) * a.ld + r16] : Elem<T>::from_f(0.f);
      }
      __builtin_amdgcn_wave_barrier();
      float in[HALO + 4];
#pragma unroll
      for (int i = 0; i < HALO + 4; ++i) in[i] = Elem<T>::to_f(raw[(4 * kq + i) * Tile::kStride + r16]);
      convolve(in, n - l0 - L, xn, bad);
      hand_over(xn, wv);
    }
    if constexpr (AHEAD) fetch_head(fhn, head);
    place(c_l, stage);
    // behind the wait for the pieces (memory answers in order), so that it is the next one's: results out, raw inputs in
    if (!serial && ends) {
      __builtin_amdgcn_wave_barrier();
      float* ol = reinterpret_cast<float*>(own_l[w]);
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
        const int r16 = ln & 15, kq = ln >> 4;
#pragma unroll 1
        for (int row = kq; row < 16 && 16 * half + row < cnt; row += 4) yr[(int64_t)row * a.wld + r16] = ol[row * kOutStride + r16];
      }
    }
    if (l0 + 2 * L < n) fetch_x(l0 + 2 * L);
    x = xn;
    f = fn;
    fh = fhn;
    __syncthreads();
  }
  int rows = N, step = E;
  asm volatile("" : "+s"(rows), "+s"(step));                     // (no addresses of 16 rows held over the loop)
  if (e_ok)
#pragma unroll
    for (int t = 0; t < HT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (row0 + 16 * t + r < rows) st[(row0 + 16 * t + r) * step] = S[t][r];
}

// A state of up to 64 rows and long requests that have a CU each: operands of fp32, the chunks of a request in turn, a wave per (request, head, 16
// columns of S) with nothing shared: four waves a workgroup for the sake of their common loads.  S [64 x 16] stays in accumulators: lane (r16,
// kq) holds rows 16 t + 4 kq + r of column r16, which is also how a wave holds the right-hand operand of a product over the rows, and so
// do the chunk's x (lane: tokens 16 j + 4 kq + s of its column), convolved in their place from raw inputs in the wave's own LDS.  Left-hand
// operands come straight into registers in the order they are used, B^T of a chunk into the registers its C was read from, the next
// chunk's C into those of B^T; there are no barriers.  Half the products of 128 rows leave the two barriers and the exchange of
// ssm_chunk_walk_kernel nothing to cover them with (see ssm_small_walk for the figures).
template <typename T>
__global__ void __launch_bounds__(256, 2) ssm_chunk_walk_small_kernel(SsmArgs a, int64_t max_chunks) {
  constexpr int NP = 64, L = kRecChunk, NT = NP / 16, HALO = kRecHalo;
  __shared__ __attribute__((aligned(16))) T in_l[4][RowTile<T>::kElems];       // a wave's own: raw inputs of its convolution
  __shared__ __attribute__((aligned(16))) float o_l[4][L * kOutStride];         // ... results on their way out (token by token: its x)
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, r16 = lane & 15, kq = lane >> 4;
  // workgroups of one (request, group) read the same operands: they go to one XCD (workgroup ids go round the 8 XCDs)
  const int H = a.H, G = a.G, N = a.N, E = a.E, taps = a.taps, per = H / G;
  const int eblocks = (E + 63) / 64, members = per * eblocks;
  const RecPlace at = rec_place((int)a.batch * G, members);
  if (at.unit < 0) return;
  const int member = at.member, b = at.unit / G, g = at.unit % G;
  const int64_t first_pos = a.seq_lens[b] - a.q_len[b], t0 = a.q_start[b];
  const int n = a.q_len[b];
  if (n <= 0 || first_pos < 0) return;
  const int64_t chunk0 = rec_chunks_before(a.q_len, b);
  if (chunk0 + (n + L - 1) / L > max_chunks) return;          // (requests that share rows: more rows than the launch has)
  const int h = g * per + member / eblocks;
  const int e0 = member % eblocks * 64 + 16 * w, e = e0 + r16;
  if (e0 >= E) return;
  const bool e_ok = e < E, wide = e0 + 16 <= E;
  const int C = H * E + 2 * G * N;
  const int64_t slot = a.state_indices[b];
  float* st = a.state + slot * a.state_ld + (int64_t)h * N * E + e;
  f32x4 S[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * t + 4 * kq + r;
      S[t][r] = (first_pos > 0 && e_ok && row < N) ? st[row * E] : 0.f;
    }
  float wt[kRecTaps];
#pragma unroll
  for (int i = 0; i < kRecTaps; ++i) wt[i] = (i < taps && e_ok) ? Elem<T>::to_f(((const T*)a.conv_w)[(int64_t)(h * E + e) * taps + taps - 1 - i]) : 0.f;
  const float bias = (a.conv_b && e_ok) ? Elem<T>::to_f(((const T*)a.conv_b)[h * E + e]) : 0.f;
  const float dskip = a.d_skip ? a.d_skip[h] : 0.f;
  const int64_t frag_ld = (int64_t)G * ssm_frag_elems(NP), head_ld = (int64_t)H * kSsmHead;
  const float* f = a.frags + chunk0 * frag_ld + g * ssm_frag_elems(NP) + 4 * lane;
  const float* fh = a.frags + max_chunks * frag_ld + (chunk0 * H + h) * kSsmHead;
  const T* p = (const T*)a.p + t0 * a.ld + a.x_off + h * E + e0;
  float* yo = a.work + t0 * a.wld + h * E + e0;
  // 16-byte pieces of the projection's and of the result's rows: everything starts on one
  const bool vec = wide && ((reinterpret_cast<uintptr_t>(p) | (uintptr_t)(a.ld * sizeof(T))) & 15) == 0 &&
                   ((reinterpret_cast<uintptr_t>(yo) | (uintptr_t)(a.wld * 4)) & 15) == 0;

  // raw inputs of the convolution, tokens 16 j + 4 kq - HALO + i of the chunk at l0 > 0
  RowTile<T> tile;
  auto fetch_x = [&](int l0) { if (vec) tile.fetch(p, a.ld, l0, n, lane); };
  // x of this lane's tokens, zero behind the portion; taps that the layer does not have see zeros
  auto convolve = [&](const float (&raw)[2][HALO + 4], int cnt, f32x4 (&x)[2], bool& bad) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        float y = bias + wt[0] * raw[j][s + HALO];
#pragma unroll
        for (int i = 1; i < kRecTaps; ++i) y += wt[i] * __int_as_float(__float_as_int(raw[j][s + HALO - i]) & (i < taps ? -1 : 0));
        float z = rec_silu(y);
        asm volatile("" : "+v"(z));                              // (straight-line code: it goes between the products)
        const bool in = 16 * j + 4 * kq + s < cnt;
        x[j][s] = in ? (rec_moderate(y) ? z : y) : 0.f;       // (one that is not: see `serial`)
        bad |= in && !rec_moderate(y);
      }
  };
  f32x4 x[2];
  bool bad = false;
  {
    float in[2][HALO + 4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int i = 0; i < HALO + 4; ++i) {
        const int l = 16 * j + 4 * kq + i - HALO;
        in[j][i] = 0.f;
        if (e_ok && l < n) {
          if (l >= 0) in[j][i] = Elem<T>::to_f(p[(int64_t)l * a.ld + r16]);
          else if (first_pos > 0 && taps - 1 + l >= 0) in[j][i] = a.conv_state[slot * a.conv_ld + (int64_t)(taps - 1 + l) * C + h * E + e];
        }
      }
    convolve(in, n, x, bad);
  }
  f32x4 A[2 * NT], M[3], eb[2], wv[2];
  float flag;
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) A[i] = *reinterpret_cast<const f32x4*>(f + 256 * i);
  flag = f[3 * L * NP - 4 * lane];
#pragma unroll
  for (int i = 0; i < 3; ++i) M[i] = *reinterpret_cast<const f32x4*>(fh + 256 * i + 4 * lane);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    eb[i] = *reinterpret_cast<const f32x4*>(fh + 768 + 16 * i + 4 * kq);
    wv[i] = *reinterpret_cast<const f32x4*>(fh + 768 + L + 16 * i + 4 * kq);
  }
  if (L < n) fetch_x(L);

  for (int l0 = 0; l0 < n; l0 += L) {
    const int cnt = n - l0 < L ? n - l0 : L;
    const bool more = l0 + L < n;
    const float* fn = f + (more ? frag_ld : 0);                 // (the last chunk fetches itself again)
    const float* fhn = fh + (more ? head_ld : 0);
    float* yr = yo + (int64_t)l0 * a.wld;
    // An infinity or a NaN in the chunk, or one that sums of large values end in, would reach the tokens in front of it through a product
    // with a weight of zero, and so would a product of a large S with rows behind a step that resets it: the wave takes such a chunk
    // token by token behind the products, which then count for nothing, from S in the state row and x in LDS (a rare path: it must
    // not set the kernel's registers)
    const bool flagged = bad || flag != 0.f;
    int rows = N, step = E;
    asm volatile("" : "+s"(rows), "+s"(step));
    bool serial;
    f32x4 xn[2];
    {
      const float keep = __shfl(eb[1][3], 63, 64);
      f32x4 O[2] = {};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i) O[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[i * NT + t][s], S[t][s], O[i], 0, 0, 0);
      // the next chunk's x between the products: a product keeps the matrix pipe for 32 cycles, in which a few of these fit
      bad = false;
      {
        float in[2][HALO + 4];
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
          for (int i = 0; i < HALO + 4; ++i) in[j][i] = Elem<T>::to_f(in_l[w][(16 * j + 4 * kq + i) * RowTile<T>::kStride + r16]);
        convolve(in, n - l0 - L, xn, bad);
      }
#pragma unroll
      for (int i = 0; i < 2 * NT; ++i) A[i] = *reinterpret_cast<const f32x4*>(f + L * NP + 256 * i);
      flag = fn[3 * L * NP - 4 * lane];
#pragma unroll
      for (int i = 0; i < 8 * NT; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
      }
      if (l0 + 2 * L < n) fetch_x(l0 + 2 * L);
      {
        float z = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) z = fmaf(O[i / 4][i % 4], 0.f, z);
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
          for (int s = 0; s < 4; ++s) o_l[w][(16 * j + 4 * kq + s) * kOutStride + r16] = rec_silu_if_large(x[j][s]);
        if (e_ok)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              if (16 * t + 4 * kq + r < rows) st[(16 * t + 4 * kq + r) * step] = S[t][r];
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) O[i] *= eb[i];
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i) O[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(M[i][s], x[0][s], O[i], 0, 0, 0);
#pragma unroll
      for (int s = 0; s < 4; ++s) O[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(M[2][s], x[1][s], O[1], 0, 0, 0);
      f32x4 U[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        O[i] += dskip * x[i];
        U[i] = x[i] * wv[i];
      }
#pragma unroll
      for (int i = 0; i < 3; ++i) M[i] = *reinterpret_cast<const f32x4*>(fhn + 256 * i + 4 * lane);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        eb[i] = *reinterpret_cast<const f32x4*>(fhn + 768 + 16 * i + 4 * kq);
        wv[i] = *reinterpret_cast<const f32x4*>(fhn + 768 + L + 16 * i + 4 * kq);
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
      for (int t = 0; t < NT; t += 2) {
        f32x4 D[2][2] = {};                                      // (tokens 0 .. 15 and 16 .. 31; added to S as a whole: a rounding of S a chunk)
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int k = 0; k < 2; ++k)
#pragma unroll
            for (int i = 0; i < 2; ++i) D[k][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[2 * (t + i) + k][s], U[k][s], D[k][i], 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int r = 0; r < 4; ++r) S[t + i][r] = fmaf(S[t + i][r], keep, D[0][i][r] + D[1][i][r]);
      }
#pragma unroll
      for (int i = 0; i < 2 * NT; ++i) A[i] = *reinterpret_cast<const f32x4*>(fn + 256 * i);
    }
    if (serial) {
#pragma unroll 1
      for (int t = 0; t < cnt; ++t) {
        const float xv = o_l[w][t * kOutStride + r16], dt = fh[768 + 2 * L + t], dec = fh[768 + 3 * L + t], dx = dt * xv;
        const float* cr = f - 4 * lane + (t >> 4) * NT * 256 + 4 * (16 * kq + (t & 15));           // row t of C: this lane group's four of every 16
        const float* br = f - 4 * lane + L * NP + (t >> 4) * 256 + 4 * (16 * ((t & 15) >> 2) + 4 * kq) + (t & 3);     // column t of B^T
        float y = 0.f;
#pragma unroll 1
        for (int u = 0; u < 4 * NT; ++u) {
          const int row = 16 * (u >> 2) + 4 * kq + (u & 3);
          if (row < rows && e_ok) {
            const float v = dec * st[row * step] + br[(u >> 2) * 512 + 4 * (u & 3)] * dx;
            st[row * step] = v;
            y += v * cr[(u >> 2) * 256 + (u & 3)];
          }
        }
        y += __shfl_xor(y, 16, 64);
        y += __shfl_xor(y, 32, 64);
        if (kq == 0 && e_ok) yr[(int64_t)t * a.wld + r16] = y + dskip * xv;
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          S[t][r] = e_ok && 16 * t + 4 * kq + r < rows ? st[(16 * t + 4 * kq + r) * step] : 0.f;
      __builtin_amdgcn_sched_barrier(0);
    }
    x[0] = xn[0];
    x[1] = xn[1];
    f = fn;
    fh = fhn;
  }
  int rows = N, step = E;
  asm volatile("" : "+s"(rows), "+s"(step));                     // (no addresses of 32 rows held over the loop)
  if (e_ok)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (16 * t + 4 * kq + r < rows) st[(16 * t + 4 * kq + r) * step] = S[t][r];
}

// gate, grouped norm, weight, one pass: a workgroup per (token, norm group), the group's elements in registers, 16-byte accesses
// (8 elements a piece, at most kPostPieces pieces a thread).  Bound by HBM: 7262 x 8192 169 us (two passes, 2- and 4-byte accesses) ->
// 86 = 5.5 TB/s; 32 rows 28 -> 7 us.
constexpr int kPostPieces = 4;
template <typename T>
__global__ void __launch_bounds__(256) ssm_post_vec_kernel(SsmArgs a, int conv_blocks) {
  __shared__ float red[16];
  // the first workgroups move the convolution's inputs on, 256 channels of a request each: the others neither read nor write them (a
  // launch of its own is 2.5 us; whole call with / without it: 128 heads of 128 x 64, 8 requests of one token 25.7 / 22.9 us, 32 of them
  // 65.8 / 62.5, on state rows that no cache holds 77 / 74)
  if ((int)blockIdx.x < conv_blocks) {
    const int per = (a.H * a.E + 2 * a.G * a.N + 255) / 256;
    if (blockIdx.y == 0) ssm_conv_state<T>(a, blockIdx.x / per, blockIdx.x % per * 256 + threadIdx.x);
    return;
  }
  const int gs = a.H * a.E / a.norm_groups;
  const int64_t t = blockIdx.x - conv_blocks, c0 = (int64_t)blockIdx.y * gs;
  const float* yr = a.work + t * a.wld + c0;
  const T* z = (const T*)a.p + t * a.ld + a.z_off + c0;
  float v[kPostPieces][8], sq = 0.f;
#pragma unroll
  for (int u = 0; u < kPostPieces; ++u) {
    const int c = 8 * (u * 256 + (int)threadIdx.x);
    if (c >= gs) break;
    const float4 y0 = *reinterpret_cast<const float4*>(yr + c), y1 = *reinterpret_cast<const float4*>(yr + c + 4);
    const float yy[8] = {y0.x, y0.y, y0.z, y0.w, y1.x, y1.y, y1.z, y1.w};
    const Vec16<T> zv = load16(z + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[u][i] = yy[i] * ssm_silu(Elem<T>::to_f(zv.e[i]));
      sq += v[u][i] * v[u][i];
    }
  }
  const float rs = 1.0f / sqrtf(block_sum(sq, red) / (float)gs + a.eps);
  T* o = (T*)a.out + t * a.out_ld + c0;
  const T* nw = (const T*)a.norm_w + c0;
#pragma unroll
  for (int u = 0; u < kPostPieces; ++u) {
    const int c = 8 * (u * 256 + (int)threadIdx.x);
    if (c >= gs) break;
    const Vec16<T> wv = load16(nw + c);
    Vec16<T> r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r.e[i] = Elem<T>::from_f(v[u][i] * rs * Elem<T>::to_f(wv.e[i]));
    store16(o + c, r);
  }
}

// ---------------------------------------------------------------------------------- gate, grouped norm, weight
template <typename T>
__device__ __forceinline__ void ssm_gate_norm_store(const SsmArgs& a, const float* y, const T* z, T* o, float* red) {
  const int inner = a.H * a.E, gs = inner / a.norm_groups;
  for (int grp = 0; grp < a.norm_groups; ++grp) {
    float sq = 0.f;
    for (int i = threadIdx.x; i < gs; i += blockDim.x) {
      const int c = grp * gs + i;
      const float v = y[c] * ssm_silu(Elem<T>::to_f(z[c]));
      sq += v * v;
    }
    const float rs = 1.0f / sqrtf(block_sum(sq, red) / (float)gs + a.eps);
    for (int i = threadIdx.x; i < gs; i += blockDim.x) {
      const int c = grp * gs + i;
      const float v = y[c] * ssm_silu(Elem<T>::to_f(z[c]));
      o[c] = Elem<T>::from_f(v * rs * Elem<T>::to_f(((const T*)a.norm_w)[c]));
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256) ssm_post_kernel(SsmArgs a) {
  __shared__ float red[16];
  const int64_t t = blockIdx.x;
  ssm_gate_norm_store<T>(a, a.work + t * a.wld, (const T*)a.p + t * a.ld + a.z_off, (T*)a.out + t * a.out_ld, red);
}

// ---------------------------------------------------------------------------------- one token per request, a state of some size
// A workgroup per (head, request): the head's x, B and C channels through the convolution into LDS, step size and decay, then S in
// 16-byte pieces, all of a thread's pieces in flight from the start: thread = four columns and every 1024 / E-th row, a step
// per piece, the read-out summed over lanes and waves.  B and C are convolved again for every head of a group (2 N channels of
// 4 taps: nothing against N E of state).  Bound by HBM, the state read and written once: 32 requests, 128 heads of 128 x 64 (268 MB):
// the recurrence's kernel for prompts, which waited for one row per lane and step of its chain, 110 us + 10 of preparation -> 50.
// With the convolution's loads in front of the state's: whole call 73.8 -> 62.0 us (64 requests 133.7 -> 115.9, 32 of 64 heads 33.9 -> 29.4;
// 5 requests 20.0 -> 19.8); behind them, tap by tap, it began when the state had arrived, a round trip a tap.
template <typename T, int NIT, bool EARLY>
__global__ void __launch_bounds__(256) ssm_step_kernel(SsmArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];       // x [E] | B [N] | C [N] | sums [4][E]
  const int h = blockIdx.x, b = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int64_t first_pos = a.seq_lens[b] - 1;
  if (first_pos < 0) return;
  const bool fresh = first_pos == 0;
  const int H = a.H, G = a.G, N = a.N, E = a.E, taps = a.taps, g = h / (H / G);
  const int inner = H * E, C = inner + 2 * G * N, quads = E / 4, rows = 256 / quads;
  const int64_t slot = a.state_indices[b];
  float* st = a.state + slot * a.state_ld + (int64_t)h * N * E;
  const int n0 = tid / quads, e = tid % quads * 4;
  const T* p = (const T*)a.p + (int64_t)b * a.ld;
  const float* cs = a.conv_state + slot * a.conv_ld;
  // Memory answers in order: what the convolution and the step size are made of is asked for in front of the state, all of it at once, and
  // their arithmetic goes on while the state is on its way.  Up to four taps (EARLY), the workgroup's first 512 channels; others one by one.
  const int channels = E + 2 * N;
  auto channel = [&](int i) { return i < E ? h * E + i : inner + (i < E + N ? g * N + (i - E) : G * N + g * N + (i - E - N)); };
  struct Inputs {
    T cur, shift, w[kRecTaps];
    float x[kRecTaps];                                            // (of k tokens back)
  } in[2];
  if constexpr (EARLY)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int c = channel(min(tid + 256 * u, channels - 1));
      const T* cw = (const T*)a.conv_w + (int64_t)c * taps;
      in[u].cur = p[a.x_off + c];
      in[u].shift = *(a.conv_b ? (const T*)a.conv_b + c : cw);
#pragma unroll
      for (int k = 0; k < kRecTaps; ++k) {
        in[u].w[k] = cw[max(taps - 1 - k, 0)];
        in[u].x[k] = k > 0 && k < taps && !fresh ? cs[(int64_t)(taps - 1 - k) * C + c] : 0.f;
      }
    }
  const T gate_dt = p[a.dt_off + h];
  const float gate_bias = a.dt_bias[h], gate_log = a.a_log[h], skip = a.d_skip ? a.d_skip[h] : 0.f;
  float4 S[NIT];
#pragma unroll
  for (int i = 0; i < NIT; ++i) {
    const int n = n0 + i * rows;
    S[i] = (!fresh && n < N) ? *reinterpret_cast<const float4*>(st + n * E + e) : float4{0.f, 0.f, 0.f, 0.f};
  }
  if constexpr (EARLY)
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int i = tid + 256 * u;
      float y = (a.conv_b ? Elem<T>::to_f(in[u].shift) : 0.f) + Elem<T>::to_f(in[u].w[0]) * Elem<T>::to_f(in[u].cur);
#pragma unroll
      for (int k = 1; k < kRecTaps; ++k)
        if (k < taps && !fresh) y += Elem<T>::to_f(in[u].w[k]) * in[u].x[k];
      if (i < channels) lds[i] = ssm_silu(y);
    }
  for (int i = EARLY ? tid + 512 : tid; i < channels; i += 256) {
    const int c = channel(i);
    const T* cw = (const T*)a.conv_w + (int64_t)c * taps;
    float y = (a.conv_b ? Elem<T>::to_f(((const T*)a.conv_b)[c]) : 0.f) + Elem<T>::to_f(cw[taps - 1]) * Elem<T>::to_f(p[a.x_off + c]);
    if (!fresh)
      for (int k = 1; k < taps; ++k) y += Elem<T>::to_f(cw[taps - 1 - k]) * cs[(int64_t)(taps - 1 - k) * C + c];
    lds[i] = ssm_silu(y);
  }
  const float dt = ssm_softplus(Elem<T>::to_f(gate_dt) + gate_bias), dec = expf(-expf(gate_log) * dt);
  __syncthreads();
  const float4 x = *reinterpret_cast<const float4*>(lds + e);
  const float4 dx = {dt * x.x, dt * x.y, dt * x.z, dt * x.w};
  float4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NIT; ++i) {
    const int n = n0 + i * rows;
    if (n < N) {
      const float bv = lds[E + n], cv = lds[E + N + n];
      S[i] = float4{dec * S[i].x + bv * dx.x, dec * S[i].y + bv * dx.y, dec * S[i].z + bv * dx.z, dec * S[i].w + bv * dx.w};
      *reinterpret_cast<float4*>(st + n * E + e) = S[i];
      y = float4{y.x + S[i].x * cv, y.y + S[i].y * cv, y.z + S[i].z * cv, y.w + S[i].w * cv};
    }
  }
  for (int o = quads; o < 64; o <<= 1) {
    y.x += __shfl_xor(y.x, o, 64);
    y.y += __shfl_xor(y.y, o, 64);
    y.z += __shfl_xor(y.z, o, 64);
    y.w += __shfl_xor(y.w, o, 64);
  }
  float* sums = lds + E + 2 * N;
  if (lane < quads) *reinterpret_cast<float4*>(sums + (tid >> 6) * E + e) = y;
  __syncthreads();
  if (tid < E)
    a.work[(int64_t)b * a.wld + h * E + tid] = (sums[tid] + sums[E + tid]) + (sums[2 * E + tid] + sums[3 * E + tid]) + skip * lds[tid];
}

// ---------------------------------------------------------------------------------- one token per request: one launch
// A workgroup per request: convolution of the token's channels into LDS (and the shifted inputs back into the state row),
// step sizes and decays, then thread (h, e) walks column e of head h's S in the state row (N multiply-adds for the update,
// N for the read-out; lanes of a wave read adjacent e), then gate, grouped norm and weight.
template <typename T>
__global__ void __launch_bounds__(1024) ssm_decode_kernel(SsmArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];       // x | B | C [C], dt [H], decay [H], y [H E]
  __shared__ float red[16];
  const int b = blockIdx.x;
  const int H = a.H, G = a.G, N = a.N, E = a.E, taps = a.taps;
  const int inner = H * E, C = inner + 2 * G * N;
  const int64_t first_pos = a.seq_lens[b] - 1;
  if (first_pos < 0) return;
  const bool fresh = first_pos == 0;
  const T* p = (const T*)a.p;
  const int64_t slot = a.state_indices[b];
  float* cs = a.conv_state + slot * a.conv_ld;
  float* xbc = lds;
  float* dts = lds + C;
  float* ys = lds + C + 2 * H;
  for (int c = threadIdx.x; c < C; c += blockDim.x) {
    const T* cw = (const T*)a.conv_w + (int64_t)c * taps;
    const float cur = Elem<T>::to_f(p[(int64_t)b * a.ld + a.x_off + c]);
    float y = (a.conv_b ? Elem<T>::to_f(((const T*)a.conv_b)[c]) : 0.f) + Elem<T>::to_f(cw[taps - 1]) * cur;
    // state entry s is the input s - (taps - 1) tokens back; every entry moves one place down and the token comes in last
    for (int s = 0; s < taps - 1; ++s) {
      const float x = fresh ? 0.f : cs[(int64_t)s * C + c];
      y += Elem<T>::to_f(cw[s]) * x;
      if (s > 0) cs[(int64_t)(s - 1) * C + c] = x;
    }
    if (taps > 1) cs[(int64_t)(taps - 2) * C + c] = cur;
    xbc[c] = ssm_silu(y);
  }
  for (int h = threadIdx.x; h < H; h += blockDim.x) {
    const float dt = ssm_softplus(Elem<T>::to_f(p[(int64_t)b * a.ld + a.dt_off + h]) + a.dt_bias[h]);
    dts[h] = dt;
    dts[H + h] = expf(-expf(a.a_log[h]) * dt);
  }
  __syncthreads();
  float* st = a.state + slot * a.state_ld;
  for (int c = threadIdx.x; c < inner; c += blockDim.x) {
    const int h = c / E, e = c - h * E, g = h / (H / G);
    const float xv = xbc[c], dec = dts[H + h], dx = dts[h] * xv;
    const float* Bv = xbc + inner + g * N;
    const float* Cv = xbc + inner + G * N + g * N;
    float* col = st + (int64_t)h * N * E + e;
    float y = 0.f;
    for (int i = 0; i < N; ++i) {
      const float s = (fresh ? 0.f : dec * col[(int64_t)i * E]) + Bv[i] * dx;
      col[(int64_t)i * E] = s;
      y += s * Cv[i];
    }
    ys[c] = y + (a.d_skip ? a.d_skip[h] : 0.f) * xv;
  }
  __syncthreads();
  ssm_gate_norm_store<T>(a, ys, p + (int64_t)b * a.ld + a.z_off, (T*)a.out + (int64_t)b * a.out_ld, red);
}

}  // namespace semipd

using namespace semipd;

extern "C" int64_t semipd_state_space_work_width(int num_heads, int groups, int state, int v_dim) {
  const int64_t w = (int64_t)num_heads * v_dim + 2 * (int64_t)groups * state + 2 * num_heads;
  return (w + 3) / 4 * 4;
}

// The rows per request from which a prompt batch goes in chunks: on average, since the lengths are on the device.  (The time token by token
// is the longest request's: an uneven batch gains from chunks at a lower average than these.)  Token by token against chunks, whole call, us,
// rows on average.  Heads of 128 x 64, 8 groups: 1 request, 128 heads: 8 rows 27 / 29, 10 rows 30 / 29; 4 requests, 128 heads: 7 rows 35 / 35, 96
// heads: 7 rows 32 / 33, 9 rows 36 / 33; 8 requests, 128 heads: 5 rows 45 / 49, 7 rows 53 / 48; 12 requests: 5 rows 63 / 61; 32 requests: 5 rows
// 143 / 137.  Requests and groups that leave XCDs without a share of the walk cost it what the next full number would: 128 heads, 1
// group, 12 requests: 5 rows 62 / 72, 7 rows 71 / 72, 9 rows 79 / 72; 8 requests: 7 rows 51 / 48.  A state of up to 64 rows is padded to
// 64 and has half the work a row: 128 heads of 64 x 64, 24 requests: 7 rows 77 / 82, 9 rows 88 / 82; 8 heads, 1 request: 8 to
// 11 rows 24.5 / 26; of 32 x 64, 16 requests: 7 rows
// 43 / 61, 11 rows 53 / 61; 256 heads of 16 x 64, 1 request of 16 rows 55 / 58, 24 rows 61 / 58; 8 of 24 rows 107 / 104; 16 of 24 rows
// 147 / 157, 32 rows 170 / 159.
constexpr int64_t kSsmChunkRows = 12;                // ... at most, states of up to 16 rows apart
static int64_t ssm_chunk_min_rows(int64_t batch, int num_heads, int groups, int state_size) {
  const int64_t heads = batch * num_heads, units = batch * groups;
  if (state_size <= 32) return state_size > 16 ? kSsmChunkRows : heads >= 4096 ? 28 : 24;
  const int64_t shares = units >= 8 ? (units + 7) / 8 * 8 : units > 4 ? 8 : units == 3 ? 4 : units;       // (see rec_unit_xcds)
  const int64_t rows = (heads < 128 ? kSsmChunkRows : state_size <= 64 ? 8 : heads >= 1152 ? 5 : heads >= 512 ? 6 : heads >= 384 ? 8 : 9) * shares / units;
  return rows < kSsmChunkRows ? rows : kSsmChunkRows;
}
static int ssm_padded_state(int state_size) { return state_size <= 64 ? 64 : 128; }

extern "C" int64_t semipd_state_space_chunk_elems(int64_t num_tokens, int64_t batch, int num_heads, int groups, int state_size, int taps) {
  if (batch <= 0 || groups <= 0 || num_tokens < ssm_chunk_min_rows(batch, num_heads, groups, state_size) * batch || state_size > 128 || taps > kRecTaps) return 0;
  const int64_t elems = rec_max_chunks(num_tokens, batch) * (groups * ssm_frag_elems(ssm_padded_state(state_size)) + (int64_t)num_heads * kSsmHead);
  return rec_short_and_large(num_tokens, batch, elems) ? 0 : elems;
}

// Which of the two walks a state of up to 64 rows takes: a workgroup a CU at most is a chain of chunks each, which the walk without barriers
// goes through faster where the chain is longer than a few and columns come in whole pieces.  Whole call, in pieces / this one, us: 8 heads of
// 64 x 64, 1 request of 300 rows 46.5 / 44.5, 1200 rows 126 / 111, 4000 rows 362 / 312; 24 heads, 8 of 900 148 / 135; 128 heads, 1 of 4000 440 / 372,
// of 60 28.5 / 29.8; 64 heads, 4 of 1900 (256 workgroups) 286 / 250; 8 of 400 (512) 103 / 111; 24 heads, 16 of 300 (384) 83 / 94; 4 heads of 64 x
// 100, 4 of 1200 233 / 275.  The state behind 3 requests of 700 rows is 9.2e-8 from the 64-bit one, in pieces 7.9e-8, with its products on
// top of S 9.6e-8.
static bool ssm_small_walk(const SsmArgs& a, int64_t workgroups) { return workgroups <= 256 && a.num_tokens >= 100 * a.batch && a.E % 16 == 0 && a.ld % 8 == 0; }

template <typename T, int NP>
static void launch_ssm_chunks(const SsmArgs& a, hipStream_t s) {
  const int64_t chunks = rec_max_chunks(a.num_tokens, a.batch), members = (int64_t)(a.H / a.G) * ((a.E + 63) / 64);
  const dim3 operands((unsigned)chunks, (unsigned)a.G, rec_head_splits(chunks * a.G, a.H / a.G)), walk(rec_walk_blocks(a.batch * a.G, members));
  if constexpr (NP == 64)
    if (ssm_small_walk(a, a.batch * a.G * members)) {
      hipLaunchKernelGGL((ssm_chunk_operands_kernel<T, NP, false>), operands, dim3(256), 0, s, a);
      hipLaunchKernelGGL((ssm_chunk_walk_small_kernel<T>), walk, dim3(256), 0, s, a, chunks);
      return;
    }
  hipLaunchKernelGGL((ssm_chunk_operands_kernel<T, NP, true>), operands, dim3(256), 0, s, a);
  if constexpr (NP > 64) {
    // 32 columns a workgroup as long as every one of them has a CU of the launch's share (rec_walk_blocks: of the XCD with the most)
    // (128 heads of 128 x 64 over 8, 1 request of 1000 rows, 256 workgroups of 32: 105 us on 256 CUs; on 224 178, with 64 columns 138)
    const unsigned narrow = rec_walk_blocks(a.batch * a.G, (int64_t)(a.H / a.G) * ((a.E + 31) / 32));
    if (narrow <= launch_cus()) {
      hipLaunchKernelGGL((ssm_chunk_walk_kernel<T, NP, 2>), dim3(narrow), dim3(512), 0, s, a, chunks);
      return;
    }
  }
  hipLaunchKernelGGL((ssm_chunk_walk_kernel<T, NP, 4>), walk, dim3(512), 0, s, a, chunks);
}

static int state_space(const void* proj, int64_t ld, int64_t z_off, int64_t x_off, int64_t dt_off, const void* conv_w,
                                  const void* conv_b, const float* dt_bias, const float* a_log, const float* d_skip,
                                  const void* norm_w, int norm_groups, float eps, float* work, int64_t work_ld, float* state,
                                  int64_t state_ld, float* conv_state, int64_t conv_ld, const int64_t* state_indices,
                                  const int64_t* seq_lens, const int32_t* q_start, const int32_t* q_len, int64_t batch,
                                  int64_t num_tokens, int num_heads, int groups, int state_size, int v_dim, int taps, void* out,
                                  int64_t out_ld, int fused_decode, float* chunk_work, int64_t chunk_elems, int dtype, void* stream) {
  SEMIPD_CHECK_ARG(batch >= 0 && num_tokens >= 0, SEMIPD_EINVAL, "state_space: bad sizes");
  if (batch == 0 || num_tokens == 0) return 0;
  SEMIPD_CHECK_ARG(num_heads > 0 && groups > 0 && num_heads % groups == 0 && state_size > 0 && v_dim > 0 && taps >= 1 && taps <= 64,
                   SEMIPD_ESHAPE, "state_space: %d heads over %d groups, state %d, values %d, %d taps", num_heads, groups,
                   state_size, v_dim, taps);
  SEMIPD_CHECK_ARG(state_size <= 256, SEMIPD_ESHAPE, "state_space: a state of %d rows per head (at most 256)", state_size);
  const int64_t inner = (int64_t)num_heads * v_dim, C = inner + 2 * (int64_t)groups * state_size;
  SEMIPD_CHECK_ARG(norm_groups > 0 && inner % norm_groups == 0, SEMIPD_ESHAPE, "state_space: %d norm groups over %lld elements",
                   norm_groups, (long long)inner);
  SEMIPD_CHECK_ARG(proj && conv_w && dt_bias && a_log && norm_w && state && out && state_indices && seq_lens &&
                       (taps == 1 || conv_state),
                   SEMIPD_EINVAL, "state_space: null pointer");
  SEMIPD_CHECK_ARG((q_start == nullptr) == (q_len == nullptr), SEMIPD_EINVAL, "state_space: q_start and q_len come together");
  SEMIPD_CHECK_ARG(q_start != nullptr || num_tokens == batch, SEMIPD_EINVAL, "state_space: one row per request without q_start");
  SEMIPD_CHECK_ARG(state_ld >= inner * state_size && (taps == 1 || conv_ld >= (int64_t)(taps - 1) * C) && out_ld >= inner,
                   SEMIPD_EINVAL, "state_space: rows too short");
  SEMIPD_CHECK_ARG(z_off >= 0 && x_off >= 0 && dt_off >= 0 && ld >= z_off + inner && ld >= x_off + C && ld >= dt_off + num_heads,
                   SEMIPD_EINVAL, "state_space: a column range leaves the row");
  SsmArgs a{proj, ld, z_off, x_off, dt_off, conv_w, conv_b, dt_bias, a_log, d_skip, norm_w, norm_groups, eps, work, work_ld, state,
            state_ld, conv_state, conv_ld, state_indices, seq_lens, q_start, q_len, batch, num_tokens, num_heads, groups, state_size,
            v_dim, taps, out, out_ld, chunk_work};
  hipStream_t s = as_stream(stream);
  const size_t dec_lds = (size_t)(C + 2 * num_heads + inner) * sizeof(float);
  if (q_start == nullptr && fused_decode && dec_lds <= 160 * 1024 - 256) {
    const int threads = inner >= 1024 ? 1024 : (int)((inner + 63) / 64 * 64);
    static std::atomic<uint64_t> done[3] = {};
    int rc = 0;
    SEMIPD_DISPATCH_DTYPE(dtype, T, {
      const int slot = sizeof(T) == 4 ? 0 : (dtype == SEMIPD_BF16 ? 1 : 2);
      if (dec_lds > 65536 && ensure_dynamic_lds((const void*)ssm_decode_kernel<T>, dec_lds, done[slot], "state_space")) rc = 1;
      if (!rc) hipLaunchKernelGGL((ssm_decode_kernel<T>), dim3((unsigned)batch), dim3(threads), dec_lds, s, a);
    });
    if (rc) return SEMIPD_EINVAL;
    return launch_status("state_space_decode");
  }
  const int64_t want = q_start ? semipd_state_space_chunk_elems(num_tokens, batch, num_heads, groups, state_size, taps) : 0;
  const bool chunks = want > 0 && chunk_work && chunk_elems >= want && aligned16(chunk_work);
  SEMIPD_CHECK_ARG(work && work_ld >= (chunks ? inner : semipd_state_space_work_width(num_heads, groups, state_size, v_dim)), SEMIPD_EINVAL,
                   "state_space: the work rows are missing or too short");
  // gate and norm with 16-byte accesses and the row in registers
  const int64_t gs = inner / norm_groups;
  const bool post8 = dtype != SEMIPD_F32 && gs % 8 == 0 && gs <= 8 * 256 * kPostPieces && z_off % 8 == 0 && ld % 8 == 0 && out_ld % 8 == 0 &&
                     work_ld % 4 == 0 && aligned16(proj) && aligned16(out) && aligned16(norm_w) && aligned16(work);
  // ... and the convolution's inputs moved on, both behind everything that reads them; in one launch unless the result may be written over
  // the inputs
  auto post = [&]() -> int {
    const int64_t blocks = taps > 1 ? (C + 255) / 256 : 0;
    const bool one = post8 && rec_apart(proj, x_off, C, ld, out, inner, out_ld, num_tokens);
    if (blocks && !one)
      SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((ssm_conv_state_kernel<T>), dim3((unsigned)blocks, (unsigned)batch), dim3(256), 0, s, a))
    const int64_t moved = one ? blocks * batch : 0;
    if (post8)
      SEMIPD_DISPATCH_HALF(dtype, T, hipLaunchKernelGGL((ssm_post_vec_kernel<T>), dim3((unsigned)(num_tokens + moved), (unsigned)norm_groups),
                                                        dim3(256), 0, s, a, (int)moved))
    else
      SEMIPD_DISPATCH_DTYPE(dtype, T, hipLaunchKernelGGL((ssm_post_kernel<T>), dim3((unsigned)num_tokens), dim3(256), 0, s, a))
    return 0;
  };
  if (chunks) {
    SEMIPD_DISPATCH_DTYPE(dtype, T, if (state_size <= 64) launch_ssm_chunks<T, 64>(a, s); else launch_ssm_chunks<T, 128>(a, s));
    if (post()) return SEMIPD_EDTYPE;
    return launch_status("state_space(chunks)");
  }
  // a decode batch whose state rows lie on 16-byte boundaries: up to 16 pieces of four columns a thread
  const bool pow2 = v_dim >= 16 && v_dim <= 256 && (v_dim & (v_dim - 1)) == 0;
  if (q_start == nullptr && batch <= 65535 && pow2 && (int64_t)state_size * v_dim <= 16 * 1024 && state_size % 4 == 0 && aligned16(state) && state_ld % 4 == 0) {
    const int nit = (state_size * v_dim + 1023) / 1024;
    const size_t bytes = (size_t)(v_dim + 2 * state_size + 4 * v_dim) * sizeof(float);
    const dim3 grid((unsigned)num_heads, (unsigned)batch);
    SEMIPD_DISPATCH_DTYPE(dtype, T, {
      const auto go = [&](auto early) {
        constexpr bool EARLY = decltype(early)::value;
        if (nit <= 4) hipLaunchKernelGGL((ssm_step_kernel<T, 4, EARLY>), grid, dim3(256), bytes, s, a);
        else if (nit <= 8) hipLaunchKernelGGL((ssm_step_kernel<T, 8, EARLY>), grid, dim3(256), bytes, s, a);
        else hipLaunchKernelGGL((ssm_step_kernel<T, 16, EARLY>), grid, dim3(256), bytes, s, a);
      };
      if (taps <= kRecTaps) go(std::true_type{});
      else go(std::false_type{});
    });
    if (post()) return SEMIPD_EDTYPE;
    return launch_status("state_space(step)");
  }
  const unsigned cblocks = (unsigned)((C + kPrepChannels - 1) / kPrepChannels);
  // four channels per thread: every row and column range starts on a multiple of four elements
  const bool prep4 = C % 4 == 0 && x_off % 4 == 0 && ld % 4 == 0 && work_ld % 4 == 0 && (taps == 1 || conv_ld % 4 == 0) &&
                     ((uintptr_t)proj % 16) == 0 && aligned16(work) && (taps == 1 || aligned16(conv_state)) &&
                     aligned16(conv_w) && taps <= kPrepMaxTaps;
  // a prompt batch: a workgroup walks a tile of tokens with its channels' taps in registers, where that leaves the chip enough of them; else a
  // token each (by tokens / by tiles, heads of 128 x 64, whole call token by token, us: 8 heads, 64 requests of 16 rows 62 / 328; 128 heads, 64 of 16
  // rows, 328 tiles' workgroups, 606 / 831, 8 of 400 rows, 1000 of them, 1095 / 988)
  const int tile = (q_start != nullptr && prep4 && num_tokens / kPrepTile * cblocks >= kPrepTileBlocks) ? kPrepTile : 1;
  const dim3 pgrid((unsigned)((num_tokens + tile - 1) / tile), cblocks);
  SEMIPD_DISPATCH_DTYPE(dtype, T, {
    if (prep4) hipLaunchKernelGGL((ssm_prep_kernel<T, true>), pgrid, dim3(256), 0, s, a, tile);
    else hipLaunchKernelGGL((ssm_prep_kernel<T, false>), pgrid, dim3(256), 0, s, a, tile);
  });
  // 16-byte staging reads: B, C and x of a token start on multiples of four floats
  const bool scan4 = work_ld % 4 == 0 && aligned16(work) && inner % 4 == 0 && state_size % 4 == 0 && v_dim % 4 == 0;
#define SEMIPD_SSM_SCAN(NPT, NS)                                                                                              \
  do {                                                                                                                        \
    constexpr int cols = 64 / NS;                                                                                             \
    const unsigned blocks = (unsigned)(batch * num_heads * ((v_dim + cols - 1) / cols));                                      \
    const size_t bytes = 2 * (size_t)kSsmStage * (2 * (NS > 1 ? NPT + 4 : NPT) * NS + cols + 4) * sizeof(float);              \
    if (scan4) hipLaunchKernelGGL((ssm_scan_kernel<NPT, NS, true>), dim3(blocks), dim3(64), bytes, s, a);                     \
    else hipLaunchKernelGGL((ssm_scan_kernel<NPT, NS, false>), dim3(blocks), dim3(64), bytes, s, a);                          \
  } while (0)
  if (state_size <= 16) SEMIPD_SSM_SCAN(16, 1);
  else if (state_size <= 32) SEMIPD_SSM_SCAN(32, 1);
  else if (state_size <= 64) SEMIPD_SSM_SCAN(32, 2);
  else if (state_size <= 128) SEMIPD_SSM_SCAN(32, 4);
  else SEMIPD_SSM_SCAN(32, 8);
#undef SEMIPD_SSM_SCAN
  if (post()) return SEMIPD_EDTYPE;
  return launch_status("state_space");
}

extern "C" int semipd_state_space(const void* proj, int64_t ld, int64_t z_off, int64_t x_off, int64_t dt_off, const void* conv_w,
                                  const void* conv_b, const float* dt_bias, const float* a_log, const float* d_skip,
                                  const void* norm_w, int norm_groups, float eps, float* work, int64_t work_ld, float* state,
                                  int64_t state_ld, float* conv_state, int64_t conv_ld, const int64_t* state_indices,
                                  const int64_t* seq_lens, const int32_t* q_start, const int32_t* q_len, int64_t batch,
                                  int64_t num_tokens, int num_heads, int groups, int state_size, int v_dim, int taps, void* out,
                                  int64_t out_ld, int fused_decode, int dtype, void* stream) {
  return state_space(proj, ld, z_off, x_off, dt_off, conv_w, conv_b, dt_bias, a_log, d_skip, norm_w, norm_groups, eps, work, work_ld, state,
                     state_ld, conv_state, conv_ld, state_indices, seq_lens, q_start, q_len, batch, num_tokens, num_heads, groups,
                     state_size, v_dim, taps, out, out_ld, fused_decode, nullptr, 0, dtype, stream);
}

extern "C" int semipd_state_space_record(const void* record) {
  SEMIPD_CHECK_ARG(record != nullptr, SEMIPD_EINVAL, "state_space: null record");
  int64_t r[35];
  double eps;
  memcpy(r, record, sizeof(r));
  memcpy(&eps, &r[12], sizeof(eps));
  auto at = [&](int i) { return reinterpret_cast<void*>(r[i]); };
  return semipd_state_space(at(0), r[1], r[2], r[3], r[4], at(5), at(6), (const float*)at(7), (const float*)at(8), (const float*)at(9), at(10), (int)r[11],
                            (float)eps, (float*)at(13), r[14], (float*)at(15), r[16], (float*)at(17), r[18], (const int64_t*)at(19), (const int64_t*)at(20),
                            (const int32_t*)at(21), (const int32_t*)at(22), r[23], r[24], (int)r[25], (int)r[26], (int)r[27], (int)r[28], (int)r[29], at(30), r[31],
                            (int)r[32], (int)r[33], at(34));
}

extern "C" int semipd_state_space_prompt(const void* proj, int64_t ld, int64_t z_off, int64_t x_off, int64_t dt_off, const void* conv_w,
                                         const void* conv_b, const float* dt_bias, const float* a_log, const float* d_skip,
                                         const void* norm_w, int norm_groups, float eps, float* work, int64_t work_ld, float* state,
                                         int64_t state_ld, float* conv_state, int64_t conv_ld, const int64_t* state_indices,
                                         const int64_t* seq_lens, const int32_t* q_start, const int32_t* q_len, int64_t batch,
                                         int64_t num_tokens, int num_heads, int groups, int state_size, int v_dim, int taps, void* out,
                                         int64_t out_ld, float* chunk_work, int64_t chunk_elems, int dtype, void* stream) {
  return state_space(proj, ld, z_off, x_off, dt_off, conv_w, conv_b, dt_bias, a_log, d_skip, norm_w, norm_groups, eps, work, work_ld, state,
                     state_ld, conv_state, conv_ld, state_indices, seq_lens, q_start, q_len, batch, num_tokens, num_heads, groups,
                     state_size, v_dim, taps, out, out_ld, 0, chunk_work, chunk_elems, dtype, stream);
}
