// What the chunked forms of the recurrences with a matrix state share (state_space.hip, delta_rule.hip): where a chunk of a
// launch lies, accurate exponentials, and the tiles that a wave moves between rows in memory and its accumulators' places.
#pragma once

#include <type_traits>
#include "common.h"
#include "mfma_frag.h"

namespace semipd {

constexpr int kRecChunk = 32;            // tokens of a chunk
constexpr int kRecTaps = 4;              // taps of the convolution at most
constexpr int kRecHalo = kRecTaps - 1;   // rows in front of a chunk that its convolution looks at

// The walks' workgroups: `units` of (request, group) with `members` each, which read the same operands.  A unit stays on one XCD (workgroup
// ids go round the 8); fewer than 8 units have several each, or most of the chip would have none (128 heads of 128 x 64 in one group, 1
// request of 12 rows, whole call: 66 -> 36 us; of 96 rows 99 -> 46).
__host__ __device__ inline int rec_unit_xcds(int64_t units) { return units < 8 ? 8 / (int)units : 1; }
inline unsigned rec_walk_blocks(int64_t units, int64_t members) {
  const int x = rec_unit_xcds(units), at_once = 8 / x;
  return (unsigned)((units + at_once - 1) / at_once * ((members + x - 1) / x) * 8);
}
struct RecPlace {
  int unit, member;                      // (unit -1: none)
};
__device__ __forceinline__ RecPlace rec_place(int units, int members) {
  const int x = rec_unit_xcds(units), turns = (members + x - 1) / x, turn = blockIdx.x / 8, xcd = blockIdx.x % 8;
  const int unit = turn / turns * (8 / x) + xcd / x, member = turn % turns * x + xcd % x;
  return unit < units && xcd / x < 8 / x && member < members ? RecPlace{unit, member} : RecPlace{-1, 0};
}

// Request at place `pos` of a launch: the longest first, so that none starts late.  Where a CU holds two of the walk's workgroups and all of
// them start together, those behind the first `firsts` (which have a CU each) come from the shortest up, so that the ones that come to a
// long one's CU are short.  State space, 4 requests of 1330, 2034, 1599 and 2303 rows: in their order the second and the fourth share CUs
// (walk 412 us, so placed 345).  A walk with one workgroup a CU passes `batch`: behind the first 256 they start as CUs come free, the
// longest of them first.  A whole wave asks.
__device__ __forceinline__ int rec_first_requests(int batch, int per_request) {       // (workgroups of a request; two a CU; more: all from the longest down)
  return batch * (int64_t)per_request > 512 ? batch : min(batch, (256 + per_request - 1) / per_request);
}
__device__ __forceinline__ int rec_by_length(const int32_t* q_len, int batch, int pos, int firsts) {
  if (batch > 64) return pos;
  const int lane = threadIdx.x & 63, n = lane < batch ? q_len[lane] : 0;
  int rank = 0;
  for (int j = 0; j < batch; ++j) {
    const int m = __builtin_amdgcn_readlane(n, j);
    rank += m > n || (m == n && j < lane) ? 1 : 0;
  }
  const int want = pos < firsts ? pos : batch - 1 - (pos - firsts);
  return __builtin_ctzll(__ballot(lane < batch && rank == want));
}

// Workgroups that share out the heads of a (chunk, group), eight each, as long as the chip is not full of them: `items` (chunk, group)s.
// 128 heads of 128 x 64 in one group, 1 request of 12 rows, whole call: one workgroup for all heads 106 us, 16 of them 66 (token by
// token 48).
inline unsigned rec_head_splits(int64_t items, int heads) {
  const int64_t most = (heads + 7) / 8, room = items < 512 ? 512 / items : 1;
  return (unsigned)(most < room ? most : room);
}

// Whether columns [off, off + n) of `rows` rows `ld` apart and the result's [rows, m] share no byte (elements of 2 bytes; the space from first
// to last byte of each is taken as its own).
inline bool rec_apart(const void* p, int64_t off, int64_t n, int64_t ld, const void* out, int64_t m, int64_t out_ld, int64_t rows) {
  const uintptr_t a = (uintptr_t)p + 2 * off, b = (uintptr_t)out;
  return a + 2 * ((rows - 1) * ld + n) <= b || b + 2 * ((rows - 1) * out_ld + m) <= a;
}

inline int64_t rec_max_chunks(int64_t num_tokens, int64_t batch) { return num_tokens / kRecChunk + batch; }

// Operands of a chunk are as large however few rows it has (state space, 128 heads of 128 x 64 in 8 groups: 852 KB, 27 KB a row of full ones
// and 197 where requests have 5 rows): requests of less than half a chunk on average go in chunks only up to 512 MB of them (that size, 5 rows: 544
// requests), or a call of short prompts would take several times the memory of one of long ones with as many rows.
inline bool rec_short_and_large(int64_t num_tokens, int64_t batch, int64_t elems) { return num_tokens < kRecChunk / 2 * batch && elems > (1ll << 27); }

// Chunk `idx` of the launch (request after request, each in chunks of 32 rows) -> request, chunk in it and what is known of the request, in
// one round trip; a whole wave asks.
struct RecChunk {
  int b, n, q_start;                     // request, its rows, its first
  int64_t c, first_pos;                  // chunk in it; rows of the sequence in front of the portion
};
__device__ __forceinline__ bool rec_find_chunk(const int32_t* q_len, const int64_t* seq_lens, const int32_t* q_start, int batch, int64_t idx, RecChunk& at) {
  const int lane = threadIdx.x & 63;
  int64_t before = 0;
  for (int r0 = 0; r0 < batch; r0 += 64) {
    const int rq = min(r0 + lane, batch - 1), rows = q_len[rq], start = q_start[rq];
    const int64_t len = seq_lens[rq];
    const int n = r0 + lane < batch ? max(0, (rows + kRecChunk - 1) / kRecChunk) : 0;
    int s = n;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int t = __shfl_up(s, o, 64);
      if (lane >= o) s += t;
    }
    const int total = __builtin_amdgcn_readlane(s, 63);
    if (idx < before + total) {
      const int first = __builtin_ctzll(__ballot(before + s > idx));
      at.b = r0 + first;
      at.c = idx - before - (__builtin_amdgcn_readlane(s, first) - __builtin_amdgcn_readlane(n, first));
      at.n = __builtin_amdgcn_readlane(rows, first);
      at.q_start = __builtin_amdgcn_readlane(start, first);
      at.first_pos = ((int64_t)(uint32_t)__builtin_amdgcn_readlane((int)len, first) | (int64_t)__builtin_amdgcn_readlane((int)(len >> 32), first) << 32) - at.n;
      return true;
    }
    before += total;
  }
  return false;
}

// A channel's taps (wt: the one for the input i tokens back), the inputs in front of a chunk of cnt rows (in) and the chunk's own (x, past its
// end the last one), all under way at once: p the channel in the chunk's first row, `inside` whether the portion has rows in front of that,
// `state` the channel's entry in the kept inputs (C apart; null: the sequence starts).  Read where they are needed, each behind a condition
// of its own, they were seven round trips: with the silu below 9.6 us of a workgroup's 30, now 5.3 of 20 (delta rule, keys of
// 128; 7266 rows, the launch: delta rule 101 -> 69 us, state space 78 -> 59).
template <typename T>
__device__ __forceinline__ void rec_channel(const T* p, int64_t ld, int cnt, const T* cw, int taps, bool inside, const float* state, int64_t C,
                                            float (&wt)[kRecTaps], float (&in)[kRecTaps], float (&x)[kRecChunk]) {
  T raw[kRecChunk], w[kRecTaps];
#pragma unroll
  for (int i = 0; i < kRecTaps; ++i) w[i] = cw[max(taps - 1 - i, 0)];
#pragma unroll
  for (int i = 0; i < kRecChunk; ++i) raw[i] = p[(int64_t)min(i, cnt - 1) * ld];
#pragma unroll
  for (int i = 0; i < kRecTaps; ++i) in[i] = 0.f;
  if (inside) {
    T back[kRecTaps];
#pragma unroll
    for (int i = 1; i < kRecTaps; ++i) back[i] = p[-(int64_t)min(i, taps - 1) * ld];
#pragma unroll
    for (int i = 1; i < kRecTaps; ++i) in[i] = i < taps ? Elem<T>::to_f(back[i]) : 0.f;
  } else if (state != nullptr) {
    float back[kRecTaps];
#pragma unroll
    for (int i = 1; i < kRecTaps; ++i) back[i] = state[(int64_t)max(taps - 1 - i, 0) * C];
#pragma unroll
    for (int i = 1; i < kRecTaps; ++i) in[i] = i < taps ? back[i] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < kRecTaps; ++i) wt[i] = i < taps ? Elem<T>::to_f(w[i]) : 0.f;
#pragma unroll
  for (int i = 0; i < kRecChunk; ++i) x[i] = Elem<T>::to_f(raw[i]);
}
// how many chunks the requests in front of b have
__device__ __forceinline__ int64_t rec_chunks_before(const int32_t* q_len, int b) {
  const int lane = threadIdx.x & 63;
  int s = 0;
  for (int r = lane; r < b; r += 64) s += max(0, (q_len[r] + kRecChunk - 1) / kRecChunk);
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  return s;
}

__device__ __forceinline__ bool rec_finite(float x) { return fabsf(x) <= 3.402823466e38f; }

// up to here a sum of 128 products of two values stays within 32 bits: a chunk with a larger one is taken token by token
__device__ __forceinline__ bool rec_moderate(float x) { return fabsf(x) <= 0x1p59f; }

// Log decays whose running sums, and the differences of these, are good to 64 bits less 26: a chunk of 32 sums to less than 2^26 (base 2),
// so a difference is off by 2^-27 at most, which costs a weight less than its own rounding.  One of -1e14 among them costs the weights
// behind it 6e-3, one of -1e16 sets them to 1: a chunk with such a step is taken token by token.
__device__ __forceinline__ bool rec_moderate_decay(float la) { return fabsf(la) <= 0x1p20f; }

// silu of a moderate x: e^(-x) as 2^(hi + lo) with lo = what the product with log2 e rounds away, the quotient by a reciprocal and one
// correction of it and of the result: at most 2.8 units in the last place from the 64-bit value (x / (1 + expf(-x)): 3.4).  The
// quotient is 2^32 times as large until the end, so that it stays in the normal range as far as e^(-x) does, to -88.722; x below has
// the value there, -2.6e-37.
__device__ __forceinline__ float rec_silu(float x) {
  const float c = fmaxf(x, -88.722f);
  const float hi = c * -1.44269502f, lo = fmaf(c, -1.44269502f, -hi) + c * -1.92596299e-8f;
  float e = __builtin_amdgcn_exp2f(hi);
  e = fmaf(e, lo * 0.693147182f, e);
  const float d = fmaf(e, 0x1p-32f, 0x1p-32f);
  float r = __builtin_amdgcn_rcpf(d);
  r = fmaf(fmaf(-d, r, 1.0f), r, r);
  const float q = c * r;
  return fmaf(fmaf(-d, q, c), r, q) * 0x1p-32f;
}
// ... where x stands for its silu because it is not moderate: x itself or 0, of minus infinity not a number
__device__ __forceinline__ float rec_silu_if_large(float x) { return rec_moderate(x) ? x : (x > 0.f ? x : x * 0.f); }

// Convolution and silu of a channel's chunk (as rec_channel has read it) into a column of LDS, zeros past its cnt rows; true where a sum is not
// moderate.  Eight rows at a time without a branch between them: with one each, every row waited for its own exponential and quotient.
__device__ __forceinline__ bool rec_conv_silu(const float (&wt)[kRecTaps], const float (&in)[kRecTaps], float (&x)[kRecChunk], float bias, int taps, int cnt,
                                              float* dst, int stride) {
  auto sums = [&](auto all) {
#pragma unroll
    for (int t = kRecChunk - 1; t >= 0; --t) {
      float y = bias;
#pragma unroll
      for (int i = 0; i < kRecTaps; ++i)
        if (decltype(all)::value || i < taps) y += wt[i] * (t >= i ? x[t >= i ? t - i : 0] : in[t >= i ? 0 : i - t]);
      x[t] = y;
    }
  };
  if (taps == kRecTaps) sums(std::true_type{});
  else sums(std::false_type{});
  bool large = false;
#pragma unroll
  for (int t0 = 0; t0 < kRecChunk; t0 += 8) {
    bool over = false;
#pragma unroll
    for (int t = t0; t < t0 + 8; ++t) over |= t < cnt && !rec_moderate(x[t]);
    large |= over;
    float y[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) y[u] = rec_silu(x[t0 + u]);
    if (__any(over))
#pragma unroll
      for (int u = 0; u < 8; ++u) y[u] = rec_moderate(x[t0 + u]) ? y[u] : rec_silu_if_large(x[t0 + u]);
#pragma unroll
    for (int u = 0; u < 8; ++u) dst[(t0 + u) * stride] = t0 + u < cnt ? y[u] : 0.f;
  }
  return large;
}

// The weight e^(b_t) of a head's chunk, by the half wave that has its 32 tokens: the last one is not a number where `no` holds for any
// of them, and the chunk is taken token by token by that.
__device__ __forceinline__ float rec_flagged(float eb, bool no) {
  const uint64_t all = __ballot(no);
  const bool any = (threadIdx.x & 32 ? all >> 32 : all & 0xffffffffull) != 0;
  return any && (threadIdx.x & 31) == 31 ? __builtin_nanf("") : eb;
}

// 2^x of a 64-bit exponent: what rounding it to 32 bits takes away is multiplied in
__device__ __forceinline__ float rec_exp2(double x) {
  const float hi = (float)x, lo = (float)(x - (double)hi);
  const float e = __builtin_amdgcn_exp2f(hi);
  return hi < -126.f ? e : fmaf(e, lo * 0.693147182f, e);
}

// ---- fp32 products on the bf16 matrix cores
// x as the sum of three bf16 values, each the rounding of what those in front of it leave: 8 + 8 + 8 bits and the signs hold all 24 of x
// (down to 2^-110, where the last piece leaves the format; what is off by 2^-134 there is below anything that is added up).
// Eight of a lane's elements make an operand of v_mfma_f32_16x16x32_bf16: lane (r16, kq) has k = 4 kq .. + 3 and 16 + 4 kq .. + 3 of a step
// of 32, both operands alike: two accumulator tiles of 16 rows are such an operand as they stand.
struct Split3 {
  Frag16 p[3];
};
__device__ __forceinline__ void rec_split2(float a, float b, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = pack2<bf16_t>(a, b);
  const float a1 = a - __uint_as_float(hi << 16), b1 = b - __uint_as_float(hi & 0xffff0000u);
  mid = pack2<bf16_t>(a1, b1);
  lo = pack2<bf16_t>(a1 - __uint_as_float(mid << 16), b1 - __uint_as_float(mid & 0xffff0000u));
}
__device__ __forceinline__ Split3 rec_split8(const f32x4& a, const f32x4& b) {
  Split3 s;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    rec_split2(a[2 * i], a[2 * i + 1], s.p[0].w[i], s.p[1].w[i], s.p[2].w[i]);
    rec_split2(b[2 * i], b[2 * i + 1], s.p[0].w[2 + i], s.p[1].w[2 + i], s.p[2].w[2 + i]);
  }
  return s;
}
// The same of values that may be anything: an infinity or a NaN stands in the first piece alone, and one that would round to an infinity
// does not, so that the three add up to what they were made of.
__device__ __forceinline__ Split3 rec_split8_any(const f32x4& a, const f32x4& b) {
  Split3 s = rec_split8(a, b);
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float x = i < 4 ? a[i] : b[i - 4];
    if (fabsf(x) <= 0x1p126f) continue;
    float x0 = x != x ? x : __uint_as_float(__float_as_uint(x) & 0xffff0000u), x1 = 0.f, x2 = 0.f;
    if (rec_finite(x)) {
      x1 = __uint_as_float(__float_as_uint(x - x0) & 0xffff0000u);
      x2 = (x - x0) - x1;
    }
    s.p[0].e[i] = (uint16_t)(__float_as_uint(x0) >> 16 | (x != x ? 0x40 : 0));
    s.p[1].e[i] = (uint16_t)(__float_as_uint(x1) >> 16);
    s.p[2].e[i] = (uint16_t)(__float_as_uint(x2) >> 16);
  }
  return s;
}
// A B of the pieces without the three products below 2^-25 of the whole (mid lo, lo mid, lo lo): `big` takes the products of the first
// pieces, `small` the other five.  On the 16 x 16 x 4 products of fp32 operands the same takes 8 x 32 cycles, here 6 x 16.
// N row tiles side by side: a product that adds to what the one in front of it wrote waits for it.
template <int N>
__device__ __forceinline__ void rec_mma(const Frag16 (&a)[N][3], const Split3& b, f32x4* big, f32x4* small) {
#pragma unroll
  for (int i = 0; i < N; ++i) small[i] = mma16<bf16_t>(a[i][2], b.p[0], small[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) big[i] = mma16<bf16_t>(a[i][0], b.p[0], big[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) small[i] = mma16<bf16_t>(a[i][0], b.p[2], small[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) small[i] = mma16<bf16_t>(a[i][1], b.p[1], small[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) small[i] = mma16<bf16_t>(a[i][1], b.p[0], small[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) small[i] = mma16<bf16_t>(a[i][0], b.p[1], small[i]);
}
// ... in one sum: the five small products of all that is summed, then, on top of them, those of the first pieces.  An addition less a value
// and a rounding less: the state behind 4 requests of 1900 tokens is 8.24e-8 from the 64-bit one (state space; 8.48e-8 with the two sums
// added at the end) and 4.00e-8 (delta rule; 4.06e-8).  What is held for the last products costs registers: not for C S of the state space's walk.
template <int N>
__device__ __forceinline__ void rec_mma_small(const Frag16 (&a)[N][3], const Split3& b, f32x4* sum) {
#pragma unroll
  for (int i = 0; i < N; ++i) sum[i] = mma16<bf16_t>(a[i][2], b.p[0], sum[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) sum[i] = mma16<bf16_t>(a[i][0], b.p[2], sum[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) sum[i] = mma16<bf16_t>(a[i][1], b.p[1], sum[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) sum[i] = mma16<bf16_t>(a[i][1], b.p[0], sum[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) sum[i] = mma16<bf16_t>(a[i][0], b.p[1], sum[i]);
}
template <int N>
__device__ __forceinline__ void rec_mma_big(const Frag16 (&a)[N][3], const Split3& b, f32x4* sum) {
#pragma unroll
  for (int i = 0; i < N; ++i) sum[i] = mma16<bf16_t>(a[i][0], b.p[0], sum[i]);
}
// ... the value that the pieces `plane` halves apart stand for
__device__ __forceinline__ float rec_joined(const uint16_t* p, int plane) {
  return (__uint_as_float((uint32_t)p[0] << 16) + __uint_as_float((uint32_t)p[plane] << 16)) + __uint_as_float((uint32_t)p[2 * plane] << 16);
}

// Rows of 16 columns that one wave needs (its convolution's inputs: a chunk and the rows in front of it), 16 bytes a lane: a load
// per token, element and lane would be 14 requests of 2 bytes for the two or three here.  `fetch` leaves them in registers,
// `place` puts them into the wave's own LDS (48 / 80 bytes a row: rows that are read together start in different banks).
template <typename T, int TOKENS = kRecChunk> struct RowTile {
  static constexpr int kPerRow = 16 * (int)sizeof(T) / 16;          // 16-byte pieces a row
  static constexpr int kRows = TOKENS + kRecHalo;
  static constexpr int kLoads = (kRows * kPerRow + 63) / 64;
  static constexpr int kStride = sizeof(T) == 2 ? 24 : 20;          // elements of T between rows in LDS
  static constexpr int kElems = kRows * kStride;
  uint4 v[kLoads];
  // rows l0 - halo .. l0 + TOKENS - 1 of `p` (row 0 = the portion's first), zeros behind row n - 1; l0 > 0
  __device__ __forceinline__ void fetch(const T* p, int64_t ld, int l0, int n, int lane) {
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int it = u * 64 + lane, row = it / kPerRow, l = l0 - kRecHalo + row;
      v[u] = uint4{0u, 0u, 0u, 0u};
      if (row < kRows && l < n) v[u] = *reinterpret_cast<const uint4*>(p + (int64_t)l * ld + it % kPerRow * (16 / (int)sizeof(T)));
    }
  }
  // ... row n - 1 in place of those behind it, rows of less than 2^26 bytes: nothing is written to the registers but by the load, and the
  // addresses are an offset of 32 bits a lane
  __device__ __forceinline__ void fetch_clamped(const T* p, int64_t ld, int l0, int n, int lane) {
    const int row0 = min(l0 - kRecHalo, n - 1), last = min(kRows, n - row0) - 1;       // (0 <= row0 <= row0 + last < n, also for l0 behind the portion)
    const char* first = reinterpret_cast<const char*>(p + (int64_t)row0 * ld);
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int it = u * 64 + lane;
      if ((u + 1) * 64 <= kRows * kPerRow || it < kRows * kPerRow)
        v[u] = *reinterpret_cast<const uint4*>(first + ((uint32_t)min(it / kPerRow, last) * (uint32_t)(ld * sizeof(T)) + (uint32_t)(it % kPerRow) * 16u));
    }
  }
  __device__ __forceinline__ void place(T* lds, int lane) const {
#pragma unroll
    for (int u = 0; u < kLoads; ++u) {
      const int it = u * 64 + lane, row = it / kPerRow;
      if (row < kRows) *reinterpret_cast<uint4*>(lds + row * kStride + it % kPerRow * (16 / (int)sizeof(T))) = v[u];
    }
  }
};

constexpr int kOutStride = 20;            // floats between rows of a wave's results in LDS, on their way to rows in memory 16 bytes a lane
// ... of its 32 x 16 results (lane (r16, kq): rows 16 i + 4 kq + r of column r16)
__device__ __forceinline__ void rec_store_tile(const f32x4 (&o)[2], float* lds, float* y, int64_t ld, int lane) {
  const int r16 = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) lds[(16 * i + 4 * kq + r) * kOutStride + r16] = o[i][r];
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 16 * i + (lane >> 2);
    *reinterpret_cast<f32x4*>(y + (int64_t)row * ld + 4 * (lane & 3)) = *reinterpret_cast<const f32x4*>(lds + row * kOutStride + 4 * (lane & 3));
  }
}

}  // namespace semipd
