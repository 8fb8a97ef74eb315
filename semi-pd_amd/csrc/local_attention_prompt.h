// Prompt attention over paged pools, 32 query rows a wave (gfx950): the form of local_attention_mfma_kernel for head sizes of 64 or
// 128 (value rows up to 256).  Included by local_attention.hip behind what it needs (LocalAttnArgs, ScoreMap, range_lo).
//
//  * A workgroup: NW waves = HW query heads of ONE key/value head x NW / HW blocks of 32 rows, so the rows of K and V that it
//    stages serve up to NW heads.  Heads share the visible range, and every wave of a workgroup has the same number of steps.
//  * Launches of few tiles: KS groups of NW waves in a workgroup, which take its steps in turn (split_prompt_attention has the rule).
//  * A step: KT keys (64; 32 for value rows of 256 and groups of two waves).  Their K and V rows go through two pairs of LDS tiles (step i + 1 lands in
//    registers while step i is multiplied; one barrier a step).  S^T = K Q^T and O^T += V^T P^T on v_mfma_f32_32x32x16: a lane holds one query's column
//    throughout, P^T goes from the accumulators into the second product in place (its key order is matched by the rows that the
//    transposing reads of V take).
//  * 16-byte chunk c of row r lies at c ^ (r & 15) of a K tile (the 32 rows of an operand read start in different banks), the 64-byte
//    group t at t ^ (r & 3) of a V tile (the four rows of a transposing read likewise).
//  * The running maximum is the row's own and is taken every 32 keys, also in steps of 64: the largest weight of every 32 is 1 and
//    rounds to 16 bits without an error (a maximum per 64 keys: the result of the window batch below was 0.5 % further from the 64-bit
//    one).  Letting it lag by up to 2^6 was 2 .. 5 % further.
//  * A weight of zero does not hide an infinity or a NaN from a product, and a wave multiplies keys that some of its rows do not see: a
//    wave that ends with sums that are not finite takes its rows again, one by one.
// Bound: a wave multiplies for 32 x 32 cycles a step of 64 keys (128 / 128), reads 32 KB of LDS and takes 32 exponentials a lane (16
// cycles each) with five instructions around each.  Of the SIMD cycles of the batch below the vector unit is busy for 49 %, the matrix
// pipe for 25 %; two waves a SIMD fill only part of each other's gaps (value rows of 256: 41 and 27).  Against 16 rows a wave, steps of 32 keys (which read all of K and V from LDS for half the rows, and had four waves of
// one head): 7262 tokens in blocks of 1024, 32 / 8 heads of 128: 271 -> 97 us (565 TFLOP/s); 32 / 2 heads with value rows of 256: 1971 ->
// 283 (steps of 32 keys there, eight waves: 64 would spill); 300 tokens behind 1000, 32 / 8 heads of 128: 76 -> 44; 8 x 40: 9.0 -> 8.6.
// A fresh prompt of at most 32 tokens is one step of either, and its 32 x 64 products are four times those of the wave of 16 rows: 20
// tokens 7.3 -> 7.4 us, 32 tokens 7.4 -> 7.9, with sigmoid weights 6.5 -> 7.1 and 6.6 -> 7.6 (behind 100 tokens 20 tokens are 12.4 -> 9.6;
// how far a request reaches back is on the device, so the host cannot choose; leaving out a step's second 32 keys where there
// are none took 0.5 us off the short ones and put 10 on the large).
#pragma once

namespace semipd {

// Rows wq0 .. wq0 + 31 of request b and head h by one wave, a row at a time from its own keys alone, fp32 throughout (rare: it must not
// set the kernel's registers)
template <typename T, int D, int E, bool SIG>
__device__ __forceinline__ void prompt_rows_one_by_one(const LocalAttnArgs& a, int b, int h, int wq0, int lane) {
  const int qn = a.q_len[b], gk = h / (a.H / a.G);
  const int base_pos = (int)(a.seq_lens[b] - qn);
  const int32_t* row = a.req_to_token + a.req_pool_indices[b] * a.r2t_stride;
  const T* kp = (const T*)a.k_pool + (int64_t)gk * D;
  const T* vp = (const T*)a.v_pool + (a.v_shared ? 0 : (int64_t)gk * E) + lane;
  const ScoreMap smap(a.scale, a.cap);
  const float hb = (SIG && a.head_bias) ? a.head_bias[h] * kLog2e : 0.f;
#pragma unroll 1
  for (int r = wq0; r < qn && r < wq0 + 32; ++r) {
    const int pos = base_pos + r, lo = (int)range_lo(a, pos), n_first = (int)kept_before(a, lo), n = n_first + pos - lo + 1;
    const int64_t t = a.q_start[b] + r;
    const T* q = (const T*)a.q + t * a.q_ld + (int64_t)h * D;
    float m = -INFINITY, l = 0.f, acc[E / 64] = {};
#pragma unroll 1
    for (int i0 = 0; i0 < n; i0 += 64) {
      const bool there = i0 + lane < n;
      const int i = there ? i0 + lane : n - 1, slot = row[i < n_first ? i : lo + i - n_first];
      float dot = 0.f;
#pragma unroll 1
      for (int d = 0; d < D; d += 8) {
        const Vec16<T> qv = load16(q + d), kv = load16(kp + (int64_t)slot * a.k_ld + d);
#pragma unroll
        for (int u = 0; u < 8; ++u) dot += Elem<T>::to_f(qv.e[u]) * Elem<T>::to_f(kv.e[u]);
      }
      const float s = smap(dot);
      float p;
      if constexpr (SIG) {
        p = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(s + hb)));
      } else {
        const float m_new = fmaxf(m, wave_max(there ? s : -INFINITY)), m_use = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m - m_use);
        p = __builtin_amdgcn_exp2f(s - m_use);
        l = l * alpha + wave_sum(there ? p : 0.f);
#pragma unroll
        for (int u = 0; u < E / 64; ++u) acc[u] *= alpha;
        m = m_new;
      }
#pragma unroll 1
      for (int k = 0; k < 64 && i0 + k < n; ++k) {
        const float pk = __shfl(p, k, 64);
        const T* v = vp + (int64_t)__shfl(slot, k, 64) * a.v_ld;
#pragma unroll
        for (int u = 0; u < E / 64; ++u) acc[u] += pk * Elem<T>::to_f(v[64 * u]);
      }
    }
    if (!SIG && a.sink != nullptr) l += __builtin_amdgcn_exp2f(a.sink[h] * kLog2e - m);
    const float inv = SIG ? a.out_scale : a.out_scale / l;
    T* out = (T*)a.out + t * a.out_ld + (int64_t)h * E + lane;
#pragma unroll
    for (int u = 0; u < E / 64; ++u) {
      float y = acc[u] * inv;
      if (a.gate) y *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-kLog2e * Elem<T>::to_f(((const T*)a.gate)[t * a.gate_ld + (int64_t)h * E + lane + 64 * u])));
      out[64 * u] = Elem<T>::from_f(y);
    }
  }
}

// How the kv heads and tiles of a launch go to the 8 XCDs: 2^shift XCDs share `heads` heads, `tiles` tiles of a head each
struct PromptShare {
  uint32_t shift, heads, tiles;
};
__host__ __device__ inline PromptShare prompt_share(int G, uint32_t n_tiles) {
  const int pow2 = G & -G, groups = pow2 < 8 ? pow2 : 8;          // (of XCDs)
  const uint32_t shift = groups == 8 ? 0 : groups == 4 ? 1 : groups == 2 ? 2 : 3;
  return PromptShare{shift, (uint32_t)(G / groups), (n_tiles + (1u << shift) - 1) >> shift};
}

// Place `at` of a launch's tiles by their keys, the most first -> request and tile in it (-1: past the last): tiles of 2^shift rows, up to 8
// requests, a lane each (its tiles and the position of its first row).  Tile j of a request has u + j (mod period) tiles' rows of keys in
// front of it, u those of the request's first row, period a block's (0: no blocks).  So the tiles of a request with at least x are counted
// without a walk, and a lane counts them for each of up to 64 levels; within a level, request after request, neighbours next to each other.
struct PromptTile {
  int request, tile;
};
__device__ __forceinline__ PromptTile prompt_tile_by_keys(uint32_t at, int batch, int tiles, uint32_t pos, int shift, uint32_t period) {
  const int lane = threadIdx.x & 63;
  uint32_t u = pos >> shift, full = 0;
  uint32_t rem = u + tiles, top = period;
  if (period > 0) {
    u %= period;
    full = (u + tiles) / period;
    rem = u + tiles - full * period;
  } else {
    for (int r = 0; r < batch; ++r) top = max(top, (uint32_t)__builtin_amdgcn_readlane((int)rem, r));
  }
  const int per = (int)((top + 63) >> 6), x = lane * per;         // (tiles' rows between levels)
  int above = 0;                                                          // tiles with at least x in front
  for (int r = 0; r < batch; ++r)
    above += __builtin_amdgcn_readlane((int)full, r) * max((int)period - x, 0) + max(__builtin_amdgcn_readlane((int)rem, r) - x, 0) -
             max(__builtin_amdgcn_readlane((int)u, r) - x, 0);
  const int level = __builtin_popcountll(__ballot(above > (int)at)) - 1;
  if (level < 0) return PromptTile{-1, 0};
  int left = (int)at - (level < 63 ? __builtin_amdgcn_readlane(above, level + 1) : 0);
  const int lo = level * per, wid = period > 0 ? min(per, (int)period - lo) : per;
  const int skip = min(max((int)u - lo, 0), wid), mine = (int)full * wid + min(max((int)rem - lo, 0), wid) - skip;
  int r = 0;
  for (; r + 1 < batch; ++r) {
    const int n = __builtin_amdgcn_readlane(mine, r);
    if (left < n) break;
    left -= n;
  }
  left += __builtin_amdgcn_readlane(skip, r);
  const int block = left / wid;
  return PromptTile{r, block * (int)period + lo + (left - block * wid) - __builtin_amdgcn_readlane((int)u, r)};
}

template <typename T, int D, int E, int NW, int KT, int KS, bool SIG>
__global__ void __launch_bounds__(64 * NW * KS, 2) prompt_attention_kernel(LocalAttnArgs a, int hw, int by_keys, int runs) {
  constexpr int NT = 64 * NW, KU = KT / 32;                     // KT: keys a step; KS: groups of NW waves that take steps in turn
  constexpr int KB = D * 2, VB = E * 2, CK = D / 8, CV = E / 8;  // bytes and 16-byte chunks of a row
  constexpr int NK = KT * CK / NT, NV = KT * CV / NT;          // chunks a thread stages
  constexpr int KSW = CK < 16 ? CK - 1 : 15, VSW = E >= 128 ? 3 : 1;
  constexpr int ET = E / 32;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int group = KS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x / NT) : 0;
  uint8_t* const k_lds = lds + group * (2 * KT * (KB + VB));    // [2][KT][KB]
  uint8_t* const v_lds = k_lds + 2 * KT * KB;                   // [2][KT][VB]
  const int tid = threadIdx.x % NT, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31, hi = lane >> 5;
  // Workgroup -> (kv head, tile, heads of the group), the last fastest.  An XCD (workgroup ids go round the 8) has kv heads of its own, or
  // shares them with the fewest others, every so many tiles its own, or (runs) a run of them: workgroups that read the same K and V rows run
  // next to each other on one L2, and every XCD has as many long tiles.  Tiles from the last (most keys) to the first, or by their keys (by_keys).  A contiguous
  // range of all items an XCD gave the one with the ends of the longest prompts up to three times the work: 32 heads over 2 of 128, values
  // of 256, 1 prompt of 7000 tokens 1352 -> 776 us (whole call), 4 of 1900 389 -> 310.
  // (32 bits and shifts: with 64-bit quotients here and in the search for the request 20 tokens took 8.3 us for 7.4)
  const int hw_shift = 31 - __builtin_clz(hw), shift = 31 - __builtin_clz(32 * NW) - hw_shift, rows_wg = 1 << shift;      // (hw: a power of two)
  const uint32_t rep = a.H / a.G, sets = (rep + hw - 1) >> hw_shift, n_tiles = (uint32_t)a.n_tiles;
  const PromptShare share = prompt_share(a.G, n_tiles);
  const uint32_t of_set = (blockIdx.x >> 3) / sets, of_head = of_set / share.tiles, of_share = of_set - of_head * share.tiles, sharer = (blockIdx.x & 7) & ((1 << share.shift) - 1);
  const uint32_t tile_at = runs ? sharer * share.tiles + of_share : of_share << share.shift | sharer;
  const int set = (int)((blockIdx.x >> 3) - of_set * sets), gk = (int)(((blockIdx.x & 7) >> share.shift) * share.heads + of_head);
  if (tile_at >= n_tiles || of_head >= share.heads) return;
  const uint32_t tile_id = n_tiles - 1 - tile_at;
  // Its request: 64 at a time, a lane each, with all that is known of them in one round trip
  int b = -1, q0 = 0, qn = 0, base_pos = 0;
  int64_t t0 = 0, pool_row = 0;
  if (by_keys) {
    const int rq = min(lane, (int)a.batch - 1);
    const int n = a.q_len[rq], len = (int)a.seq_lens[rq], start = a.q_start[rq];
    const int64_t in_pool = a.req_pool_indices[rq];
    const int tiles = lane < (int)a.batch ? (max(n, 0) + rows_wg - 1) >> shift : 0;
    const PromptTile at = prompt_tile_by_keys(tile_at, (int)a.batch, tiles, tiles > 0 ? (uint32_t)(len - n) : 0u, shift, (uint32_t)a.chunk >> shift);
    if (at.request >= 0) {
      b = at.request;
      q0 = at.tile << shift;
      qn = __builtin_amdgcn_readlane(n, b);
      base_pos = __builtin_amdgcn_readlane(len, b) - qn;
      t0 = __builtin_amdgcn_readlane(start, b);
      pool_row = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)in_pool, b) | (int64_t)__builtin_amdgcn_readlane((int)(in_pool >> 32), b) << 32;
    }
  } else {
    int left = (int)tile_id;
    for (int rq0 = 0; rq0 < (int)a.batch && b < 0; rq0 += 64) {
      const int rq = min(rq0 + lane, (int)a.batch - 1);
      const int n = a.q_len[rq], len = (int)a.seq_lens[rq], at = a.q_start[rq];
      const int64_t in_pool = a.req_pool_indices[rq];
      const int tiles = rq0 + lane < (int)a.batch ? (max(n, 0) + rows_wg - 1) >> shift : 0;
      int upto = tiles;
#pragma unroll
      for (int d = 1; d < 64; d <<= 1) {
        const int below = __shfl_up(upto, d, 64);
        if (lane >= d) upto += below;
      }
      const uint64_t past = __ballot(left < upto);
      if (past != 0) {
        const int first = __builtin_ctzll(past);
        b = rq0 + first;
        q0 = (left - (__builtin_amdgcn_readlane(upto, first) - __builtin_amdgcn_readlane(tiles, first))) << shift;
        qn = __builtin_amdgcn_readlane(n, first);
        base_pos = __builtin_amdgcn_readlane(len, first) - qn;
        t0 = __builtin_amdgcn_readlane(at, first);
        pool_row = (int64_t)(uint32_t)__builtin_amdgcn_readlane((int)in_pool, first) | (int64_t)__builtin_amdgcn_readlane((int)(in_pool >> 32), first) << 32;
      } else {
        left -= __builtin_amdgcn_readlane(upto, 63);
      }
    }
  }
  if (b < 0) return;
  b = __builtin_amdgcn_readfirstlane(b);
  q0 = __builtin_amdgcn_readfirstlane(q0);
  const int hg = set * hw + (wave & (hw - 1));                  // head of the group (the last set may not be full)
  const bool h_ok = hg < (int)rep;
  const int h = gk * (int)rep + (h_ok ? hg : (int)rep - 1);
  const int keep = a.window > 0 ? a.keep_first : 0;
  const int wg_last = min(q0 + rows_wg, qn) - 1;
  const int key_lo = (int)range_lo(a, base_pos + q0), key_hi = base_pos + wg_last;
  // this wave's 32 rows
  const int wq0 = q0 + 32 * (wave >> hw_shift);
  const bool wave_on = wq0 < qn && h_ok;
  const int wq_last = min(wq0 + 31, qn - 1);
  const int w_first = base_pos + wq0, w_hi = base_pos + wq_last;
  const int w_lo = (int)range_lo(a, w_first), w_full = (int)range_lo(a, w_hi);     // first key that any / every row of the wave sees
  const bool q_ok = wq0 + col < qn;
  const int my_q = q_ok ? wq0 + col : (wave_on ? wq_last : 0);
  const int my_pos = q_ok ? base_pos + my_q : -1, my_lo = (int)range_lo(a, base_pos + my_q);
  Frag16 qf[D / 16];
  {
    const T* q = (const T*)a.q + (t0 + my_q) * a.q_ld + (int64_t)h * D + hi * 8;
#pragma unroll
    for (int ks = 0; ks < D / 16; ++ks) qf[ks].u = *reinterpret_cast<const uint4*>(q + ks * 16);
  }
  f32x16 o[ET];
#pragma unroll
  for (int t = 0; t < ET; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[t][r] = 0.f;
  float m = -INFINITY, l = 0.f;
  const ScoreMap smap(a.scale, a.cap);
  const bool capped_scores = smap.A != 0.f;
  const float c = capped_scores ? 1.0f : smap.c;                // what multiplies a score in the exponent
  const float hb = (SIG && a.head_bias) ? a.head_bias[h] * kLog2e : 0.f;

  // the walk: the kept first positions in front of the tile's range, then the range; steps of 64 keys, each within one of the two
  const int n_first = keep < key_lo ? keep : key_lo;
  const int first_steps = (n_first + KT - 1) / KT, steps = first_steps + (key_hi - key_lo) / KT + 1;
  const int32_t* row = a.req_to_token + pool_row * a.r2t_stride;
  const int kr0 = tid / CK, kc = tid % CK, vr0 = tid / CV, vc = tid % CV;      // this thread's chunks: rows kr0 + i NT / CK, chunk kc
  const char* kp = (const char*)((const T*)a.k_pool + (int64_t)gk * D + kc * 8);
  const char* vp = (const char*)((const T*)a.v_pool + (a.v_shared ? 0 : (int64_t)gk * E) + vc * 8);
  const uint32_t k_row = (uint32_t)a.k_ld * 2u, v_row = (uint32_t)a.v_ld * 2u;       // (bytes between rows: 32 bits, see prompt_attention)
  uint32_t k_slot[NK] = {}, v_slot[NV] = {};
  u32x4 kv[NK], vv[NV];
  auto load_slots = [&](int it) {
    const bool first = it < first_steps;
    const int j0 = first ? it * KT : key_lo + (it - first_steps) * KT, last = first ? n_first - 1 : key_hi;
#pragma unroll
    for (int i = 0; i < NK; ++i) k_slot[i] = row[min(j0 + kr0 + i * (NT / CK), last)];       // (past the end: the last key, masked)
#pragma unroll
    for (int i = 0; i < NV; ++i) v_slot[i] = CV == CK ? k_slot[i < NK ? i : 0] : row[min(j0 + vr0 + i * (NT / CV), last)];
  };
  auto load_rows = [&]() {
#pragma unroll
    for (int i = 0; i < NK; ++i) kv[i] = *reinterpret_cast<const u32x4*>(kp + (uint64_t)k_slot[i] * k_row);
#pragma unroll
    for (int i = 0; i < NV; ++i) vv[i] = *reinterpret_cast<const u32x4*>(vp + (uint64_t)v_slot[i] * v_row);
  };
  auto store_rows = [&](int buf) {
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int r = kr0 + i * (NT / CK);
      *reinterpret_cast<u32x4*>(k_lds + buf * KT * KB + r * KB + ((kc ^ (r & KSW)) << 4)) = kv[i];
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int r = vr0 + i * (NT / CV);
      *reinterpret_cast<u32x4*>(v_lds + buf * KT * VB + r * VB + ((vc ^ ((r & VSW) << 2)) << 4)) = vv[i];
    }
  };
  // operand addresses: K row `col` (+ 32), chunk 2 ks + hi; V rows 4 hi + gi / 4 (+ 8, + 16 s), columns 32 t + 16 g1 + 4 (gi & 3)
  const int gi = lane & 15, g1 = (lane >> 4) & 1, vrow = 4 * hi + (gi >> 2);
  const uint8_t* ka = k_lds + col * KB;
  const uint8_t* va = v_lds + vrow * VB + g1 * 32 + (gi & 3) * 8;
  const int kx = col & KSW, vx = vrow & VSW;

  load_slots(group);                                            // (a step behind the last: the last key)
  load_rows();
  if (group + KS < steps) load_slots(group + KS);
  store_rows(0);
  __syncthreads();
  for (int it = group, buf = 0; it - group < steps; it += KS, buf ^= 1) {
    auto fetch = [&]() __attribute__((always_inline)) {
      if (it + KS < steps) {
        load_rows();
        if (it + 2 * KS < steps) load_slots(it + 2 * KS);
      }
    };
    // (value rows of 256 in two groups: the next rows are asked for behind the first products, whose operands the registers hold until then: 1
    // prompt of 600 tokens 41.5 -> 36.7 us; 1 .. 4 % slower elsewhere)
    constexpr bool late = E > 128 && KS > 1;
    if (!late) fetch();
    const bool first = it < first_steps;
    const int j0 = first ? it * KT : key_lo + (it - first_steps) * KT;
    // 0: no row of the wave sees a key of the step; 2: every row sees all of them
    const bool some = wave_on && (KS == 1 || it < steps) && (first || (j0 <= w_hi && (j0 + KT - 1 >= w_lo || j0 < keep)));
    if (late && !some) fetch();
    if (some) {
      const uint8_t* kb = ka + buf * KT * KB;
      const uint8_t* vb = va + buf * KT * VB;
      f32x16 s[KU] = {};
#pragma unroll
      for (int ks = 0; ks < D / 16; ++ks) {
        Frag16 kf[KU];
#pragma unroll
        for (int u = 0; u < KU; ++u) kf[u].u = *reinterpret_cast<const uint4*>(kb + u * 32 * KB + (((2 * ks + hi) ^ kx) << 4));
#pragma unroll
        for (int u = 0; u < KU; ++u) s[u] = Mfma<T>::mma(as_frag<T>(kf[u]), as_frag<T>(qf[ks]), s[u]);
      }
      // rows of K three products ahead (left alone, they are read one at a time, the latency of LDS behind each: 1116 cycles a step of a
      // wave for these, so 834)
      __builtin_amdgcn_sched_group_barrier(0x100, 3 * KU, 0);
#pragma unroll
      for (int i = 0; i < D / 16 - 3; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, KU, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, KU, 0);
      }
      __builtin_amdgcn_sched_group_barrier(0x008, 3 * KU, 0);
      if (late) {
        __builtin_amdgcn_sched_barrier(0);
        fetch();
      }
      if (capped_scores)
#pragma unroll
        for (int u = 0; u < KU; ++u)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[u][r] = smap(s[u][r]);
      const bool whole = first ? j0 + KT <= n_first : (j0 + KT - 1 <= w_first && j0 >= w_full);
      if (!whole) {
        // (row (r & 3) + 8 (r >> 2) + 4 hi of a 32-key block)
        const int top = (first ? (q_ok ? n_first - 1 : -1) : my_pos) - j0 - 4 * hi, from = first ? -KT : my_lo - j0 - 4 * hi, kept = first ? 0 : keep - j0 - 4 * hi;
#pragma unroll
        for (int u = 0; u < KU; ++u)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int j = 32 * u + (r & 3) + 8 * (r >> 2);
            s[u][r] = j <= top && (j >= from || j < kept) ? s[u][r] : -INFINITY;
          }
      }
      Frag16 p[2 * KU];                                              // keys 16 s + {0 .. 3, 8 .. 11} + 4 hi of this lane's column
      float m_of[KU], l_next = 0.f;                                  // running maximum behind every 32 keys, the second 32's share of l
      auto rescale = [&](float by) {
        l *= by;
#pragma unroll
        for (int t = 0; t < ET; ++t)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[t][r] *= by;
      };
      if constexpr (SIG) {
        // independent weights sigmoid(score + hb), base 2: a masked key has score -inf: exp2(+inf) = inf, 1 / inf = 0
#pragma unroll
        for (int u = 0; u < KU; ++u)
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const float p0 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-fmaf(s[u][r], c, hb)));
            const float p1 = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-fmaf(s[u][r + 1], c, hb)));
            p[2 * u + (r >> 3)].w[(r & 7) >> 1] = pack2<T>(p0, p1);
          }
      } else {
        float mx[KU];
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          mx[u] = s[u][0];
#pragma unroll
          for (int r = 1; r < 16; ++r) mx[u] = fmaxf(mx[u], s[u][r]);
          const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx[u]), __float_as_uint(mx[u]), false, false);
          mx[u] = fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])) * c;        // (c > 0; -inf stays -inf)
        }
        if (__any(mx[0] > m)) {
          const float m_new = fmaxf(m, mx[0]);
          rescale(m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new));
          m = m_new;
        }
        m_of[0] = m;
        if constexpr (KU == 2) m = m_of[1] = fmaxf(m, mx[1]);
        float sum[KU] = {};
#pragma unroll
        for (int u = 0; u < KU; ++u) {
          const float m_use = m_of[u] == -INFINITY ? 0.f : m_of[u];
#pragma unroll
          for (int r = 0; r < 16; r += 2) {
            const float p0 = __builtin_amdgcn_exp2f(fmaf(s[u][r], c, -m_use)), p1 = __builtin_amdgcn_exp2f(fmaf(s[u][r + 1], c, -m_use));
            sum[u] += p0 + p1;
            p[2 * u + (r >> 3)].w[(r & 7) >> 1] = pack2<T>(p0, p1);
          }
        }
        l += sum[0];
        if constexpr (KU == 2) l_next = sum[1];
      }
      if constexpr (KU == 1) {
        // Operands of V three ahead of their products (left alone, they are read one at a time, the latency of LDS in front of each product; with
        // steps of 64 and two workgroups a CU the other one covers that, and the registers are worth more: 1 .. 2 % slower so).  32 / 2 heads
        // with value rows of 256 behind a mix of heads, 4 prompts of 1900 tokens, whole call, 288 -> 262 us, 1 of 7000 753 -> 690; the exponentials
        // go between the products.
        constexpr int NF = 2 * KU * ET, VA = 3;                       // operands; how many are ahead
        Frag16 vf[VA];
        auto load_v = [&](int f, Frag16& x) __attribute__((always_inline)) {
          const uint8_t* vq = vb + (f / ET) * 16 * VB + (((f % ET) ^ vx) << 6);
          x.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vq));
          x.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vq + 8 * VB));
        };
#pragma unroll
        for (int f = 0; f < VA; ++f) load_v(f, vf[f]);
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          o[f % ET] = Mfma<T>::mma(as_frag<T>(vf[f % VA]), as_frag<T>(p[f / ET]), o[f % ET]);
          if (f + VA < NF) load_v(f + VA, vf[f % VA]);
        }
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * VA, 0);
#pragma unroll
        for (int i = 0; i < NF - VA; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x008, VA, 0);
      } else {
#pragma unroll
        for (int s4 = 0; s4 < 2 * KU; ++s4) {
          if constexpr (!SIG && KU == 2)
            if (s4 == 2) {
              if (__any(m_of[1] > m_of[0])) rescale(m_of[0] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_of[0] - m_of[1]));
              l += l_next;
            }
#pragma unroll
          for (int t = 0; t < ET; ++t) {
            Frag16 vf;
            const uint8_t* vq = vb + s4 * 16 * VB + ((t ^ vx) << 6);
            vf.s[0] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vq));
            vf.s[1] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vq + 8 * VB));
            o[t] = Mfma<T>::mma(as_frag<T>(vf), as_frag<T>(p[s4]), o[t]);
          }
        }
      }
    }
    if (it + KS < steps) store_rows(buf ^ 1);
    __syncthreads();                                            // the next step's rows are in place, everyone is done with this step's
  }
  // the groups' sums, by way of LDS (the walk ended on a barrier)
  constexpr int MERGE = ET * 4096 + 512;                        // bytes of a wave
  if constexpr (KS > 1) {
    if (steps > 1) {
      if (group > 0) {
        float* const ml = reinterpret_cast<float*>(lds + ((group - 1) * NW + wave) * MERGE);
#pragma unroll
        for (int t = 0; t < ET; ++t)
#pragma unroll
          for (int r = 0; r < 16; r += 4) *reinterpret_cast<f32x4*>(ml + (4 * t + r / 4) * 256 + 4 * lane) = f32x4{o[t][r], o[t][r + 1], o[t][r + 2], o[t][r + 3]};
        ml[ET * 1024 + lane] = m;
        ml[ET * 1024 + 64 + lane] = l;
      }
      __syncthreads();
    }
    if (group > 0) return;
    for (int other = 1; other < KS && other < steps; ++other) {
      const float* const ml = reinterpret_cast<const float*>(lds + ((other - 1) * NW + wave) * MERGE);
      float f0 = 1.f, f1 = 1.f;
      if constexpr (!SIG) {
        const float m1 = ml[ET * 1024 + lane], m0 = m;
        m = fmaxf(m0, m1);
        f0 = m0 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m0 - m);
        f1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - m);
        l = fmaf(l, f0, ml[ET * 1024 + 64 + lane] * f1);
      }
#pragma unroll
      for (int t = 0; t < ET; ++t)
#pragma unroll
        for (int r = 0; r < 16; r += 4) {
          const f32x4 v = *reinterpret_cast<const f32x4*>(ml + (4 * t + r / 4) * 256 + 4 * lane);
#pragma unroll
          for (int u = 0; u < 4; ++u) o[t][r + u] = SIG ? o[t][r + u] + v[u] : fmaf(o[t][r + u], f0, v[u] * f1);
        }
    }
  }
  if constexpr (!SIG) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    if (a.sink != nullptr) l += __builtin_amdgcn_exp2f(a.sink[h] * kLog2e - m);
  }
  if (!wave_on) return;
  {
    float z[4] = {};
#pragma unroll
    for (int t = 0; t < ET; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) z[r & 3] = fmaf(o[t][r], 0.f, z[r & 3]);
    if (__any(!((z[0] + z[1]) + (z[2] + z[3]) == 0.f))) {
      auto args = (const __attribute__((address_space(4))) void*)__builtin_amdgcn_kernarg_segment_ptr();
      int b1 = b, h1 = h, row1 = wq0, lane1 = lane;
      asm volatile("" : "+s"(args), "+s"(b1), "+s"(h1), "+s"(row1), "+v"(lane1));      // (read and computed again, not held over the walk)
      LocalAttnArgs again;
      __builtin_memcpy(&again, (const void*)args, sizeof(again));
      prompt_rows_one_by_one<T, D, E, SIG>(again, b1, h1, row1, lane1);
      return;
    }
  }
  const float inv = q_ok ? (SIG ? a.out_scale : a.out_scale / l) : 0.f;
  // out through the wave's part of the tiles (the walk ended on a barrier): a lane holds four neighbouring elements of one row at a
  // time, rows leave in 16-byte pieces of consecutive lanes
  constexpr int OS = E * 2 + 16;
  static_assert(32 * OS <= MERGE, "a wave leaves by way of what it has merged");
  uint8_t* ol = lds + wave * (KS == 1 ? 32 * OS : MERGE);
#pragma unroll
  for (int t = 0; t < ET; ++t)
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
      uint2 w;
      w.x = pack2<T>(o[t][r] * inv, o[t][r + 1] * inv);
      w.y = pack2<T>(o[t][r + 2] * inv, o[t][r + 3] * inv);
      *reinterpret_cast<uint2*>(ol + col * OS + (32 * t + 2 * r + 4 * hi) * 2) = w;
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll 4
  for (int i = lane; i < 32 * CV; i += 64) {
    const int rr = i / CV, ec = i % CV;
    if (wq0 + rr >= qn) break;
    Vec16<T> v = *reinterpret_cast<const Vec16<T>*>(ol + rr * OS + ec * 16);
    const int64_t t = t0 + wq0 + rr;
    if (a.gate) {
      const Vec16<T> gv = load16((const T*)a.gate + t * a.gate_ld + (int64_t)h * E + ec * 8);
#pragma unroll
      for (int u = 0; u < 8; ++u)
        v.e[u] = Elem<T>::from_f(Elem<T>::to_f(v.e[u]) * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-kLog2e * Elem<T>::to_f(gv.e[u]))));
    }
    store16((T*)a.out + t * a.out_ld + (int64_t)h * E + ec * 8, v);
  }
}

// true: launched.  Head sizes 64 / 64, 64 / 128, 128 / 128, 128 / 256 (sigmoid weights: 64 / 64, 128 / 128), a positive scale, 16-bit
// types, everything aligned as local_attention_mfma_kernel wants it.
struct PromptPlan {
  int hw;
  int64_t avg, n_tiles, blocks, expected;          // expected: workgroups that find a tile where half of the requests end in one of few rows
  PromptShare share;
};
static PromptPlan prompt_plan(const LocalAttnArgs& a, int NW) {
  const int rep = a.H / a.G;
  // heads of a group in a workgroup: the largest power of two that divides them, or the next one above them (the last set's waves are not all
  // busy) where that makes fewer workgroups of requests of the average length.  24 / 8 heads, 32 requests of 20 tokens: one head and room
  // for 128 rows a workgroup 14.2 us, the three heads of a group 8.5; the same with 1900 tokens keeps the 128 rows.
  int hw = NW, wide = 1;
  while (rep % hw) hw >>= 1;
  while (wide < rep && wide < NW) wide <<= 1;
  const int64_t avg = (a.num_tokens + a.batch - 1) / a.batch;
  const auto count = [&](int w) { return (avg + 32 * (NW / w) - 1) / (32 * (NW / w)) * ((rep + w - 1) / w); };
  if (count(wide) < count(hw)) hw = wide;
  const int rows = 32 * (NW / hw);
  const int64_t n_tiles = (a.num_tokens + rows - 1) / rows + a.batch;
  const PromptShare share = prompt_share(a.G, (uint32_t)n_tiles), likely = prompt_share(a.G, (uint32_t)(n_tiles - a.batch + (a.batch - 1) / 2));
  const int64_t sets = 8ll * share.heads * ((rep + hw - 1) / hw);
  return PromptPlan{hw, avg, n_tiles, share.tiles * sets, likely.tiles * sets, share};
}
template <typename T, int D, int E, int NW, int KT, int KS, bool SIG>
static int launch_prompt_attention(LocalAttnArgs a, const PromptPlan& plan, hipStream_t s) {
  const int rep = a.H / a.G, hw = plan.hw, rows = 32 * (NW / hw);
  const int64_t avg = plan.avg, blocks = plan.blocks;
  const PromptShare share = plan.share;
  a.n_tiles = plan.n_tiles;
  constexpr size_t tiles = KS * 2 * KT * (size_t)(D + E) * 2, epilogue = NW * (KS > 1 ? (KS - 1) * (size_t)(E * 128 + 512) : 32 * (size_t)(E * 2 + 16)), bytes = tiles > epilogue ? tiles : epilogue;
  static std::atomic<uint64_t> done{0};
  if (ensure_dynamic_lds((const void*)prompt_attention_kernel<T, D, E, NW, KT, KS, SIG>, bytes, done, "local_attention")) return SEMIPD_EINVAL;
  // Tiles by their keys where they differ by blocks or by requests (one sequence without blocks is in that order anyway, and windows make
  // most tiles alike) and the launch is between one (two) and eight times what the chip takes at once: below that all start together, above
  // the end of the launch is little of it. (Blocks of a few steps: a tile's start and end are most of its time, and all are nearly alike.)
  // Whole call, last tile first / by keys, us: 32 / 8 heads of 128, blocks of 1024, 4 prompts of 1900 tokens 107.5 / 97.7, 2 of 1500 46.4 /
  // 38.5, 1 of 16000 217.7 / 211.1, 4 of 6000 (12 times) 337 / 338; 24 / 8 heads, blocks of 256, 4 of 1900 45.8 / 44.3, 2 of 1500 21.6 /
  // 25.0; without blocks 2 of 3000 168 / 154, 2 of 1500 (1.5 times) 52.6 / 53.9, 16 of 500 (each workgroup asks for all 16) 83.8 / 86.8;
  // values of 256, 2 heads, 2 of 3000 326 / 299.
  const int64_t at_once = 256 * 8 / (NW * KS);
  const bool by_keys = a.window == 0 && a.batch <= 8 && (a.chunk > 0 ? a.chunk >= 512 && a.chunk % rows == 0 && blocks > at_once : a.batch > 1 && blocks > 2 * at_once) &&
                       blocks <= 8 * at_once;
  // A run of tiles an XCD where tiles next to each other read the same few keys and are nearly alike: blocks of up to 256 of a few requests, and
  // more than 8 requests whose heads all XCDs share (an odd number of kv heads), all of more than a few tiles; not where the launch is hardly
  // more than the chip takes at once, since the tiles that do not exist (n_tiles is a bound) are the first XCD's then.  Every so many
  // tiles / runs, whole call, us: 24 / 3 heads, blocks of 256, 1 prompt of 6000 44.2 / 36.1; 16 / 2 heads, 3 of 1700 27.8 / 21.8; 28 / 7 heads, 8
  // of 800 46.6 / 42.6; without blocks 8 / 1 heads, 20 of 300 22.8 / 20.2, 20 / 5 heads of 64, 9 of 700 42.4 / 39.8; but 32 / 4 heads, 9 of 700 73 / 81,
  // blocks of 256, 28 / 4 heads, 9 of 700 45 / 50, 12 of 120 15.4 / 24, windows of 1000, 24 / 3 heads, 8 of 800 69.5 / 70.4.
  const int64_t over = blocks / 8 - at_once / 8, few = (int64_t)share.heads * ((rep + hw - 1) / hw) * ((a.batch + 7) / 8);
  const int64_t bound = a.window > 0 ? a.window : a.chunk;
  const bool runs = !by_keys && avg >= 256 && !(over > 0 && over <= few) &&
                    (a.batch <= 8 ? a.chunk > 0 && a.chunk <= 256 : share.shift == 3 && (bound == 0 || bound > 256));
  hipLaunchKernelGGL((prompt_attention_kernel<T, D, E, NW, KT, KS, SIG>), dim3((unsigned)blocks), dim3(64 * NW * KS), bytes, s, a, hw, (int)by_keys, (int)runs);
  return 0;
}
// Launches of at most a workgroup a CU are as long as their longest tile, a chain of steps at 1.7 us with a wave on every SIMD and 2.7 with
// two: tiles of 64 rows and heads whose steps four groups of two waves take in turn, then of 128 and two groups of four, as long as every
// tile has a CU of its own; not where all walks are short, which gain nothing from it.  (Behind that a CU has the second wave from another
// tile.)  One / two / four groups, whole call, us: 32 / 8 heads of 128, 1 prompt of 300 tokens 15.4 / 15.5 / 14.2, of 600 23.6 / 21.4 / 21.9
// (320 tiles), of 933 33.0 / 30.0 / 32.3 (480), 30 tokens behind 900 30.6 / 27.0 / 21.9, 2 of 339 behind 104 21.3 / 19.4 / 23.5 (384); 24 / 8 heads, 1 of
// 600 24.5 / 21.3 / 18.3; 32 / 8 of 64, 30 behind 900 22.2 / 19.6 / 15.6; blocks of 128, 1 of 933 13.0 / 13.9 / 22.4, of 256, 1 of 600 14.9 / 14.8 / 19.3.  Values
// of 256 (the second form of 512 against eight waves in one group): 1 of 600 51.8 / 45.2, 1 of 933 72 / 62, 7 of 101 24.9 / 24.5.
// Up to two tiles a CU where they differ most, in one or two requests whose rows see all in front of them: two tiles at once take as long as
// the longer one, one behind the other (the longest first) as their mean.  One / two groups: 32 / 8 heads of 128, 1 prompt of 1500 tokens 50.1 / 42.6, 2 of
// 1000 38.4 / 36.4 (24 / 8 heads 48.5 / 39.9, 37.1 / 31.7; of 64 34.1 / 28.0, 26.6 / 24.5), values of 256, 1 of 1500 107 / 91; but windows of 1000, 1 of 2000 49.8
// / 60.6, 4 of 300 19.6 / 23.8, values of 128 and keys of 64, 2 of 1086 46.8 / 48.6; beyond, 1 of 3000 103 / 111.  Short tiles have more start and end than
// that gives back where they are many: 40 / 8 heads of 128, 2 of 600 (440 tiles) 26.3 / 27.9, 32 / 8, 2 of 600 (288) 24.3 / 21.2.
// On a share of the CUs the same by the share's, and by the tiles that are likely there.  One group / the former rule, which counted on 256 / this, on 224
// CUs: 32 / 8 heads of 128, 2 prompts of 1000 36.3 / 39.2 / 36.2, 4 of 100 behind 800 35.3 / 23.4 / 23.5; on 192, 2 of 1000 36.3 / 43.8 / 36.2, 24 / 8 heads 35.4 / 39.6 /
// 35.4; on 128, 1 of 300 14.6 / 18.7 / 14.7, 1 of 1500 57.3 / 71.7 / 57.3.  Two tiles a CU, one / two groups, of one request: on 192 CUs 1 of 1500 47.9 / 46.7, on 128
// 1 of 933 32.9 / 35.6; of two: on 224 2 of 1000 (24 / 8 heads) 36.4 / 35.0, on 160 2 of 600 26.1 / 28.9.
template <typename T, int D, int E, bool SIG>
static int split_prompt_attention(const LocalAttnArgs& a, hipStream_t s) {
  constexpr int NW = E > 128 ? 8 : 4, KT = E > 128 ? 32 : 64;
  const int64_t bound = a.window > 0 ? a.window : a.chunk, cus = std::min<int64_t>(launch_cus(), 256);
  const auto fits = [&](const PromptPlan& p) { return p.blocks <= 256 && p.expected <= cus; };
  if (bound == 0 || bound >= 512) {
    if constexpr (E <= 128) {
      const PromptPlan few = prompt_plan(a, 2);
      if (fits(few)) return launch_prompt_attention<T, D, E, 2, (D + E > 128 ? 32 : 64), 4, SIG>(a, few, s);
    }
    const PromptPlan few = prompt_plan(a, 4);
    const bool uneven = (a.batch == 1 ? cus >= 160 : a.batch == 2 && E == D && cus >= 224) && (a.window == 0 || a.window >= few.avg);
    if (fits(few) || (uneven && few.blocks <= 2 * cus && (few.blocks <= 384 || few.avg >= 800))) return launch_prompt_attention<T, D, E, 4, KT, 2, SIG>(a, few, s);
  }
  return launch_prompt_attention<T, D, E, NW, KT, 1, SIG>(a, prompt_plan(a, NW), s);
}
template <typename T>
static bool prompt_attention(const LocalAttnArgs& a, hipStream_t s, int& rc) {
  const bool sig = a.sigmoid != 0;
  if (!(a.scale > 0.f) || a.k_ld <= 0 || a.v_ld <= 0 || a.k_ld >= (1ll << 31) || a.v_ld >= (1ll << 31)) return false;
  if (a.D == 128 && a.E == 128) rc = sig ? split_prompt_attention<T, 128, 128, true>(a, s) : split_prompt_attention<T, 128, 128, false>(a, s);
  else if (a.D == 64 && a.E == 64) rc = sig ? split_prompt_attention<T, 64, 64, true>(a, s) : split_prompt_attention<T, 64, 64, false>(a, s);
  else if (a.D == 64 && a.E == 128 && !sig) rc = split_prompt_attention<T, 64, 128, false>(a, s);
  else if (a.D == 128 && a.E == 256 && !sig) rc = split_prompt_attention<T, 128, 256, false>(a, s);
  else return false;
  return true;
}

}  // namespace semipd
