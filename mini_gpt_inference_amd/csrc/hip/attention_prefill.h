// The body of the attention kernel for prompt portions (attention_prefill.hip says what it does and why), for that kernel and
// for the one that also has a step's single tokens (attention_mixed.hip).
#pragma once
#include "attention_mask.h"
#include "common.h"

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short bf16x4_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned int)))) unsigned int u32x4_t;

#define PF_W 32       // queries of a wave, and keys of a wave and step
#define PF_PAGES 768  // block-table entries in LDS
// Buffers of keys and values: a stretch is asked for a step ahead (two or three steps ahead, 2 x 1,024 tokens x 8 heads: 16.7 to
// 17.1 us for 16.7).
#define PF_BUFS 2

// max over the lanes lane and lane ^ 32, the same in both: the swap hands every lane its partner's value.
__device__ __forceinline__ float pf_max_of_pair(float v) {
  const unsigned int u = __float_as_uint(v);
  const auto b = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// Where 16-byte chunk c of LDS row `row` lies within the row: chunks XORed with bits of the row, so that neither the operand
// reads (32 rows, one chunk each) nor the transposing ones (4 rows, 64 bytes each) meet in a bank.
template <int D>
__device__ __forceinline__ int pf_chunk(int row, int c) {
  if (D == 128) return c ^ (((row & 3) << 2) | ((row >> 2) & 3));
  if (D == 64) return c ^ (((row & 2) << 1) | ((row & 4) >> 1) | ((row & 8) >> 3));
  return c ^ ((row >> 2) & 3);   // rows of 64 and 192 bytes
}

// Waves a SIMD that it is built for (128 registers, or 256).
template <int D, int K>
constexpr int pf_waves() { return D <= 64 && K < 4 ? 4 : 2; }

// Bytes of LDS that it takes.
template <int D, int Q, int K, int BIAS>
constexpr int pf_lds_bytes() {
  constexpr int sb = K * PF_W, staged = PF_BUFS * 2 * sb * D * (int)sizeof(bf16_t);
  constexpr int shared = Q * K * 64 * (2 + D / 2) * 4;   // what the key groups put together at the end
  return (staged > shared ? staged : shared) + PF_PAGES * 4 + (BIAS == 1 ? 2 * (sb + Q * PF_W) * 4 : 0);
}

// Tile `tile` of request r, head h: 32 Q queries.
//
// Q waves of 32 queries each, times K groups that share the keys: of every stretch of 32 K keys that is staged at a time a
// group has 32, with a running max, sum and output of its own that are put together at the end.
template <int D, int Q, int K, int BIAS>
__device__ __forceinline__ void pf_tile(
    const bf16_t* __restrict__ q, long ldq, bf16_t* __restrict__ out, long ldo,
    const bf16_t* __restrict__ kpool, const bf16_t* __restrict__ vpool,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ cu_q,
    const int* __restrict__ seq_lens, int n_head, int n_kv_head, int page_size, float scale, int window,
    int single_below, const float* __restrict__ sinks, float softcap, const bf16_t* __restrict__ gate, long ldg,
    int keep_first, const float* __restrict__ score_bias, int chunked, const float* __restrict__ dist_bias,
    int bias_len, const float* __restrict__ slopes, int tile, int r, int h,
    bf16_t* __restrict__ pf_lds) {
  constexpr int WAVES = Q * K, THREADS = 64 * WAVES, QT = Q * PF_W;
  constexpr int SB = K * PF_W;     // keys staged per step
  constexpr int BUFS = PF_BUFS, AHEAD = BUFS - 1;
  constexpr int KK = D / 16;       // MFMA k steps over the head size
  constexpr int CT = D / 32;       // 32-channel tiles of the output
  constexpr int CH = D / 8;        // 16-byte chunks of a row
  constexpr bool EARLY = pf_waves<D, K>() == 2;
  constexpr int LOADS = SB * CH / 64 / WAVES;   // a wave's 1 KB pieces of a stretch's keys (and as many of its values)
  static_assert(SB * CH % (64 * WAVES) == 0, "the stretch's chunks must divide among the waves");
  // pf_lds: [BUFS][2][SB][D] keys, values; then the block table's entries
  // The block-table entries of the keys that the tile sees lie in LDS before the first stretch is asked for (of longer contexts
  // PF_PAGES at a time), so that no load from memory stands between those of two stretches and steps can be asked for ahead.
  constexpr int STAGED = pf_lds_bytes<D, Q, K, 0>() / (int)sizeof(bf16_t) - PF_PAGES * 2;
  int* const pages = reinterpret_cast<int*>(pf_lds + STAGED);
  // entry e of a buffer: the number (times log2 e) for distance tile_pos_hi - first key of the stretch - e
  constexpr int NB = SB + QT;
  float* const bias_tab = reinterpret_cast<float*>(pages + PF_PAGES);  // [2][NB]

  const int q_start = cu_q[r], q_len = cu_q[r + 1] - q_start;
  const int q0 = tile * QT;
  if (q0 >= q_len || (q_len == 1 && q_start < single_below)) return;   // the same for the whole workgroup
  const int seq_len = seq_lens[r];
  const int ctx = seq_len - q_len;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qw = wave % Q, kg = wave / Q;
  const int hk = h / (n_head / n_kv_head);
  const int* bt = block_tables + (long)r * max_blocks;
  const int l31 = lane & 31, g = lane >> 5;

  // this lane's query (for masks and the final store) and the tile's key range
  const int my_q = q0 + qw * 32 + l31;
  const bool q_ok = my_q < q_len;
  const int my_pos = ctx + my_q;
  const int tile_q_hi = (q0 + QT < q_len ? q0 + QT : q_len) - 1;
  const int pos_lo = ctx + q0, pos_hi = ctx + tile_q_hi;
  const int kv_begin = first_seen(pos_lo, window, chunked);
  const int my_begin = first_seen(my_pos, window, chunked);
  const int kv_end = pos_hi + 1;
  // the wave's queries: positions wave_lo .. wave_hi (none of them: wave_hi < wave_lo)
  const int wave_lo = pos_lo + qw * 32, wave_hi = wave_lo + 31 < pos_hi ? wave_lo + 31 : pos_hi;
  const int wave_begin = first_seen(wave_lo, window, chunked);
  const int wave_begin_hi = first_seen(wave_lo + 31, window, chunked);   // what the wave's last query sees from

  bf16x8_t qf[KK];
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
  for (int kk = 0; kk < KK; ++kk)
    qf[kk] = q_ok ? *reinterpret_cast<const bf16x8_t*>(q + (long)(q_start + my_q) * ldq + (long)h * D + kk * 16 + g * 8)
                  : zero8;

  float m = -INFINITY, l = 0.f;   // m in units of log2 e; l: this lane's share of the row sum
  f32x16_t o[CT];
#pragma unroll
  for (int ct = 0; ct < CT; ++ct)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[ct][i] = 0.f;

  typedef __attribute__((address_space(1))) const void* global_ptr_t;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  // scores are kept in units of log2(e), so that the exponential is one v_exp_f32 (scale > 0 here; with numbers
  // by distance the scores are scaled when those are added)
  const float raw2 = scale * 1.4426950408889634f;
  const float sc2 = BIAS ? 1.0f : raw2;
  const float slope2 = BIAS == 2 ? slopes[h] * 1.4426950408889634f : 0.f;
  const bool weigh = score_bias != nullptr;   // sigmoid weights, no softmax
  const float bias2 = weigh ? score_bias[h] * 1.4426950408889634f : 0.f;
  if (weigh) m = 0.f;
  const int c_first = (kv_begin / SB) * SB;
  // the stretches of the kept first keys (those before the window's first stretch), then the window's
  const int kept_steps = keep_first > 0 ? ((keep_first + SB - 1) / SB < c_first / SB ? (keep_first + SB - 1) / SB : c_first / SB) : 0;
  const int n_steps = kept_steps + (kv_end - c_first + SB - 1) / SB;
  auto stretch_start = [&](int step) -> int { return step < kept_steps ? step * SB : c_first + (step - kept_steps) * SB; };
  auto fill_bias = [&](int step) {
    const int c_start = stretch_start(step);
    for (int e = tid; e < NB; e += THREADS)
      bias_tab[(step & 1) * NB + e] =
          dist_bias[(long)h * bias_len + distance_entry(pos_lo + QT - 1 - c_start - e, bias_len)] * 1.4426950408889634f;
  };
  // Entries are numbered over the kept stretches' pages and then the window's: slot `first_slot + i` lies in pages[i].
  const int page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
  auto page_of = [&](int j) -> int { return page_shift >= 0 ? j >> page_shift : j / page_size; };
  const int kept_pages = kept_steps > 0 ? page_of(kept_steps * SB - 1) + 1 : 0, window_page = page_of(c_first);
  const int slots = kept_pages + page_of(kv_end - 1) - window_page + 1;
  int first_slot = 0;
  const bool whole_pages = page_shift >= 0 && SB % page_size == 0;
  const long page_values = (long)n_kv_head * page_size * D;
  auto bring = [&](int from) {
    first_slot = from;
    for (int i = tid; i < PF_PAGES && from + i < slots; i += THREADS) {
      const int slot = from + i;
      pages[i] = bt[slot < kept_pages ? slot : slot - kept_pages + window_page];
    }
  };
  // The slots of a stretch (the first and the last one that fetch reads; a last stretch may read its first query's position instead).
  auto low_slot = [&](int step) -> int {
    if (step < kept_steps) return page_of(step * SB);
    const int start = stretch_start(step), j = start + SB > kv_end && pos_lo < start ? pos_lo : start;
    return kept_pages + page_of(j) - window_page;
  };
  auto high_slot = [&](int step) -> int {
    if (step < kept_steps) return page_of(step * SB + SB - 1);
    const int end = stretch_start(step) + SB - 1;
    return kept_pages + page_of(end < kv_end ? end : kv_end - 1) - window_page;
  };
  // A stretch's rows go straight into LDS, 1 KB a load: the lane that fills chunk p of a row fetches the chunk that belongs there.
  // A key that the tile does not see is read from one that it does (its score is masked): behind the last query's from the first
  // query's position, before a window from the window's first; of a kept stretch from the sequence's first.
  auto fetch = [&](int step) {
    bf16_t* ks = pf_lds + step % BUFS * (2 * SB * D);
    const bool kept = step < kept_steps;
    const int start = stretch_start(step), base = (kept ? 0 : kept_pages - window_page) - first_slot;
    // Every key of the stretch is seen, and the stretch is whole pages: where a row lies within its page does not change from
    // stretch to stretch, and its page is as many behind the stretch's first (2 x 1,024 tokens x 8 heads 16.7 -> 15.5 us; with 128
    // registers it spills and costs 8 %).
    if (EARLY && whole_pages && !kept && start >= kv_begin && start + SB <= kv_end) {
      const int* own = pages + base + (start >> page_shift);
#pragma unroll
      for (int u = 0; u < LOADS; ++u) {
        const int piece = u * WAVES + wave, idx = piece * 64 + lane;
        const int row = idx / CH, c = pf_chunk<D>(row, idx - row * CH);
        const long at = (long)own[row >> page_shift] * page_values + (hk * page_size + (row & (page_size - 1))) * D + c * 8;
        __builtin_amdgcn_global_load_lds((global_ptr_t)(kpool + at), (lds_ptr_t)(ks + piece * 512), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((global_ptr_t)(vpool + at), (lds_ptr_t)(ks + SB * D + piece * 512), 16, 0, 0);
      }
      return;
    }
#pragma unroll
    for (int u = 0; u < LOADS; ++u) {
      const int piece = u * WAVES + wave, idx = piece * 64 + lane;
      const int row = idx / CH, c = pf_chunk<D>(row, idx - row * CH);
      int j = start + row;
      if (kept) j = j < keep_first ? j : start;
      else j = j >= kv_end ? pos_lo : (j < kv_begin && j >= keep_first ? kv_begin : j);
      const int pg = page_of(j);
      const long at = (long)((pages[base + pg] * n_kv_head + hk) * page_size + (j - pg * page_size)) * D + c * 8;
      __builtin_amdgcn_global_load_lds((global_ptr_t)(kpool + at), (lds_ptr_t)(ks + piece * 512), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((global_ptr_t)(vpool + at), (lds_ptr_t)(ks + SB * D + piece * 512), 16, 0, 0);
    }
  };
  bring(0);
  if (BIAS == 1) fill_bias(0);
  // the queries have arrived from here on: left to its first use, their wait would be one for all loads, in every step
#pragma unroll
  for (int kk = 0; kk < KK; ++kk) asm volatile("" : "+v"(qf[kk]));
  __syncthreads();
#pragma unroll
  for (int b = 0; b < AHEAD; ++b)
    if (b < n_steps) fetch(b);
  for (int b = 0; b < n_steps; ++b) {
    // this wave's loads of step b have arrived (those of AHEAD - 1 younger steps may be on their way), then everybody's; nobody
    // reads the buffer of step b - 1 any more, which is where step b + AHEAD goes
    if (b + AHEAD <= n_steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * 2 * LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const int c0 = stretch_start(b) + kg * PF_W;   // first key of this wave's part
    if (BIAS == 1 && b + 1 < n_steps) fill_bias(b + 1);
    // a part with no key that the wave's queries see (behind the last one's, or before a window) is left out
    const bool sees = c0 <= wave_hi && wave_lo <= pos_hi && (c0 + PF_W > wave_begin || c0 < keep_first);
    const bf16_t* ks = pf_lds + b % BUFS * (2 * SB * D) + kg * PF_W * D;
    const bf16_t* vs = ks + SB * D;
    auto key_part = [&](int kk) { return *reinterpret_cast<const bf16x8_t*>(ks + l31 * D + pf_chunk<D>(l31, kk * 2 + g) * 8); };
    bf16x8_t kf[KK];                                 // with registers to spare, on their way while the next loads are worked out
    if (EARLY && sees) {
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) kf[kk] = key_part(kk);
    }
    if (b + AHEAD < n_steps) {
      if (high_slot(b + AHEAD) >= first_slot + PF_PAGES) {   // the same for the whole workgroup; everybody has passed the barrier
        __syncthreads();
        bring(low_slot(b + AHEAD));
        __syncthreads();
      }
      fetch(b + AHEAD);
    }
    if (sees) {

      // scores: lane (query l31, half g) holds keys c0 + 8 (i / 4) + 4 g + i % 4
      f32x16_t s;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[i] = 0.f;
#pragma unroll
      for (int kk = 0; kk < KK; ++kk) s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(EARLY ? kf[kk] : key_part(kk), qf[kk], s, 0, 0, 0);
      // The value operands do not depend on the scores: asked for now, they arrive while the softmax keeps the wave busy.
      // k-slot (g, e) of operand t: key 16 t + 4 g + e for e < 4, key 16 t + 8 + 4 g + (e - 4) otherwise, which are the scores 8 t + e
      // of the lane.  Lanes 16 a .. 16 a + 15 of a half bring channels 16 a .. 16 a + 15 of four keys: lane j of them points at key
      // j / 4, channels 4 (j % 4) .., and gets channel j of the four.
      bf16x4_t vlo[2][CT], vhi[2][CT];
      typedef bf16x4_t __attribute__((address_space(3))) * lds_b64_t;
      const int vrow = 4 * g + ((lane & 15) >> 2), vch = ((lane >> 4) & 1) * 2 + ((lane & 3) >> 1);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const int lo = 16 * t + vrow, hi = lo + 8;
          vlo[t][ct] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_b64_t)(vs + lo * D + pf_chunk<D>(lo, ct * 4 + vch) * 8 + (lane & 1) * 4));
          vhi[t][ct] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_b64_t)(vs + hi * D + pf_chunk<D>(hi, ct * 4 + vch) * 8 + (lane & 1) * 4));
        }
      __builtin_amdgcn_sched_barrier(0);   // or the compiler moves each read down to its use

      if (BIAS == 1) {
        const float* mine = bias_tab + (b & 1) * NB + kg * PF_W + (QT - 1 - (qw * 32 + l31)) + g * 4;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = __builtin_fmaf(s[i], raw2, mine[8 * (i >> 2) + (i & 3)]);
      }
      if (BIAS == 2) {
        // scaled and capped scores in units of log2 e, then minus slope * distance (the lane's first key's, and
        // the keys' places behind it as constants)
        float first = slope2 * (float)(c0 + g * 4 - my_pos);
        const float in = scale * __builtin_amdgcn_rcpf(softcap), cap2 = softcap * 1.4426950408889634f;
        auto off = [&](int i) { return __builtin_fmaf(slope2, (float)(8 * (i >> 2) + (i & 3)), first); };
        if (Q == 1 || D == 32) {
          // one branch: one an element spills 70 scalar registers here (33 tokens behind 700 x 9 heads of 64 17.1 us, so 13.8; 3 x 130
          // tokens x 25 heads 10.2, 8.8); in the other forms this one spills up to 9 vector registers
          if (softcap > 0.f) {
            asm volatile("" : "+v"(first));   // or the branches share 16 offsets, made and kept in front of them
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = __builtin_fmaf(cap2, tanh_fast(s[i] * in), off(i));
          } else {
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = __builtin_fmaf(s[i], raw2, off(i));
          }
        } else {
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[i] = softcap > 0.f ? __builtin_fmaf(cap2, tanh_fast(s[i] * in), off(i)) : __builtin_fmaf(s[i], raw2, off(i));
        }
      } else if (softcap > 0.f) {
        // capped scores: cap * tanh(s * scale / cap), kept in the raw scores' units (times cap / scale)
        const float in = scale * __builtin_amdgcn_rcpf(softcap), back = softcap * __builtin_amdgcn_rcpf(scale);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = back * tanh_fast(s[i] * in);
      }
      // keys that every query of this wave sees (the common case away from the diagonal) need no mask
      if (!(c0 + PF_W - 1 <= wave_lo && wave_lo + 31 < ctx + q_len && c0 >= wave_begin_hi)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = c0 + 8 * (i >> 2) + 4 * g + (i & 3);
          const bool see = q_ok && key <= my_pos && (key >= my_begin || key < keep_first);
          s[i] = see ? s[i] : -INFINITY;
        }
      }
      if (!weigh) {
        float mx = s[0];
#pragma unroll
        for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
        mx = pf_max_of_pair(mx) * sc2;   // -inf stays -inf
        if (__any(mx > m)) {                       // else nothing is scaled
          const float m_new = fmaxf(m, mx);
          const float alpha = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);   // nothing to scale before the first keys
          l *= alpha;
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[ct][i] *= alpha;
          m = m_new;
        }
      }
      const float m_sub = m == -INFINITY ? 0.f : m;   // exp2(-inf - 0) = 0 for masked scores
      float rs[2] = {0.f, 0.f};
      bf16x8_t pf[2];
      // (a masked score is -inf: exp2(-inf) = 0, and 1 / (1 + exp2(inf)) = 0)
      if (weigh) {
#pragma unroll
        for (int i = 0; i < 16; ++i)
          s[i] = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(__builtin_fmaf(s[i], sc2, bias2))));
      } else {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i], sc2, -m_sub));
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int i = 0; i < 8; ++i) rs[t] += s[8 * t + i];
        const u32x4_t packed = {pack_bf16x2(s[8 * t], s[8 * t + 1]), pack_bf16x2(s[8 * t + 2], s[8 * t + 3]),
                                pack_bf16x2(s[8 * t + 4], s[8 * t + 5]), pack_bf16x2(s[8 * t + 6], s[8 * t + 7])};
        pf[t] = __builtin_bit_cast(bf16x8_t, packed);
      }
      l += rs[0] + rs[1];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const bf16x8_t vf = {vlo[t][ct][0], vlo[t][ct][1], vlo[t][ct][2], vlo[t][ct][3],
                               vhi[t][ct][0], vhi[t][ct][1], vhi[t][ct][2], vhi[t][ct][3]};
          o[ct] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf, pf[t], o[ct], 0, 0, 0);
        }
    }
  }

  // Every wave puts its max, sum and output into LDS (the staged keys are done with); then the K waves of the same queries
  // put a K-th of the channels together each.
  __syncthreads();
  constexpr int EACH = 64 * (2 + CT * 16), RUNS = CT * 4, MINE = (RUNS + K - 1) / K;   // runs of four channels
  float* const xch = reinterpret_cast<float*>(pf_lds) + qw * EACH + lane;
  {
    float* mine = xch + kg * Q * EACH;
    mine[0] = m;
    mine[64] = l;
#pragma unroll
    for (int ct = 0; ct < CT; ++ct)
#pragma unroll
      for (int i = 0; i < 16; ++i) mine[(2 + ct * 16 + i) * 64] = o[ct][i];
  }
  __syncthreads();
  if (!q_ok || kg * MINE >= RUNS) return;
  float part[K];                     // a group that saw no key has max -inf and nothing to add
  float m_all = xch[0];
#pragma unroll
  for (int k = 1; k < K; ++k) m_all = fmaxf(m_all, xch[k * Q * EACH]);
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const float mk = xch[k * Q * EACH];
    part[k] = mk == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mk - m_all);
    sum += (xch[k * Q * EACH + 64] + xch[k * Q * EACH + 64 + (lane < 32 ? 32 : -32)]) * part[k];
  }
  if (sinks) {
    // one more term of the denominator, exp(sink), with no value (m is in units of log2 e)
    const float sink = sinks[h] * 1.4426950408889634f;
    const float m_sink = fmaxf(m_all, sink);
    const float a = m_all == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_all - m_sink);
    sum = sum * a + __builtin_amdgcn_exp2f(sink - m_sink);
#pragma unroll
    for (int k = 0; k < K; ++k) part[k] *= a;
  }
  float inv = weigh ? 1.0f : 1.0f / sum;
  if (gate)   // the head's output times sigmoid(gate[token][head])
    inv *= __builtin_amdgcn_rcpf(1.0f + __expf(-bf16_to_float(gate[(long)(q_start + my_q) * ldg + h])));
  bf16_t* orow = out + (long)(q_start + my_q) * ldo + (long)h * D;
  // a lane's four neighbouring channels are one 8-byte store (the launcher has checked
  // that rows start 8 bytes aligned)
#pragma unroll
  for (int n = 0; n < MINE; ++n) {
    const int run = kg * MINE + n;
    if (RUNS % K != 0 && run >= RUNS) break;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = __builtin_fmaf(xch[k * Q * EACH + (2 + run * 4 + i) * 64], part[k], v[i]);
    uint2 pk;
    pk.x = pack_bf16x2(v[0] * inv, v[1] * inv);
    pk.y = pack_bf16x2(v[2] * inv, v[3] * inv);
    *reinterpret_cast<uint2*>(orow + run * 8 + g * 4) = pk;   // run 4 ct + i / 4: channels 32 ct + 8 (i / 4) + 4 g ..
  }
}
