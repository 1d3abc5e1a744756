// Attention of the 32-bit path on the float32 matrix cores (v_mfma_f32_16x16x4_f32), paged, causal, softmax in float32:
// what the general kernel (attention_generic.hip, which says what the arguments mean) computes, for head sizes 16, 32,
// 64 and 128 and softmax weights (reference: src/minigpt_infer/model.py:61-87).
//
// A workgroup has 16 queries of one request, a head and eight waves.  Keys are taken in chunks of 64 that start at
// multiples of 64; chunk c belongs to wave c % 8, which walks its chunks with a running maximum and sum; the waves'
// results are put together in the order of the waves.  All of that depends on a key's position only, and what a query
// does not see adds zeros, so a query's output is the same bits in a prompt, in a portion of one and in a decode step.
// Keys that no query of the tile sees are never loaded.  A value that is infinite or NaN shows in the wave's sums, where a
// weight of zero has made NaN of it for queries that do not see its key: the wave then walks its chunks again and takes such
// values out of the products of chunks that not all queries see whole, adding them to the queries that see them.  The walk
// is there twice for that: with the look at the values in the one loop, prompts of 15 requests x 12 heads of 64 took 48.2 us
// for 44.6, now 45; so they did with more than 96 registers, which the launch bounds of that head size keep to.
//
// The scores of a chunk are made transposed, S^T = K Q^T: a lane then has, of query lane % 16, the keys
// 16 t + 4 (lane / 16) + i, which is just how O^T = V^T P^T takes them as its second operand.  Weights, maxima and sums
// stay in the lanes; nothing goes through LDS before the end.  Keys and values come straight from the pages, 16 bytes a
// lane; of the values a lane takes the head size / 16 consecutive channels that are its row in as many tiles of O^T.
//
// Tiles whose last query is among the first 16 have a walk of their own with the one group of 16 keys that there is: 8 heads
// of 64 behind one key 5.5 us (with the chunk's other groups, all zeros, 8.7), behind 16 5.8 (8.9); of 128 6.3 (11.4).  The
// same in chunks of any number of groups, a test for each, kept the loads of one group behind the products of the one
// before: 16 requests x 8 heads of 64 behind 700 keys 23.6 -> 35.0 us.
//
// The general kernel walks a query's keys with one wave and 4-byte loads: prompts of 640, 295, 265 and 1 tokens x 8 heads of
// 64 326 us, here 38; decode steps of 16 requests x 12 heads behind 16 to 280 keys 68 us, here 12.4 (7.9 with the kernel for
// steps of single tokens, further down).
#include "attention_exact.h"
#include "attention_mask.h"
#include "common.h"
#include <type_traits>

#define AX_WAVES 8
#define AX_QUERIES 16
#define AX_CHUNK 64
#define AX_NONE 0xffffffffu     // not a row of the pool

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float ax_f4;

// over the four lanes that share a query
__device__ __forceinline__ float ax_max4(float v) {
  v = fmaxf(v, __shfl_xor(v, 16, MGPT_WAVE));
  return fmaxf(v, __shfl_xor(v, 32, MGPT_WAVE));
}
__device__ __forceinline__ float ax_sum4(float v) {
  v += __shfl_xor(v, 16, MGPT_WAVE);
  return v + __shfl_xor(v, 32, MGPT_WAVE);
}

__device__ __forceinline__ bool ax_unusual(float v) { return !(fabsf(v) <= 3.402823466e38f); }   // infinite or NaN

// Takes the infinite and NaN values out of vf (values of keys j0 .. j0 + 15, whose rows of the pool the lanes' `row` says,
// as the kernel holds them) and adds each, times its weight, to the outputs of the queries that see its key.
template <int G>
__device__ __forceinline__ void ax_take_unusual(float (&vf)[4][G], const ax_f4& p, ax_f4 (&acc)[G],
                                                const float* __restrict__ vpool, unsigned int row, int j0, int my_pos,
                                                int my_begin, int keep_first) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, lk = lane >> 4;
  float zero = 0.f;                                                     // NaN if one of them is unusual
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int g = 0; g < G; ++g) zero = fmaf(vf[i][g], 0.f, zero);
  const uint64_t all = __ballot(zero != zero);
  if (!all) return;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int g = 0; g < G; ++g) vf[i][g] = ax_unusual(vf[i][g]) ? 0.f : vf[i][g];
  for (uint64_t lanes = all; lanes; lanes &= lanes - 1) {               // lanes that have one, in order
    const int from = __builtin_amdgcn_readfirstlane(__ffsll((unsigned long long)lanes) - 1);
    const int from_k = from >> 4, from_c = from & 15;
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
      const int j = j0 + 4 * from_k + i;
      const unsigned int vr = __builtin_amdgcn_readlane(row, 4 * from_k + i);
      const float w = __shfl(i == 0 ? p[0] : (i == 1 ? p[1] : (i == 2 ? p[2] : p[3])), 16 * from_k + l16, MGPT_WAVE);
      const bool mine = vr != AX_NONE && j <= my_pos && (j >= my_begin || j < keep_first) && lk == from_c >> 2;
      if (!mine) continue;
      const float* src = vpool + (long)vr * (16 * G) + G * from_c;     // channel G from_c + g: element from_c % 4 of acc[g]
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float v = src[g];
        if (!ax_unusual(v)) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[g][e] = e == (from_c & 3) ? fmaf(w, v, acc[g][e]) : acc[g][e];
      }
    }
  }
}

template <int D>
__global__ __launch_bounds__(64 * AX_WAVES, D == 64 ? 5 : 1) void attention_exact_kernel(AttentionExactArgs a) {
  constexpr int G = D / 16;            // groups of 16 channels; also the channels of a lane's row of V^T
  constexpr int LD = D + 4;
  extern __shared__ __align__(16) float ax_lds[];      // [waves][queries][LD]
  __shared__ float m_s[AX_WAVES][AX_QUERIES], l_s[AX_WAVES][AX_QUERIES];
  __shared__ int req_s[AX_QUERIES];                    // negative: a token of the padding, left alone

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int h = blockIdx.y, hk = h / (a.n_head / a.n_kv_head);

  // the request and the tile of it that this workgroup has: requests' tiles are numbered one behind the other
  int tile = blockIdx.x;
  int r = piece_owner(a.n_req, tile, [&](int i) { return (a.cu_q[i + 1] - a.cu_q[i] + AX_QUERIES - 1) / AX_QUERIES; });
  if (r < 0) return;                                    // beyond the step's tiles: the whole workgroup
  r = __builtin_amdgcn_readfirstlane(r);
  const int q_start = a.cu_q[r], q_len = a.cu_q[r + 1] - q_start;
  const int q0 = __builtin_amdgcn_readfirstlane(tile) * AX_QUERIES;
  const int ctx = a.seq_lens[r] - q_len;
  int n_here = q_len - q0 < AX_QUERIES ? q_len - q0 : AX_QUERIES;
  if (a.n_tokens - q_start - q0 < n_here) n_here = a.n_tokens - q_start - q0;   // rows that the caller does not have
  if (n_here <= 0) return;
  const int token_req = a.q_req[q_start + q0 + (l16 < n_here ? l16 : 0)];       // for the end
  const int pos_lo = ctx + q0, pos_hi = pos_lo + n_here - 1;
  const int tile_begin = first_seen(pos_lo, a.window, a.chunked), last_begin = first_seen(pos_hi, a.window, a.chunked);
  const bool q_ok = l16 < n_here;
  const int my_pos = pos_lo + l16, my_begin = first_seen(my_pos, a.window, a.chunked);
  const int* bt = a.block_tables + (long)r * a.max_blocks;

  ax_f4 qf[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    qf[g] = (ax_f4){0.f, 0.f, 0.f, 0.f};
    if (q_ok) qf[g] = *reinterpret_cast<const ax_f4*>(a.q + (long)(q_start + q0 + l16) * a.ldq + (long)h * D + 16 * g + 4 * lk);
  }
  const float slope = a.slopes ? a.slopes[h] : 0.f;
  const float* dist = a.dist_bias ? a.dist_bias + (long)h * a.bias_len : nullptr;

  float m, l;
  ax_f4 acc[G];                                         // O^T tile dt, rows 4 lk + i: channel G (4 lk + i) + dt
  // the wave's walk over its chunks; CAREFUL: for values that are infinite or NaN; GROUPS: of 16 keys that a chunk can have
  auto walk = [&](auto careful, auto groups) __attribute__((always_inline)) {
    constexpr bool CAREFUL = decltype(careful)::value;
    constexpr int GROUPS = decltype(groups)::value;
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int g = 0; g < G; ++g) acc[g] = (ax_f4){0.f, 0.f, 0.f, 0.f};
    for (int c = wave; c * AX_CHUNK <= pos_hi; c += AX_WAVES) {
      const int c0 = c * AX_CHUNK;
      if (c0 + AX_CHUNK <= tile_begin && c0 >= a.keep_first) continue;
      // whether every query of the tile sees every key that is loaded (always so for a single query)
      const bool whole = (c0 + AX_CHUNK - 1 < pos_hi ? c0 + AX_CHUNK - 1 : pos_hi) <= pos_lo &&
                         ((c0 > tile_begin ? c0 : tile_begin) >= last_begin || c0 + AX_CHUNK <= a.keep_first);
      // the pool rows of this lane's four keys, c0 + 16 t + l16
      unsigned int row[GROUPS];                                // 2^32 rows of 16 channels are 275 GB
#pragma unroll
      for (int t = 0; t < GROUPS; ++t) {
        const int j = c0 + 16 * t + l16;
        row[t] = AX_NONE;
        if (j <= pos_hi && (j >= tile_begin || j < a.keep_first)) {
          const int idx = j / a.page_size;
          row[t] = ((unsigned int)bt[idx] * a.n_kv_head + hk) * a.page_size + (j - idx * a.page_size);
        }
      }
      ax_f4 s[GROUPS];
#pragma unroll
      for (int t = 0; t < GROUPS; ++t) {
        s[t] = (ax_f4){0.f, 0.f, 0.f, 0.f};
        ax_f4 kf[G];
#pragma unroll
        for (int g = 0; g < G; ++g) {
          kf[g] = (ax_f4){0.f, 0.f, 0.f, 0.f};
          if (row[t] != AX_NONE) kf[g] = *reinterpret_cast<const ax_f4*>(a.kpool + (long)row[t] * D + 16 * g + 4 * lk);
        }
#pragma unroll
        for (int g = 0; g < G; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[g][e], qf[g][e], s[t], 0, 0, 0);
      }
      float top = -INFINITY;
#pragma unroll
      for (int t = 0; t < GROUPS; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = c0 + 16 * t + 4 * lk + i;
          float v = s[t][i] * a.scale;
          if (dist) v += dist[distance_entry(my_pos - j, a.bias_len)];
          if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
          if (a.slopes) v -= slope * (float)(my_pos - j);
          if (!(q_ok && j <= my_pos && (j >= my_begin || j < a.keep_first))) v = -INFINITY;
          s[t][i] = v;
          top = fmaxf(top, v);
        }
      const float m_new = fmaxf(m, ax_max4(top));
      const float m_sub = m_new == -INFINITY ? 0.f : m_new;   // nothing seen so far: every weight is exp(-inf)
      const float alpha = expf(m - m_sub);
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < GROUPS; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[t][i] = expf(s[t][i] - m_sub);
          sum += s[t][i];
        }
      l = l * alpha + ax_sum4(sum);
      m = m_new;
#pragma unroll
      for (int g = 0; g < G; ++g) acc[g] *= alpha;
#pragma unroll
      for (int t = 0; t < GROUPS; ++t) {
        float vf[4][G];                                   // of key 16 t + 4 lk + i the channels G l16 .. G l16 + G - 1
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned int vr = __shfl(row[t], 4 * lk + i, MGPT_WAVE);
          const float* src = a.vpool + (long)vr * D + G * l16;
          if constexpr (G >= 4) {
#pragma unroll
            for (int g = 0; g < G; g += 4) {
              ax_f4 v = {0.f, 0.f, 0.f, 0.f};
              if (vr != AX_NONE) v = *reinterpret_cast<const ax_f4*>(src + g);
#pragma unroll
              for (int e = 0; e < 4; ++e) vf[i][g + e] = v[e];
            }
          } else {
#pragma unroll
            for (int g = 0; g < G; ++g) vf[i][g] = vr != AX_NONE ? src[g] : 0.f;
          }
        }
        if (CAREFUL && !whole) ax_take_unusual<G>(vf, s[t], acc, a.vpool, row[t], c0 + 16 * t, my_pos, my_begin, a.keep_first);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int g = 0; g < G; ++g) acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][g], s[t][i], acc[g], 0, 0, 0);
      }
    }
  };
  if (pos_hi < 16) walk(std::false_type{}, std::integral_constant<int, 1>{});
  else walk(std::false_type{}, std::integral_constant<int, 4>{});
  float zero = 0.f;                                     // an infinity or NaN among the sums stays one to the end
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < 4; ++i) zero = fmaf(acc[g][i], 0.f, zero);
  if (__ballot(zero != zero)) walk(std::true_type{}, std::integral_constant<int, 4>{});
  if (lk == 0) {
    m_s[wave][l16] = m;
    l_s[wave][l16] = l;
    if (wave == 0) req_s[l16] = token_req;
  }
  float* mine = ax_lds + (wave * AX_QUERIES + l16) * LD + 4 * G * lk;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int g = 0; g < G; ++g) mine[i * G + g] = acc[g][i];
  __syncthreads();

  for (int e = tid; e < n_here * D; e += 64 * AX_WAVES) {
    const int qi = e / D, d = e % D;
    if (req_s[qi] < 0) continue;
    float top = a.sinks ? a.sinks[h] : -INFINITY;       // one more term of the denominator, with no value
#pragma unroll
    for (int w = 0; w < AX_WAVES; ++w) top = fmaxf(top, m_s[w][qi]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < AX_WAVES; ++w) {
      const float f = expf(m_s[w][qi] - top);
      den += l_s[w][qi] * f;
      num += ax_lds[(w * AX_QUERIES + qi) * LD + d] * f;
    }
    if (a.sinks) den += expf(a.sinks[h] - top);
    const long n = q_start + q0 + qi;
    float inv = 1.0f / den;
    if (a.gate) inv *= 1.0f / (1.0f + expf(-a.gate[n * a.ldg + h]));
    a.out[n * a.ldo + (long)h * D + d] = num * inv;
  }
}

// A step of single tokens (token n is request n's only one): a workgroup per (token, head) with the same eight waves, chunks
// and sums, so the same bits, without what the general walk spends on finding its work, on waiting and on the 15 queries
// that are not there.
//  * The request is the block's number; position, query, padding mark and the first chunk's block table entries are asked
//    for together, and all of a chunk's keys at once, its values behind them as the keys' registers come free: two trips to
//    memory, the general walk has six.  Keys that are not seen are read from the pool's first rows and dropped, which keeps
//    the loads free of branches.
//  * The scores come from the same matrix products, with the query in all 16 columns; of the 16 copies of its 16 scores
//    that a row of lanes then holds each lane takes one, so that mask and exponential are done once a key.
//  * v_mfma_f32_16x16x4_f32 is the chain of four fused multiply-adds over its k in order (compared bit for bit over 40
//    million sums: ordinary, denormal and overflowing ones), so the values are weighted on the vector unit in the order of
//    the general walk's products, a lane a channel: 64 instructions of 4 cycles for 64 of 32.
// A query sees every key that it weighs, so infinite and NaN values need no second walk.
// us in a graph of such calls, general walk / here: 1 request x 12 heads of 64 behind 100 keys 9.9 / 5.5; 16 x 12 behind 16 to
// 280 12.0 / 7.9, 64 x 12 30 / 19; 8 x 8 behind 700 20 / 12; 64 x 8 behind 900 to 1,000 (bound by the 250 MB) 42.8 / 39.5;
// 16 x 8 heads of 128 behind 200 to 300 19.5 / 12.5; 3 x 4 heads of 16 behind 5 to 42 7.0 / 4.6.  Heads of 64 need the 128
// registers that let a compute unit have two workgroups: with scores kept for all 64 keys and ten registers spilled 64 x 8
// took 44.5.  A chunk of which at most one group of 16 keys is there (a short request's only one, every fourth one's last) is walked
// without the other three: behind 1 to 5 keys 64 x 25 heads of 64 take 11 us, of 128 24, with the keys that are not there 18 and
// 40, the general walk, which leaves them out too, 16 and 31.  What is left at 16 x 12: the launch (1.6), two trips to memory, 64
// matrix products (0.9) and the merge.
//
// PAGE16: pages are multiples of 16 positions, so 16 keys lie one behind the other.
template <int D, bool PAGE16>
__global__ __launch_bounds__(64 * AX_WAVES, D == 128 ? 2 : 4) void attention_exact_single_kernel(AttentionExactArgs a, int page_shift) {
  constexpr int G = D / 16;
  constexpr int C = D > 64 ? D / 64 : 1;                // channels of a lane
  constexpr int AHEAD = G <= 4 ? 4 : 2;                 // groups of 16 keys on their way
  typedef __attribute__((__vector_size__(C * sizeof(float)))) float ax_fc;
  __shared__ __align__(16) float p_s[AX_WAVES][AX_CHUNK];
  __shared__ float o_s[AX_WAVES][D];
  __shared__ float m_s[AX_WAVES], l_s[AX_WAVES];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, lk = lane >> 4;
  const int n = blockIdx.x, h = blockIdx.y, hk = h / (a.n_head / a.n_kv_head);
  const int* bt = a.block_tables + (long)n * a.max_blocks;
  auto page_of = [&](int j) { return page_shift >= 0 ? j >> page_shift : j / a.page_size; };
  int entry[4];                                         // block table entries of the keys c0 + 16 t + l16
  auto look_up = [&](int c) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int idx = page_of(c * AX_CHUNK + 16 * t + l16);
      entry[t] = bt[idx < a.max_blocks ? idx : a.max_blocks - 1];
    }
  };
  look_up(wave);
  ax_f4 qf[G];
#pragma unroll
  for (int g = 0; g < G; ++g) qf[g] = *reinterpret_cast<const ax_f4*>(a.q + (long)n * a.ldq + (long)h * D + 16 * g + 4 * lk);
  const int pos = a.seq_lens[n] - 1;
  if (a.q_req[n] < 0) return;                           // a token of the padding: the whole workgroup
  const int begin = first_seen(pos, a.window, a.chunked);
  const float slope = a.slopes ? a.slopes[h] : 0.f;
  const float* dist = a.dist_bias ? a.dist_bias + (long)h * a.bias_len : nullptr;
  const float* vlane = a.vpool + C * (D >= 64 ? lane : lane % D);
  auto sees = [&](int j) { return j <= pos && (j >= begin || j < a.keep_first); };

  float m = -INFINITY, l = 0.f;
  ax_fc acc;                                            // channels C lane ..
#pragma unroll
  for (int x = 0; x < C; ++x) acc[x] = 0.f;
  // chunk c, of which the first GROUPS groups of 16 keys are there
  auto walk = [&](int c, auto groups) {
    constexpr int GROUPS = decltype(groups)::value;
    const int c0 = c * AX_CHUNK;
    unsigned int row[4];                                // of the keys c0 + 16 t + l16
    uint64_t seen[4];                                   // the 16 keys' bits, four times over
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int j = c0 + 16 * t + l16, idx = page_of(j);
      const bool ok = sees(j);
      seen[t] = __ballot(ok);
      row[t] = (PAGE16 ? seen[t] != 0 : ok) ? ((unsigned int)entry[t] * a.n_kv_head + hk) * a.page_size + (j - idx * a.page_size)
                                            : (PAGE16 ? l16 : 0);
    }
    if ((c + AX_WAVES) * AX_CHUNK <= pos) look_up(c + AX_WAVES);
    if (c0 + AX_CHUNK <= begin && c0 >= a.keep_first) return;
    ax_f4 kf[AHEAD][G];
    auto load_keys = [&](int t) {
      const float* src = a.kpool + (long)row[t] * D + 4 * lk;
#pragma unroll
      for (int g = 0; g < G; ++g) kf[t % AHEAD][g] = *reinterpret_cast<const ax_f4*>(src + 16 * g);
    };
    ax_fc vf[4][16];
    auto load_values = [&](int t) {
      if constexpr (PAGE16) {
        const float* src = vlane + (long)(unsigned int)__builtin_amdgcn_readfirstlane((int)row[t]) * D;
#pragma unroll
        for (int x = 0; x < 16; ++x) vf[t][x] = *reinterpret_cast<const ax_fc*>(src + x * D);
      } else {
#pragma unroll
        for (int x = 0; x < 16; ++x)
          vf[t][x] = *reinterpret_cast<const ax_fc*>(vlane + (long)(unsigned int)__builtin_amdgcn_readlane((int)row[t], x) * D);
      }
    };
#pragma unroll
    for (int t = 0; t < AHEAD && t < GROUPS; ++t) load_keys(t);
    float v = 0.f;                                      // this lane's key: 16 (l16 / 4) + 4 lk + l16 % 4
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
      ax_f4 s = {0.f, 0.f, 0.f, 0.f};                   // keys 16 t + 4 lk + i, the same in all 16 lanes
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t % AHEAD][g][e], qf[g][e], s, 0, 0, 0);
#pragma unroll
      for (int i = 0; i < 4; ++i) v = l16 == 4 * t + i ? s[i] : v;
      if (t + AHEAD < GROUPS) load_keys(t + AHEAD);
      load_values(t);                                   // into the registers of keys that are done with
      __builtin_amdgcn_sched_barrier(0);
    }
    const int key = 16 * (l16 >> 2) + 4 * lk + (l16 & 3), j = c0 + key;
    v *= a.scale;
    if (dist) v += dist[distance_entry(pos - j, a.bias_len)];
    if (a.softcap > 0.f) v = a.softcap * tanhf(v / a.softcap);
    if (a.slopes) v -= slope * (float)(pos - j);
    if (!sees(j)) v = -INFINITY;
    const float m_new = fmaxf(m, wave_max(v));
    const float m_sub = m_new == -INFINITY ? 0.f : m_new;   // nothing seen so far: every weight is exp(-inf)
    const float alpha = expf(m - m_sub);
    p_s[wave][key] = expf(v - m_sub);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    float sum = 0.f;
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) {
      const ax_f4 p = *reinterpret_cast<const ax_f4*>(&p_s[wave][16 * t + 4 * lk]);
#pragma unroll
      for (int i = 0; i < 4; ++i) sum += p[i];
    }
    l = l * alpha + ax_sum4(sum);
    m = m_new;
    acc *= alpha;
    uint64_t both = ~0ull;
#pragma unroll
    for (int t = 0; t < GROUPS; ++t) both &= seen[t];
    const bool whole = both == ~0ull;
    auto weigh = [&](auto all) {
#pragma unroll
      for (int t = 0; t < GROUPS; ++t) {
        __builtin_amdgcn_sched_barrier(0);              // (or all weights are read at once, into registers that are not there)
        ax_f4 p[4];                                     // the keys 16 t + 4 k + i, for everybody
#pragma unroll
        for (int k = 0; k < 4; ++k) p[k] = *reinterpret_cast<const ax_f4*>(&p_s[wave][16 * t + 4 * k]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int x = 0; x < C; ++x) {
              const float val = decltype(all)::value || (seen[t] >> (4 * k + i) & 1) ? vf[t][4 * k + i][x] : 0.f;
              acc[x] = fmaf(val, p[k][i], acc[x]);
            }
      }
    };
    if (whole) weigh(std::true_type{});
    else weigh(std::false_type{});
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  };
  for (int c = wave; c * AX_CHUNK <= pos; c += AX_WAVES) {
    if (c * AX_CHUNK + 16 > pos) walk(c, std::integral_constant<int, 1>{});
    else walk(c, std::integral_constant<int, 4>{});
  }
  if (lane == 0) {
    m_s[wave] = m;
    l_s[wave] = l;
  }
  if (D >= 64 || lane < D) *reinterpret_cast<ax_fc*>(&o_s[wave][C * lane]) = acc;
  __syncthreads();
  if (tid >= D) return;
  float top = a.sinks ? a.sinks[h] : -INFINITY;
#pragma unroll
  for (int w = 0; w < AX_WAVES; ++w) top = fmaxf(top, m_s[w]);
  float num = 0.f, den = 0.f;
#pragma unroll
  for (int w = 0; w < AX_WAVES; ++w) {
    const float f = expf(m_s[w] - top);
    den += l_s[w] * f;
    num += o_s[w][tid] * f;
  }
  if (a.sinks) den += expf(a.sinks[h] - top);
  float inv = 1.0f / den;
  if (a.gate) inv *= 1.0f / (1.0f + expf(-a.gate[(long)n * a.ldg + h]));
  a.out[(long)n * a.ldo + (long)h * D + tid] = num * inv;
}

template <int D>
static int launch_single(const AttentionExactArgs& a, hipStream_t stream) {
  const int shift = (a.page_size & (a.page_size - 1)) == 0 ? __builtin_ctz(a.page_size) : -1;
  const dim3 grid(a.n_tokens, a.n_head), block(64 * AX_WAVES);
  if (a.page_size % 16 == 0) hipLaunchKernelGGL((attention_exact_single_kernel<D, true>), grid, block, 0, stream, a, shift);
  else hipLaunchKernelGGL((attention_exact_single_kernel<D, false>), grid, block, 0, stream, a, shift);
  return mgpt_last_error();
}

template <int D>
static int launch(const AttentionExactArgs& a, hipStream_t stream) {
  constexpr int bytes = AX_WAVES * AX_QUERIES * (D + 4) * (int)sizeof(float);
  static bool allowed = bytes <= 48 * 1024;            // more LDS than a kernel gets without asking
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_exact_kernel<D>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  // at most so many tiles: a request's last one may be short
  const long tiles = ((long)a.n_tokens + (long)(AX_QUERIES - 1) * (a.n_req < a.n_tokens ? a.n_req : a.n_tokens)) / AX_QUERIES;
  if (tiles > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;
  hipLaunchKernelGGL(attention_exact_kernel<D>, dim3((unsigned int)tiles, a.n_head), dim3(64 * AX_WAVES), bytes, stream, a);
  return mgpt_last_error();
}

bool mgpt_attention_exact_takes(const AttentionExactArgs& a, int head_dim) {
  const uintptr_t together = reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.kpool) |
                             reinterpret_cast<uintptr_t>(a.vpool);
  return (head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128) && (together & 15) == 0 && a.ldq % 4 == 0 &&
         a.n_req > 0;   // (without requests all tokens are padding: the general kernel leaves them alone)
}

int mgpt_attention_exact_launch(const AttentionExactArgs& a, int head_dim, int single, hipStream_t stream) {
  if (single && a.n_tokens <= a.n_req) {
    if (head_dim == 16) return launch_single<16>(a, stream);
    if (head_dim == 32) return launch_single<32>(a, stream);
    if (head_dim == 64) return launch_single<64>(a, stream);
    return launch_single<128>(a, stream);
  }
  if (head_dim == 16) return launch<16>(a, stream);
  if (head_dim == 32) return launch<32>(a, stream);
  if (head_dim == 64) return launch<64>(a, stream);
  return launch<128>(a, stream);
}
