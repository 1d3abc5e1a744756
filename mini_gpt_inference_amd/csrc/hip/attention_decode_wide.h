// The body of the attention kernel for single tokens (attention_decode_wide.hip says what it does and why), for that kernel
// and for the one that also has a step's prompt portions (attention_mixed.hip).
#pragma once
#include "attention_mask.h"
#include "common.h"

typedef __attribute__((ext_vector_type(2))) __bf16 aw_bf16x2_t;

template <int CTRL>
__device__ __forceinline__ float aw_dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

// sum over the LPK neighbouring lanes of an aligned group; every lane of the group gets it
template <int LPK>
__device__ __forceinline__ float aw_group_sum(float v) {
  v += aw_dpp<0xB1>(v);                 // quad_perm [1,0,3,2]
  if (LPK >= 4) v += aw_dpp<0x4E>(v);   // quad_perm [2,3,0,1]
  if (LPK >= 8) v += aw_dpp<0x141>(v);  // row_half_mirror: lane i of each 8 reads lane 7 - i
  if (LPK >= 16) v += aw_dpp<0x140>(v); // row_mirror: lane i of each 16 reads lane 15 - i
  return v;
}

// maximum over the 64 lanes, as a value that is the same in all of them
__device__ __forceinline__ float aw_wave_max(float v) {
  v = fmaxf(v, aw_dpp<0xB1>(v));
  v = fmaxf(v, aw_dpp<0x4E>(v));
  v = fmaxf(v, aw_dpp<0x141>(v));
  v = fmaxf(v, aw_dpp<0x140>(v));
  const int b = __float_as_int(v);
  const float r0 = __int_as_float(__builtin_amdgcn_readlane(b, 0));
  const float r1 = __int_as_float(__builtin_amdgcn_readlane(b, 16));
  const float r2 = __int_as_float(__builtin_amdgcn_readlane(b, 32));
  const float r3 = __int_as_float(__builtin_amdgcn_readlane(b, 48));
  return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

__device__ __forceinline__ float aw_dot2(unsigned int a, unsigned int b, float c) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(aw_bf16x2_t, a), __builtin_bit_cast(aw_bf16x2_t, b),
                                         c, false);
}

// Floats of LDS that it takes.
template <int D, int W>
constexpr int aw_lds_floats() {
  return (W * (64 / (D / 8)) + W * 64 / D) * (D + 1) + W;
}

// Token n, head h, by W waves: a workgroup, or each half of one with its own LDS, both for the same token.  IDENT: token n is request n (or padded), so its block table row is known before
// anything is loaded.  SIDE: 0: any token; otherwise tokens that see up to (1) or more than (-1)
// `keys` keys; others are left alone.
template <int D, bool IDENT, int BIAS, int W, int SIDE = 0>
__device__ __forceinline__ void aw_decode(
    const bf16_t* __restrict__ q, long ldq, bf16_t* __restrict__ out, long ldo,
    const bf16_t* __restrict__ kpool, const bf16_t* __restrict__ vpool,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ positions,
    const int* __restrict__ q_req, const int* __restrict__ cu_q, int n_head, int n_kv_head, int page_shift,
    int num_pages, unsigned int page_bytes, float scale_log2e, int window, const float* __restrict__ sinks,
    float cap_log2e, const bf16_t* __restrict__ gate, long ldg, int keep_first, const float* __restrict__ score_bias,
    int chunked, const float* __restrict__ dist_bias, int bias_len, const float* __restrict__ slopes, int n,
    int h, float* __restrict__ lds, int keys = 0) {
  constexpr int LPK = D / 8;     // lanes per key
  constexpr int KPI = 64 / LPK;  // keys per load instruction
  constexpr int ROWS = W * KPI;      // partial results: one per (key subgroup, wave)
  constexpr int SUBSETS = W * 64 / D;  // groups of 8 partial rows, one thread per channel each
  static_assert(ROWS == SUBSETS * 8 && 8 % W == 0, "a thread adds up 8 partial rows of its channel");
  float* const acc_s = lds;                    // [sub][wave][channel]
  float* const part_s = acc_s + ROWS * D;      // [subset][channel]
  float* const l_s = part_s + SUBSETS * D;     // [sub][wave]
  float* const lpart_s = l_s + ROWS;
  float* const m_s = lpart_s + SUBSETS;        // [wave]

  const int tid = threadIdx.x & (W * 64 - 1), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int sub = lane / LPK, dg = lane % LPK;
  const int hk = h / (n_head / n_kv_head);

  // ---- first round trip: the token's request and position, its query, and (decode-only steps)
  // the block table entries of the first pass
  int qr = q_req[n];
  const int qpos = positions[n];
  uint4 qraw = *reinterpret_cast<const uint4*>(q + (long)n * ldq + (long)h * D + dg * 8);
  int r = n;
  if (!IDENT) {
    r = qr < 0 ? 0 : qr;  // waits for qr
    // a step that also holds prompt portions: their tokens are another kernel's, and count as padding here
    if (cu_q && cu_q[r + 1] - cu_q[r] != 1) qr = -1;
  }
  const int first_key = first_seen(qpos, window, chunked);   // (with a window: waits for qpos)
  if (SIDE != 0 && (qpos + 1 - first_key + keep_first > keys) != (SIDE < 0)) return;   // the whole workgroup
  const int first_chunk = first_key / 64;
  const int* bt = block_tables + (long)r * max_blocks;
  const bool weigh = score_bias != nullptr;   // sigmoid weights, no softmax
  const float bias_log2e = weigh ? score_bias[h] * 1.4426950408889634f : 0.f;
  const float slope_log2e = BIAS == 2 ? slopes[h] * 1.4426950408889634f : 0.f;

  float m = -INFINITY, l = 0.f;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;

  int c_base = keep_first > 0 ? 0 : first_chunk * 64;
  int kv_end = 0, kv_begin = 0;
  do {
    // a pass that lies wholly between the kept first keys and the window's first chunk: on to that chunk
    if (c_base >= keep_first && c_base < first_chunk * 64) c_base = first_chunk * 64;
    const int c0 = c_base + wave * 64;
    const int page_mask = (1 << page_shift) - 1;
    int page[LPK];
#pragma unroll
    for (int i = 0; i < LPK; ++i) {
      const int e = (c0 + i * KPI + sub) >> page_shift;
      page[i] = bt[e < max_blocks ? e : max_blocks - 1];
    }
    kv_end = qr < 0 ? 0 : qpos + 1;
    kv_begin = first_key;
    c_base += 64 * W;
    // a chunk without a visible key costs its wave nothing more (the same decision in all lanes)
    if (__builtin_amdgcn_readfirstlane((c0 >= kv_end) | ((c0 + 64 <= kv_begin) & (c0 >= keep_first)))) continue;
    // ---- second round trip: keys and values of this wave's chunk.  Every lane loads (a masked
    // key reads the pool's first row instead and is zeroed afterwards), so that no branch stands
    // between the loads.  Offsets are 32-bit byte offsets from the pools' bases.
    uint4 kraw[LPK], vraw[LPK];
    bool valid[LPK];
    float by_dist[LPK];
    const unsigned int lane_off = ((unsigned int)(hk << page_shift) * D + dg * 8) * 2u;
#pragma unroll
    for (int i = 0; i < LPK; ++i) {
      const int j = c0 + i * KPI + sub;
      valid[i] = (j >= kv_begin || j < keep_first) && (j < kv_end);
      const bool follow = valid[i] && (unsigned int)page[i] < (unsigned int)num_pages;
      const unsigned int row_off = ((unsigned int)page[i] * page_bytes) + (unsigned int)(j & page_mask) * (D * 2u);
      const unsigned int off = follow ? row_off + lane_off : 0u;
      kraw[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(kpool) + off);
      vraw[i] = *reinterpret_cast<const uint4*>(reinterpret_cast<const char*>(vpool) + off);
      if (BIAS == 1) by_dist[i] = dist_bias[(long)h * bias_len + distance_entry(qpos - j, bias_len)];
    }
#pragma unroll
    for (int i = 0; i < LPK; ++i)
      if (!valid[i]) vraw[i] = make_uint4(0, 0, 0, 0);  // its weight is 0, but 0 * NaN is not
    // ---- scores (in units of log2 e, so that exp2 serves)
    float s[LPK];
    float cmax = -INFINITY;
#pragma unroll
    for (int i = 0; i < LPK; ++i) {
      float dot = aw_dot2(qraw.x, kraw[i].x, 0.f);
      dot = aw_dot2(qraw.y, kraw[i].y, dot);
      dot = aw_dot2(qraw.z, kraw[i].z, dot);
      dot = aw_dot2(qraw.w, kraw[i].w, dot);
      s[i] = aw_group_sum<LPK>(dot) * scale_log2e;
    }
    // capped scores, in one branch around all keys: a test for every key is turned into a tanh for every key, capped or not
    if (cap_log2e > 0.f) {
#pragma unroll
      for (int i = 0; i < LPK; ++i) s[i] = cap_log2e * tanh_fast(s[i] * __builtin_amdgcn_rcpf(cap_log2e));
    }
#pragma unroll
    for (int i = 0; i < LPK; ++i) {
      if (BIAS == 1) s[i] = fmaf(by_dist[i], 1.4426950408889634f, s[i]);
      if (BIAS == 2) s[i] = fmaf(-slope_log2e, (float)(qpos - (c0 + i * KPI + sub)), s[i]);
      s[i] = valid[i] ? s[i] : -INFINITY;
      cmax = fmaxf(cmax, s[i]);
    }
    const float m_new = weigh ? 0.f : fmaxf(m, aw_wave_max(cmax));
    if (m_new != -INFINITY) {  // the same in all lanes; false only while the wave has seen no key
      const float alpha = __builtin_amdgcn_exp2f(m - m_new);  // m = -inf: 0
      l *= alpha;
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] *= alpha;
      m = m_new;
#pragma unroll
      for (int i = 0; i < LPK; i += 2) {
        // a masked key: exp2(-inf) = 0, and 1 / (1 + exp2(inf)) = 0
        const float pa = weigh ? __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(s[i] + bias_log2e))) : __builtin_amdgcn_exp2f(s[i] - m_new);
        const float pb = weigh ? __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-(s[i + 1] + bias_log2e))) : __builtin_amdgcn_exp2f(s[i + 1] - m_new);
        l += pa + pb;
        const unsigned int pp = pack_bf16x2(pa, pb);
        const unsigned int va[4] = {vraw[i].x, vraw[i].y, vraw[i].z, vraw[i].w};
        const unsigned int vb[4] = {vraw[i + 1].x, vraw[i + 1].y, vraw[i + 1].z, vraw[i + 1].w};
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          // (va.low half, vb.low half) and (va.high half, vb.high half): channel 2w and 2w+1 of both keys
          const unsigned int lo = __builtin_amdgcn_perm(vb[w], va[w], 0x05040100u);
          const unsigned int hi = __builtin_amdgcn_perm(vb[w], va[w], 0x07060302u);
          acc[2 * w] = aw_dot2(pp, lo, acc[2 * w]);
          acc[2 * w + 1] = aw_dot2(pp, hi, acc[2 * w + 1]);
        }
      }
    }
  } while (c_base < kv_end);
  if (qr < 0) return;  // padded token (the whole workgroup)

  // ---- merge: partial rows [sub][wave] of D channels; every key's weight sits on LPK lanes, so
  // lane dg == 0 speaks for the group's sum
  if (lane == 0) m_s[wave] = m;
  if (dg == 0) l_s[sub * W + wave] = l;
  {
    float4* dst = reinterpret_cast<float4*>(acc_s + (sub * W + wave) * D + dg * 8);
    dst[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
    dst[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
  }
  __syncthreads();
  {
    float mx = m_s[0];
#pragma unroll
    for (int w = 1; w < W; ++w) mx = fmaxf(mx, m_s[w]);
    if (sinks) mx = fmaxf(mx, sinks[h] * 1.4426950408889634f);   // the sink, in the scores' units of log2 e
    const int c = tid % D, sset = tid / D;  // this thread: channel c of the partial rows 8 * sset ..
    float a = 0.f, lt = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float f = __builtin_amdgcn_exp2f(m_s[i % W] - mx);  // a wave without keys: exp2(-inf) = 0, and its sums are 0
      a = fmaf(acc_s[(sset * 8 + i) * D + c], f, a);
      lt = fmaf(l_s[sset * 8 + i], f, lt);
    }
    part_s[sset * D + c] = a;
    if (c == 0) lpart_s[sset] = lt;
  }
  __syncthreads();
  if (tid < D) {
    float a = 0.f, lt = 0.f;
#pragma unroll
    for (int s2 = 0; s2 < SUBSETS; ++s2) {
      a += part_s[s2 * D + tid];
      lt += lpart_s[s2];
    }
    if (sinks) {
      // one more term of the denominator, with no value
      const float sink = sinks[h] * 1.4426950408889634f;
      float mx = sink;
#pragma unroll
      for (int w = 0; w < W; ++w) mx = fmaxf(mx, m_s[w]);
      lt += __builtin_amdgcn_exp2f(sink - mx);
    }
    float res = score_bias ? a : a / lt;
    if (gate) res *= __builtin_amdgcn_rcpf(1.0f + __expf(-bf16_to_float(gate[(long)n * ldg + h])));   // sigmoid gate of the head
    out[(long)n * ldo + (long)h * D + tid] = float_to_bf16(res);
  }
}
