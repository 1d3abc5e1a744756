// Paged attention for the single tokens of a decode step (bfloat16 cache, head sizes 16, 32, 64
// and 128), laid out for latency.  The rule is the general kernel's (a query at position p sees
// the keys max(0, p-window+1)..p of its own request; reference: src/minigpt_infer/model.py:61-87
// and the Triton decode kernel src/minigpt_infer/attention/triton_paged.py:44-123).
//
// A decode step is a chain of dependent kernels, and this one used to be the longest link: four
// memory round trips in a row (token -> request -> lengths -> block table -> keys) and
// cross-lane reductions through LDS for every 64 keys.  Here:
//  * a token's position comes from the step's position array and, when token n is request n (a
//    decode-only step), its block table row is read at once, before the position is known:
//    two round trips, block table then keys and values.  Block table entries that turn out to
//    lie beyond the sequence are never followed (their keys are masked before the load), and
//    an entry's page number is clamped to the pool so that a stale entry cannot send a load
//    outside it;
//  * eight waves (four for short contexts with many tokens and heads), each with one 64-key chunk in flight (sixteen 16-byte loads per lane), so a
//    context of up to 512 keys is one pass;
//  * D/8 lanes share a key: scores with v_dot2_f32_bf16 on the packed rows as loaded, summed
//    over the D/8 lanes with DPP moves; one wave-wide maximum per chunk (DPP within rows of 16,
//    then the four rows' values through scalar registers); the weighted sum of values again with
//    v_dot2_f32_bf16, two keys at a time, the weights rounded to bfloat16 as the tile kernel
//    for prompts does;
//  * with `keep_first` > 0 a query behind a window also sees the keys at positions below keep_first: the first
//    pass then starts at key 0 and the passes behind the kept keys go on at the window's first chunk; with
//    `score_bias` a visible key's weight is sigmoid(score + score_bias[head]) and nothing is normalised;
//  * with `chunked` a query sees its own chunk of `window` positions; with a table of numbers by distance
//    (BIAS 1) a lane asks for its keys' numbers together with the keys; with a slope per head (BIAS 2) slope *
//    distance is taken off a score, behind the cap;
//  * the waves' partial results (maximum, sum, weighted values per key subgroup) are merged
//    through LDS once, in a fixed order.
#include "attention_decode_wide.h"
#include "launchers.h"

// Waves of a (token, head) pair.  A context of up to 512 keys is one pass of eight waves; with more pairs than the chip holds
// such workgroups at a time (two a compute unit, one with a head size of 128 and its 166 registers) four are better where
// contexts are short: more pairs at a time, and fewer waves without a chunk.  Behind long contexts four waves are a chain twice
// as long, which a few long requests among short ones then wait for.
//  AW_EIGHT: eight waves a pair.
//  AW_FOUR: four, a workgroup each: where no token can see more than AW_SHORT keys.
//  AW_HALVES: each token by its own length, which only the device knows: with up to AW_SHORT keys an even head's workgroup
//  has the odd head behind it as well, four waves each (the odd head's workgroup leaves at once), with more each head has eight.
//  The wait for the position in front of all other loads is what it costs, too much for heads of 16 and 32.
// us, always eight / always four / this rule: 64 tokens x 12 heads of 64 behind 1 to 256 keys 8.6 / 6.4 / 6.3 (AW_FOUR), behind
// 512 18.3 / 18.4 / 18.5, one behind 1,024 or 2,048 and the others behind 100 12.8 / 15.0 / 11.3 and 19.4 / 25.0 / 18.1; 64 x 16
// heads of 128 on 4 of keys behind 256 and 1,024 19.9 / 12.9 / 12.7 and 43.7 / 37.0 / 39.2; 48 x 8 of 128, one behind 2,048
// 24.8 / 30.7 / 24.7.  Worst case found: 171 x 12 of 64, half behind 60 and half behind 1,024 45.9 / 46.4 / 49.0.
enum { AW_EIGHT, AW_FOUR, AW_HALVES };
#define AW_SHORT(D) ((D) == 128 ? 512 : 256)
template <int D, bool IDENT, int BIAS, int WAVES>
__global__ __launch_bounds__(WAVES == AW_FOUR ? 256 : 512) void paged_attention_decode_kernel(
    const bf16_t* __restrict__ q, long ldq, bf16_t* __restrict__ out, long ldo,
    const bf16_t* __restrict__ kpool, const bf16_t* __restrict__ vpool,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ positions,
    const int* __restrict__ q_req, const int* __restrict__ cu_q, int n_head, int n_kv_head, int page_shift,
    int num_pages, unsigned int page_bytes, float scale_log2e, int window, const float* __restrict__ sinks,
    float cap_log2e, const bf16_t* __restrict__ gate, long ldg, int keep_first, const float* __restrict__ score_bias,
    int chunked, const float* __restrict__ dist_bias, int bias_len, const float* __restrict__ slopes) {
  constexpr int FOUR = (aw_lds_floats<D, 4>() + 3) & ~3, EIGHT = aw_lds_floats<D, 8>();
  __shared__ __align__(16) float lds[WAVES == AW_FOUR ? FOUR : (WAVES == AW_HALVES && 2 * FOUR > EIGHT ? 2 * FOUR : EIGHT)];
  const int n = blockIdx.x, h = blockIdx.y;
  bool four = WAVES == AW_FOUR;
  int half = 0;
  if (WAVES == AW_HALVES) {
    const int qpos = positions[n];
    four = qpos + 1 - first_seen(qpos, window, chunked) + keep_first <= AW_SHORT(D) && (h | 1) < n_head;
    if (four && (h & 1)) return;
    half = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
  }
  if (WAVES != AW_EIGHT && four)
    aw_decode<D, IDENT, BIAS, 4>(q, ldq, out, ldo, kpool, vpool, block_tables, max_blocks, positions, q_req, cu_q, n_head,
                                 n_kv_head, page_shift, num_pages, page_bytes, scale_log2e, window, sinks, cap_log2e, gate,
                                 ldg, keep_first, score_bias, chunked, dist_bias, bias_len, slopes, n, h + half,
                                 lds + half * FOUR);
  else if (WAVES != AW_FOUR)
    aw_decode<D, IDENT, BIAS, 8>(q, ldq, out, ldo, kpool, vpool, block_tables, max_blocks, positions, q_req, cu_q, n_head,
                                 n_kv_head, page_shift, num_pages, page_bytes, scale_log2e, window, sinks, cap_log2e, gate,
                                 ldg, keep_first, score_bias, chunked, dist_bias, bias_len, slopes, n, h, lds);
}

// positions[n]: absolute position of token n; q_req[n]: its request (block table row), -1 for a
// padded token.  identity != 0 promises q_req[n] is n or -1 (a decode-only step).  cu_q (optional,
// without identity): the requests' token offsets; tokens of requests that bring more than one token
// are then left to another kernel.  Refuses
// (MGPT_ERR_BAD_SHAPE) other head sizes than 16, 32, 64, 128, page sizes that are no power of two
// and pools of 4 GiB or more.
extern "C" int mgpt_paged_attention_decode_bf16(
    const void* q, long ldq, void* out, long ldo, const void* kpool, const void* vpool,
    const int* block_tables, int max_blocks, const int* positions, const int* q_req, const int* cu_q,
    int n_tokens, int n_head, int n_kv_head, int head_dim, int page_size, int num_pages, float scale, int window,
    int identity, const float* sinks, float softcap, const void* gate, long ldg, int keep_first, const float* score_bias,
    int chunked, const float* dist_bias, int bias_len, const float* slopes, hipStream_t stream) {
  if (n_tokens == 0) return MGPT_OK;
  if (!q || !out || !kpool || !vpool || !block_tables || !positions || !q_req) return MGPT_ERR_NULL;
  if (n_tokens < 0 || n_head <= 0 || n_kv_head <= 0 || (n_head % n_kv_head) != 0 || page_size <= 0 ||
      max_blocks <= 0 || num_pages <= 0 || window < 0 || (ldq % 8) != 0 || (identity && cu_q) || keep_first < 0 ||
      (score_bias && (sinks || softcap > 0.f)) || (dist_bias && (bias_len <= 0 || score_bias || softcap > 0.f)) || (slopes && (dist_bias || score_bias)))
    return MGPT_ERR_BAD_SHAPE;
  if (window == 0) keep_first = 0;
  if (n_head > 65535) return MGPT_ERR_TOO_LARGE;
  int page_shift = -1;
  for (int s = 0; s < 30; ++s)
    if ((1 << s) == page_size) page_shift = s;
  if (page_shift < 0) return MGPT_ERR_BAD_SHAPE;
  // the kernel addresses a pool by 32-bit byte offsets
  const long pool_bytes = (long)num_pages * n_kv_head * page_size * head_dim * 2;
  if (pool_bytes >= (1L << 32)) return MGPT_ERR_BAD_SHAPE;
  const unsigned int page_bytes = (unsigned int)(n_kv_head * page_size * head_dim * 2);
  const float scale_log2e = scale * 1.4426950408889634f;
  const bool many = (long)n_tokens * n_head > (head_dim == 128 ? 256 : 512);
  const long most = window > 0 ? (long)window + keep_first : (long)max_blocks * page_size;   // keys that a token can see
  dim3 grid(n_tokens, n_head);
#define AW_LAUNCH4(DD, ID, BI, WAVES)                                                                          \
  hipLaunchKernelGGL((paged_attention_decode_kernel<DD, ID, BI, WAVES>), grid, dim3(WAVES == AW_FOUR ? 256 : 512), 0, stream, \
                     (const bf16_t*)q, ldq, (bf16_t*)out, ldo, (const bf16_t*)kpool, (const bf16_t*)vpool, block_tables,          \
                     max_blocks, positions, q_req, cu_q, n_head, n_kv_head, page_shift, num_pages, page_bytes, \
                     scale_log2e, window, sinks, softcap > 0.f ? softcap * 1.4426950408889634f : 0.f, \
                     (const bf16_t*)gate, ldg, keep_first, score_bias, chunked, dist_bias, bias_len, slopes)
#define AW_LAUNCH3(DD, ID, BI)                 \
  do {                                         \
    if (many && most <= AW_SHORT(DD)) AW_LAUNCH4(DD, ID, BI, AW_FOUR);                    \
    else if (many && DD >= 64) AW_LAUNCH4(DD, ID, BI, (DD >= 64 ? AW_HALVES : AW_EIGHT)); \
    else AW_LAUNCH4(DD, ID, BI, AW_EIGHT);                                                \
  } while (0)
#define AW_LAUNCH2(DD, ID)                     \
  do {                                         \
    if (slopes) AW_LAUNCH3(DD, ID, 2);         \
    else if (dist_bias) AW_LAUNCH3(DD, ID, 1); \
    else AW_LAUNCH3(DD, ID, 0);                \
  } while (0)
#define AW_LAUNCH(DD)              \
  do {                             \
    if (identity) AW_LAUNCH2(DD, true); \
    else AW_LAUNCH2(DD, false);    \
  } while (0)
  switch (head_dim) {
    case 16: AW_LAUNCH(16); break;
    case 32: AW_LAUNCH(32); break;
    case 64: AW_LAUNCH(64); break;
    case 128: AW_LAUNCH(128); break;
    default: return MGPT_ERR_BAD_SHAPE;
  }
#undef AW_LAUNCH
#undef AW_LAUNCH2
#undef AW_LAUNCH3
#undef AW_LAUNCH4
  return mgpt_last_error();
}
