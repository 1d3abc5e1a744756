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
//  * eight waves (four with many tokens and heads), each with one 64-key chunk in flight (sixteen 16-byte loads per lane), so a
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

// W: waves of the workgroup.  A context of up to 512 keys is one pass of eight waves; with more (token, head) pairs than
// the chip holds such workgroups at a time (two a compute unit, one with a head size of 128 and its 166 registers), four
// waves: more workgroups at a time, and fewer waves without a chunk under short contexts.  Eight / four waves, us: 32
// tokens x 25 heads of 64 behind 40, 150, 400 and 1,000 keys 8.0 / 5.3, 9.0 / 6.8, 16.7 / 16.6, 34.4 / 34.4; 256 x 25 behind 40
// and 400 40 / 20, 116 / 116 (5.6 TB/s); 40 x 16 of 128 behind 150 and 1,000 19.4 / 12.7, 64 / 59.  (With the cap's branch
// around a pass both are 1 to 10 % faster: 100 x 12 of 64 behind 150 and 1,000 keys 6.0 and 31.4.)
template <int D, bool IDENT, int BIAS, int W>
__global__ __launch_bounds__(W * 64) void paged_attention_decode_kernel(
    const bf16_t* __restrict__ q, long ldq, bf16_t* __restrict__ out, long ldo,
    const bf16_t* __restrict__ kpool, const bf16_t* __restrict__ vpool,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ positions,
    const int* __restrict__ q_req, const int* __restrict__ cu_q, int n_head, int n_kv_head, int page_shift,
    int num_pages, unsigned int page_bytes, float scale_log2e, int window, const float* __restrict__ sinks,
    float cap_log2e, const bf16_t* __restrict__ gate, long ldg, int keep_first, const float* __restrict__ score_bias,
    int chunked, const float* __restrict__ dist_bias, int bias_len, const float* __restrict__ slopes) {
  __shared__ __align__(16) float lds[aw_lds_floats<D, W>()];
  aw_decode<D, IDENT, BIAS, W>(q, ldq, out, ldo, kpool, vpool, block_tables, max_blocks, positions, q_req, cu_q, n_head, n_kv_head,
                               page_shift, num_pages, page_bytes, scale_log2e, window, sinks, cap_log2e, gate,
                               ldg, keep_first, score_bias, chunked, dist_bias, bias_len, slopes, blockIdx.x,
                               blockIdx.y, lds);
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
  dim3 grid(n_tokens, n_head);
#define AW_LAUNCH4(DD, ID, BI, W)                                                                              \
  hipLaunchKernelGGL((paged_attention_decode_kernel<DD, ID, BI, W>), grid, dim3(W * 64), 0, stream, (const bf16_t*)q, ldq, \
                     (bf16_t*)out, ldo, (const bf16_t*)kpool, (const bf16_t*)vpool, block_tables,          \
                     max_blocks, positions, q_req, cu_q, n_head, n_kv_head, page_shift, num_pages, page_bytes, \
                     scale_log2e, window, sinks, softcap > 0.f ? softcap * 1.4426950408889634f : 0.f, \
                     (const bf16_t*)gate, ldg, keep_first, score_bias, chunked, dist_bias, bias_len, slopes)
#define AW_LAUNCH3(DD, ID, BI)                 \
  do {                                         \
    if (many) AW_LAUNCH4(DD, ID, BI, 4);       \
    else AW_LAUNCH4(DD, ID, BI, 8);            \
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
