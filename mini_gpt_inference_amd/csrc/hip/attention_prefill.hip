// Paged causal attention for prompt portions in bfloat16 on the MFMA units (flash style).
//
// Same rule as the general kernel: a query at absolute position p sees the keys
// max(0, p-window+1)..p of its own request, some of them written by earlier steps (a portion
// with ctx > 0 is the offset-causal case of src/minigpt_infer/batch.py:202-227), scores scaled,
// softmax and all sums in float32 (src/minigpt_infer/model.py:61-87).
//
// With `keep_first` > 0 a query behind a window also sees the keys at positions below keep_first (a tile walks
// the stretches of those keys first, then the window's); with `score_bias` a visible key's weight is
// sigmoid(score + score_bias[head]) and nothing is normalised.  With `chunked` a query sees its own chunk of
// `window` positions instead of the last `window`.
//
// With a slope per head (BIAS 2) slope * distance is taken off a score, behind the cap.
// With a table of numbers by distance (BIAS 1; in the scores' units before log2 e) the numbers that a step's
// stretch of keys needs for the tile's 64 queries, one per distance, lie in LDS in the order of the key, so that a
// lane's four neighbouring keys read four neighbouring numbers.
//
// A workgroup takes 64 consecutive queries of one request and one head, 16 per wave (four waves,
// or eight in two groups that share the keys between them, see the kernel).  It walks the keys in blocks of 128 (aligned to multiples of 128 of the key position):
// the block's key and value rows go to LDS as they are, gathered row by row through the block
// table, so any page size works and nothing outside [begin, end) is loaded.  LDS holds two
// blocks: while one is multiplied, the next (fetched from memory into registers a block earlier)
// is put beside it and the one after is sent for, with one barrier per block.
//
// S = K Q^T uses the keys as the first MFMA operand, so a lane holds, for one query, four
// neighbouring keys of each 16-key tile; those are exactly the k-slots of the second MFMA
// (values^T times P) if the values are read transposed with the same interleaving, so the
// probabilities never leave their registers.  The transposing LDS read of this chip
// (ds_read_b64_tr_b16) does that: the 16 lanes of a block point at 4 rows x 4 chunks of 4
// channels, row j / 4 and chunk j % 4 for lane j, and lane i comes back with channel i of the
// four rows.  Running max, sum and rescaling per query are the usual online softmax, kept short because at head size 64 it, not the MFMAs, is what a block
// costs: exp2(score * scale' - max) is one fused multiply-add and one v_exp_f32 (scale' holds
// log2 e), the maximum over the four lanes that share a query goes through two lane swaps
// instead of LDS, and the row sum stays split over those lanes until the end.
#include "attention_prefill.h"
#include "launchers.h"

template <int D, int G, int BIAS>
__global__ __launch_bounds__(256 * G) void prefill_attention_kernel(
    const bf16_t* __restrict__ q, long ldq, bf16_t* __restrict__ out, long ldo,
    const bf16_t* __restrict__ kpool, const bf16_t* __restrict__ vpool,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ cu_q,
    const int* __restrict__ seq_lens, int n_head, int n_kv_head, int page_size, float scale, int window,
    int single_below, const float* __restrict__ sinks, float softcap, const bf16_t* __restrict__ gate, long ldg,
    int keep_first, const float* __restrict__ score_bias, int chunked, const float* __restrict__ dist_bias,
    int bias_len, const float* __restrict__ slopes) {
  extern __shared__ __align__(16) bf16_t pf_lds[];
  pf_tile<D, G, BIAS>(q, ldq, out, ldo, kpool, vpool, block_tables, max_blocks, cu_q, seq_lens, n_head, n_kv_head, page_size, scale,
                      window, single_below, sinks, softcap, gate, ldg, keep_first, score_bias, chunked,
                      dist_bias, bias_len, slopes, blockIdx.x, blockIdx.y, blockIdx.z, pf_lds);
}

// One workgroup per (64-query tile, request, head); max_q_len sizes the grid and is the host's
// upper bound on the tokens any request brings (a request may bring none: its workgroups leave at
// once).  single_below: requests that bring exactly one token, and that as one of the step's first
// single_below tokens, are left to another kernel.  Head
// sizes 32, 64, 96, 128 and a positive scale; others are refused.
extern "C" int mgpt_prefill_attention_bf16(
    const void* q, long ldq, void* out, long ldo, const void* kpool, const void* vpool,
    const int* block_tables, int max_blocks, const int* cu_q, const int* seq_lens, int n_req,
    int max_q_len, int n_head, int n_kv_head, int head_dim, int page_size, float scale, int window,
    int single_below, const float* sinks, float softcap, const void* gate, long ldg, int keep_first,
    const float* score_bias, int chunked, const float* dist_bias, int bias_len, const float* slopes, hipStream_t stream) {
  if (n_req == 0 || max_q_len == 0) return MGPT_OK;
  if (!q || !out || !kpool || !vpool || !block_tables || !cu_q || !seq_lens) return MGPT_ERR_NULL;
  if (n_req < 0 || max_q_len < 0 || n_head <= 0 || n_kv_head <= 0 || (n_head % n_kv_head) != 0 ||
      page_size <= 0 || max_blocks <= 0 || window < 0 || (ldq % 8) != 0 || (ldo % 4) != 0 ||
      (((size_t)out) & 7) != 0 || !(scale > 0.f) || keep_first < 0 || (score_bias && (sinks || softcap > 0.f)) ||
      (dist_bias && (bias_len <= 0 || score_bias || softcap > 0.f)) || (slopes && (dist_bias || score_bias)))
    return MGPT_ERR_BAD_SHAPE;
  if (window == 0) keep_first = 0;
  if (n_req > 65535 || n_head > 65535) return MGPT_ERR_TOO_LARGE;
  dim3 grid((max_q_len + PF_QT - 1) / PF_QT, n_req, n_head);
#define PF_LAUNCH2(DD, GG, BI)                                                                                      \
  {                                                                                                                 \
    constexpr int lds_bytes = pf_lds_bytes<DD, GG, BI>();                                                            \
    static bool allowed = false; /* more LDS than a kernel gets without asking */                                   \
    if (!allowed) {                                                                                                 \
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(prefill_attention_kernel<DD, GG, BI>), \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);             \
      if (e != hipSuccess) return (int)e;                                                                           \
      allowed = true;                                                                                               \
    }                                                                                                               \
    hipLaunchKernelGGL((prefill_attention_kernel<DD, GG, BI>), grid, dim3(256 * GG), lds_bytes, stream,             \
                       (const bf16_t*)q, ldq, (bf16_t*)out, ldo, (const bf16_t*)kpool, (const bf16_t*)vpool,        \
                       block_tables, max_blocks, cu_q, seq_lens, n_head, n_kv_head, page_size, scale, window,       \
                       single_below, sinks, softcap, (const bf16_t*)gate, ldg, keep_first, score_bias, chunked,     \
                       dist_bias, bias_len, slopes);                                                                        \
  }
#define PF_LAUNCH(DD, GG)                                               \
  {                                                                     \
    if (slopes) PF_LAUNCH2(DD, GG, 2)                                   \
    else if (dist_bias) PF_LAUNCH2(DD, GG, 1)                           \
    else PF_LAUNCH2(DD, GG, 0)                                          \
  }
  // Two wave groups halve the walk of a tile over its keys; one group leaves LDS for a second
  // workgroup on the compute unit.  The first serves a step with few tiles, the second one with many.
  const long tiles = (long)grid.x * grid.y * grid.z;
  const bool two = tiles <= 320;
  switch (head_dim) {
    case 32: if (two) PF_LAUNCH(32, 2) else PF_LAUNCH(32, 1) break;
    case 64: if (two) PF_LAUNCH(64, 2) else PF_LAUNCH(64, 1) break;
    case 96: PF_LAUNCH(96, 1); break;
    case 128: PF_LAUNCH(128, 1); break;
    default: return MGPT_ERR_BAD_SHAPE;
  }
#undef PF_LAUNCH
#undef PF_LAUNCH2
  return mgpt_last_error();
}
