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
// A workgroup takes 32 Q consecutive queries of one request and one head, 32 per wave, with K groups of waves that share the keys.
// It walks the keys in stretches of 32 K: the stretch's key and value rows go from memory straight into LDS, gathered row by row
// through the block table, so any page size works and nothing outside the visible keys is loaded.  LDS holds two stretches
// at a time: while one is multiplied the next is on its way, with one barrier per stretch and no register for it.
//
// S = K Q^T uses the keys as the first MFMA operand, so a lane holds, for one query, 16 of 32 keys, in runs of four; those are
// exactly the k-slots of the second MFMA (values^T times P) if the values are read transposed with the same interleaving, so the
// probabilities never leave their registers.  The transposing LDS read of this chip (ds_read_b64_tr_b16) does that: the 16 lanes
// of a block point at 4 rows x 4 chunks of 4 channels, row j / 4 and chunk j % 4 for lane j, and lane i comes back with channel i
// of the four rows.  Running max, sum and rescaling per query are the usual online softmax: exp2(score * scale' - max) is one
// fused multiply-add and one v_exp_f32 (scale' holds log2 e), the maximum over the two lanes that share a query goes through
// one lane swap, and the row sum stays split over those lanes until the end.
//
// What bounds it is the softmax arithmetic (for 32 x 32 scores about 500 cycles of a wave beside 256 of the matrix units), so what
// counts is that waves of several workgroups share a SIMD: four at head sizes up to 64, held to 128 registers, where waves of
// 16 queries x 128 keys with the keys staged through registers had two, one on average.  us before / now, with keys, values and
// queries written anew in front of every call: 4 x 1,024 tokens x 25 heads of 64 90 / 38 (353 TFLOP/s of causal work), 8 x 1,024
// 152 / 65, 4 x 512 x 12 heads 22 / 15.3, 8 x 560 x 8 heads of 128 50 / 31; of the first of these the order of the tiles is worth 20.
// Error against 64 bits 0.00200 / 0.00196.  A running max that is left alone until it lags by 2^8 saves 3 % more and costs 4 % of
// the error: not taken.
#include "attention_prefill.h"
#include "launchers.h"

// Division of numbers below 2^31 by one that the host knows (0: never asked): a multiplication that is one short at most.
struct Divisor {
  unsigned int by, m;
  explicit Divisor(long d) : by((unsigned int)d), m(d > 0 ? (unsigned int)(0xffffffffL / d) : 0u) {}
  __device__ __forceinline__ unsigned int of(unsigned int x) const {
    const unsigned int q = __umulhi(x, m);
    return x - q * by >= by ? q + 1 : q;
  }
};
// Which tile of which request's head a block takes: n = requests x heads, of which a die has `own` to itself and `left` are dealt out.
struct PrefillDeal {
  Divisor n, own, left, head;
  unsigned int tiles;
};

template <int D, int Q, int K, int BIAS>
__global__ __launch_bounds__(64 * Q * K, (pf_waves<D, K>())) void prefill_attention_kernel(
    const bf16_t* __restrict__ q, long ldq, bf16_t* __restrict__ out, long ldo,
    const bf16_t* __restrict__ kpool, const bf16_t* __restrict__ vpool,
    const int* __restrict__ block_tables, int max_blocks, const int* __restrict__ cu_q,
    const int* __restrict__ seq_lens, int n_head, int n_kv_head, int page_size, float scale, int window,
    int single_below, const float* __restrict__ sinks, float softcap, const bf16_t* __restrict__ gate, long ldg,
    int keep_first, const float* __restrict__ score_bias, int chunked, const float* __restrict__ dist_bias,
    int bias_len, const float* __restrict__ slopes, PrefillDeal deal) {
  // Block b runs on die b % 8.  The tiles with the most keys come first.  All tiles of a request's head go to one die, whose L2 then has
  // its keys, as far as eight heads at a time go; the tiles of the heads left over are dealt out, so that no die has more than the
  // others, and (but for seven) no block is there in vain, which would wait for LDS like the others.  A die's turns are rounds of eight
  // tiles of each of its own heads with its share of the dealt ones in front.  us, all tiles of a head on one die and blocks up to a
  // multiple of eight heads / so: 1 request, 4,096 tokens behind 4,096, 1 head 148 / 49, 4 heads 129 / 74, 12 heads 178 / 148; 640 tokens x
  // 12 heads 13.0 / 10.4, x 9 behind 2,000 34.6 / 21.8, behind a window of 256 17.9 / 11.0.
  const unsigned int at = (blockIdx.y * gridDim.x + blockIdx.x) >> 3, die = blockIdx.x & 7;
  const unsigned int round = deal.n.of(at), in = at - round * deal.n.by, own = deal.own.by, left = deal.left.by;
  const bool dealt = in < (round < deal.tiles >> 3 ? left : ((deal.tiles & 7) * left + 7) >> 3);
  unsigned int who, turn;
  if (!dealt && own == 0) return;
  if (dealt) {
    const unsigned int i = (round * left + in) * 8 + die;
    turn = deal.left.of(i);
    who = own * 8 + i - turn * left;
  } else {
    const unsigned int i = at - (round < deal.tiles >> 3 ? (round + 1) * left : round * left + (((deal.tiles & 7) * left + 7) >> 3));
    turn = deal.own.of(i);
    who = (i - turn * own) * 8 + die;
  }
  if (turn >= deal.tiles) return;
  const int tile = __builtin_amdgcn_readfirstlane((int)(deal.tiles - 1 - turn)), req = __builtin_amdgcn_readfirstlane((int)deal.head.of(who));
  extern __shared__ __align__(16) bf16_t pf_lds[];
  pf_tile<D, Q, K, BIAS>(q, ldq, out, ldo, kpool, vpool, block_tables, max_blocks, cu_q, seq_lens, n_head, n_kv_head, page_size, scale,
                      window, single_below, sinks, softcap, gate, ldg, keep_first, score_bias, chunked,
                      dist_bias, bias_len, slopes, tile, req, __builtin_amdgcn_readfirstlane((int)who - req * n_head), pf_lds);
}

// One workgroup per (tile of 32 or 64 queries, request, head); max_q_len sizes the grid and is the host's
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
  const long whos = (long)n_req * n_head;
  constexpr long PF_GRID_X = 0xffffffffL / 512 / 8 * 8;   // threads of a grid along x, whole turns of all dies
#define PF_LAUNCH2(DD, QQ, KK, BI)                                                                                  \
  {                                                                                                                 \
    constexpr int lds_bytes = pf_lds_bytes<DD, QQ, KK, BI>();                                                       \
    static bool allowed = false; /* more LDS than a kernel gets without asking */                                   \
    if (!allowed) {                                                                                                 \
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(prefill_attention_kernel<DD, QQ, KK, BI>), \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);             \
      if (e != hipSuccess) return (int)e;                                                                           \
      allowed = true;                                                                                               \
    }                                                                                                               \
    const long q_tiles = ((long)max_q_len + QQ * PF_W - 1) / (QQ * PF_W);                                           \
    const long turns = q_tiles / 8 * whos + (q_tiles % 8 * (whos % 8) + 7) / 8 + q_tiles % 8 * (whos / 8);          \
    if (8 * turns > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;                                                         \
    const long x = 8 * turns <= PF_GRID_X ? 8 * turns : PF_GRID_X;                                                  \
    const dim3 grid((unsigned int)x, (unsigned int)((8 * turns + x - 1) / x));                                      \
    hipLaunchKernelGGL((prefill_attention_kernel<DD, QQ, KK, BI>), grid, dim3(64 * QQ * KK), lds_bytes, stream,     \
                       (const bf16_t*)q, ldq, (bf16_t*)out, ldo, (const bf16_t*)kpool, (const bf16_t*)vpool,        \
                       block_tables, max_blocks, cu_q, seq_lens, n_head, n_kv_head, page_size, scale, window,       \
                       single_below, sinks, softcap, (const bf16_t*)gate, ldg, keep_first, score_bias, chunked,     \
                       dist_bias, bias_len, slopes,                                                                 \
                       PrefillDeal{Divisor(whos), Divisor(whos / 8), Divisor(whos % 8), Divisor(n_head), (unsigned int)q_tiles}); \
  }
#define PF_LAUNCH(DD, QQ, KK)                                           \
  {                                                                     \
    if (slopes) PF_LAUNCH2(DD, QQ, KK, 2)                               \
    else if (dist_bias) PF_LAUNCH2(DD, QQ, KK, 1)                       \
    else PF_LAUNCH2(DD, QQ, KK, 0)                                      \
  }
  const long tiles = ((long)max_q_len + 63) / 64 * n_req * n_head;
  const long most = window > 0 ? (long)window + keep_first : (long)max_blocks * page_size;   // keys that a query can see
  // Few tiles (64 queries): 32 queries a workgroup, in four waves, and eight where even those leave compute units idle and there
  // are keys for them.  64 queries with four waves / 32 with four / 32 with eight (as before), us: 2 x 1,024 tokens x 8 heads 21.9 / 15.5 /
  // 18.1 (21.0); 512 tokens behind 448 x 12 heads 19.7 / 14.7 / 11.7 (17.9); 128 tokens x 8 heads 6.4 / 5.5 / 6.3 (6.8); 64 tokens behind 900
  // x 12 heads 21.0 / 14.6 / 11.4 (16.1); 384 tiles, 4 x 512 tokens x 12 heads 15.3 / 17.1 / 22.3 (21.9).
  const bool few = tiles <= 320, fewer = tiles <= 128 && (max_q_len > 128 || most > 1024);
  switch (head_dim) {
    case 32: if (fewer) PF_LAUNCH(32, 1, 8) else if (few) PF_LAUNCH(32, 1, 4) else PF_LAUNCH(32, 2, 2) break;
    case 64: if (fewer) PF_LAUNCH(64, 1, 8) else if (few) PF_LAUNCH(64, 1, 4) else PF_LAUNCH(64, 2, 2) break;
    case 96: PF_LAUNCH(96, 2, 2); break;
    case 128: PF_LAUNCH(128, 2, 2); break;
    default: return MGPT_ERR_BAD_SHAPE;
  }
#undef PF_LAUNCH
#undef PF_LAUNCH2
  return mgpt_last_error();
}
