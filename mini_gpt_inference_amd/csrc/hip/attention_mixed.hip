// Attention of a step that has both, single tokens of decoding requests and prompt portions (bfloat16, head sizes 64 and 128),
// in one launch.
//
// The two kinds of tokens have kernels of their own (attention_decode_wide.hip, attention_prefill.hip), neither of which fills
// the chip in such a step: a portion of 512 tokens x 12 heads is 192 tiles, eleven decoding requests are 132 workgroups, on 256
// compute units, one behind the other 11.4 + 8.9 us a layer.  Here the first workgroups of the launch are tiles and the ones
// behind them (token, head) pairs, both with the bodies of those kernels, so that they run side by side.  A pair's workgroup
// holds a tile's LDS and registers, a compute unit or half of one, so it is done for up to 256 pairs; more go to their own kernel.
//
// Where a tile has four waves (head size 128, and 64 with many tiles or short contexts) a pair has four as well, a pass of 256 keys at a time,
// and behind long contexts that chain outlasts tiles and eight waves one behind the other: 8 requests x 8 heads of 128 beside
// a portion of 256 tokens, behind 8,000 keys: one behind the other 84.7 us, here 110.  Lengths are known on the
// device only (a recorded launch serves steps of any length), so tokens that see more than `keys` keys are left out here and
// done by a second launch with eight waves each, which is made where the block table or the window allows such tokens at
// all: 81.6 us; where no token is that long it costs 1.5 us.
//
// Tiles are numbered over the requests on the device, 32 or 64 queries each: the launch is sized by how many tiles so many tokens of
// so many requests can make at most, not by the longest portion times the requests.
#include "attention_decode_wide.h"
#include "attention_prefill.h"
#include "launchers.h"

struct MixedArgs {
  const bf16_t* q; long ldq; bf16_t* out; long ldo;
  const bf16_t* kpool; const bf16_t* vpool;
  const int* block_tables; int max_blocks;
  const int* positions; const int* q_req; const int* cu_q; const int* seq_lens;
  int n_decode, first_req, n_req, tiles, single_below, n_head, n_kv_head, page_size, page_shift, num_pages;
  unsigned int page_bytes;
  float scale; int window;
  const float* sinks; float softcap;
  const bf16_t* gate; long ldg;
  int keep_first; const float* score_bias; int chunked;
  int keys;                  // a pair with four waves: up to so many keys
};

// Pair number b of the step's single tokens and heads.
template <int D, bool IDENT, int W, int SIDE>
__device__ __forceinline__ void mx_pair(const MixedArgs& a, int b, float* lds) {
  const float log2e = 1.4426950408889634f;
  aw_decode<D, IDENT, 0, W, SIDE>(a.q, a.ldq, a.out, a.ldo, a.kpool, a.vpool, a.block_tables, a.max_blocks, a.positions,
                                  a.q_req, IDENT ? nullptr : a.cu_q, a.n_head, a.n_kv_head, a.page_shift, a.num_pages,
                                  a.page_bytes, a.scale * log2e, a.window, a.sinks,
                                  a.softcap > 0.f ? a.softcap * log2e : 0.f, a.gate, a.ldg, a.keep_first, a.score_bias,
                                  a.chunked, nullptr, 0, nullptr, b % a.n_decode, b / a.n_decode, lds, a.keys);
}

// IDENT: the single tokens are those of requests 0 .. n_decode - 1; else q_req names a token's request, and requests with more
// than one token are passed over
template <int D, int Q, int K, bool IDENT>
__global__ __launch_bounds__(64 * Q * K, (pf_waves<D, K>())) void mixed_attention_kernel(MixedArgs a) {
  constexpr int W = Q * K, QT = Q * PF_W;
  static_assert(W == 4 || W == 8, "what a pair's kernel takes");
  static_assert(aw_lds_floats<D, W>() * (int)sizeof(float) <= pf_lds_bytes<D, Q, K, 0>(), "one kind's LDS serves the other");
  extern __shared__ __align__(16) bf16_t mx_lds[];
  int b = blockIdx.x;
  const int n_tiles = a.tiles * a.n_head;
  if (b >= n_tiles) {
    b -= n_tiles;
    mx_pair<D, IDENT, W, W == 8 ? 0 : 1>(a, b, reinterpret_cast<float*>(mx_lds));
    return;
  }
  // the tiles with the most keys first
  int tile = a.tiles - 1 - b / a.n_head;
  const int h = b % a.n_head;
  const int* cu_q = a.cu_q + a.first_req;
  const int r = piece_owner(a.n_req, tile, [&](int i) {
    const int start = cu_q[i], len = cu_q[i + 1] - start;
    return len == 1 && start < a.single_below ? 0 : (len + QT - 1) / QT;
  });
  if (r < 0) return;                                    // beyond the step's tiles: the whole workgroup
  pf_tile<D, Q, K, 0>(a.q, a.ldq, a.out, a.ldo, a.kpool, a.vpool, a.block_tables, a.max_blocks, a.cu_q, a.seq_lens, a.n_head,
                   a.n_kv_head, a.page_size, a.scale, a.window, a.single_below, a.sinks, a.softcap, a.gate, a.ldg, a.keep_first,
                   a.score_bias, a.chunked, nullptr, 0, nullptr, __builtin_amdgcn_readfirstlane(tile),
                   __builtin_amdgcn_readfirstlane(a.first_req + r), h, mx_lds);
}

// Single tokens that see more than a.keys keys.
template <int D, bool IDENT>
__global__ __launch_bounds__(512) void long_pairs_kernel(MixedArgs a) {
  __shared__ __align__(16) float lds[aw_lds_floats<D, 8>()];
  mx_pair<D, IDENT, 8, -1>(a, blockIdx.x, lds);
}

template <int D, int Q, int K, bool IDENT>
static int launch(MixedArgs a, int n_tokens, hipStream_t stream) {
  constexpr int bytes = pf_lds_bytes<D, Q, K, 0>(), QT = Q * PF_W;
  const long tiles = ((long)n_tokens + (long)(QT - 1) * (a.n_req < n_tokens ? a.n_req : n_tokens)) / QT;
  if ((tiles + a.n_decode) * a.n_head > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;
  a.tiles = (int)tiles;
  static bool allowed = false;  // more LDS than a kernel gets without asking
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(mixed_attention_kernel<D, Q, K, IDENT>),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  hipLaunchKernelGGL((mixed_attention_kernel<D, Q, K, IDENT>), dim3((a.tiles + a.n_decode) * a.n_head), dim3(64 * Q * K), bytes, stream,
                     a);
  if constexpr (Q * K == 4) {
    const long most = a.window > 0 ? (long)a.window + a.keep_first : (long)a.max_blocks * a.page_size;   // that a token can see
    if (most > a.keys)
      hipLaunchKernelGGL((long_pairs_kernel<D, IDENT>), dim3(a.n_decode * a.n_head), dim3(512), 0, stream, a);
  }
  return mgpt_last_error();
}

// The step's first n_decode tokens: identity != 0: one each of requests 0 .. n_decode - 1; else those of them whose request
// brings no other token.  And the tokens of requests first_req .. first_req + n_req - 1, n_tokens at most, without requests that
// bring a single token as one of the step's first single_below.  positions, q_req: per token; cu_q, seq_lens, block_tables: per
// request, from request 0 on.  The rest as mgpt_prefill_attention_bf16.  Refused (MGPT_ERR_BAD_SHAPE, nothing launched): other
// head sizes than 64 and 128, page sizes that are no power of two, pools of 4 GiB and more, more than 256 (token, head) pairs.
extern "C" int mgpt_mixed_attention_bf16(
    const void* q, long ldq, void* out, long ldo, const void* kpool, const void* vpool, const int* block_tables, int max_blocks,
    const int* positions, const int* q_req, const int* cu_q, const int* seq_lens, int n_decode, int identity, int first_req,
    int n_req, int n_tokens, int single_below, int n_head, int n_kv_head, int head_dim, int page_size, int num_pages, float scale,
    int window, const float* sinks, float softcap, const void* gate, long ldg, int keep_first, const float* score_bias,
    int chunked, hipStream_t stream) {
  if (!q || !out || !kpool || !vpool || !block_tables || !positions || !q_req || !cu_q || !seq_lens) return MGPT_ERR_NULL;
  if (n_decode <= 0 || first_req < 0 || n_req <= 0 || n_tokens <= 0 || n_head <= 0 || n_kv_head <= 0 || n_head % n_kv_head != 0 ||
      page_size <= 0 || (page_size & (page_size - 1)) != 0 || num_pages <= 0 || max_blocks <= 0 || window < 0 || ldq % 8 != 0 ||
      ldo % 4 != 0 || (((size_t)out) & 7) != 0 || !(scale > 0.f) || keep_first < 0 || (score_bias && (sinks || softcap > 0.f)) ||
      (head_dim != 64 && head_dim != 128) || (long)n_decode * n_head > 256 ||
      (long)num_pages * n_kv_head * page_size * head_dim * 2 >= (1L << 32))
    return MGPT_ERR_BAD_SHAPE;
  int page_shift = 0;
  while ((1 << page_shift) < page_size) ++page_shift;
  // What four waves lose on a token against eight, 0.005 us a key, is to be no more than what the tiles beside them take and a
  // launch, 7 us for a portion of 64 tokens, 13 for 512 (19 are saved there, but a token beyond the line then waits for those
  // below it: one behind 8,363 keys and others behind some 4,000 beside 630 tokens 97 us as two launches, 113 with a line at
  // 4,096 keys, 93 here).  Head size 64 comes here with
  // hundreds of tiles, where it loses less, or with 1,024 keys at most.
  const int keys = head_dim == 64 ? 16384 : (n_tokens < 512 ? 1024 + 3 * n_tokens : 2560);
  const MixedArgs a = {(const bf16_t*)q, ldq, (bf16_t*)out, ldo, (const bf16_t*)kpool, (const bf16_t*)vpool, block_tables,
                       max_blocks, positions, q_req, cu_q, seq_lens, n_decode, first_req, n_req, 0, single_below, n_head,
                       n_kv_head, page_size, page_shift, num_pages, (unsigned int)(n_kv_head * page_size * head_dim * 2), scale,
                       window, sinks, softcap, (const bf16_t*)gate, ldg, window == 0 ? 0 : keep_first, score_bias, chunked,
                       keys};
  // Tiles of 32 queries while the tiles are few, as for prompt portions alone: eight waves each where that leaves a compute unit
  // for every workgroup, else four, of which two workgroups share one (11 single tokens behind 500 keys beside a portion of 512
  // tokens x 12 heads: 11.0 us, with eight 12.1, with tiles of 64 queries and eight waves 11.8; 3 of them: 9.8 / 9.8 / 11.2), also beside
  // short portions (64 tokens, 5 single ones, 8 heads: 6.3 / 7.8 / 7.5).  A pair has as many waves as a tile, so where tokens may
  // see more than 1,024 keys there are eight.  The tiles' number is taken for up to eight portions: a padded step's n_req is its
  // capacity, of which it fills few.
  const long portions = n_req < 8 ? n_req : 8, likely = (n_tokens + 63L) / 64 + portions;
  const long wgs = ((n_tokens + 31L) / 32 + portions + n_decode) * n_head;
  const long most = window > 0 ? (long)window + a.keep_first : (long)max_blocks * page_size;
#define MX_LAUNCH(D, Q, K) return identity ? launch<D, Q, K, true>(a, n_tokens, stream) : launch<D, Q, K, false>(a, n_tokens, stream)
  if (head_dim == 128) MX_LAUNCH(128, 2, 2);
  if (likely * n_head > 320) MX_LAUNCH(64, 2, 2);
  if (most <= 1024 && (wgs > 256 || n_tokens <= 128)) MX_LAUNCH(64, 1, 4);
  if (wgs > 256) MX_LAUNCH(64, 2, 4);
  MX_LAUNCH(64, 1, 8);
#undef MX_LAUNCH
}
