// Tiled bfloat16 matrix product on the MFMA units for many rows (prompt portions):
// out[n, o] = sum_k act[n, k] * W[o, k] (+ bias[o]) with an optional GELU-tanh or residual-add
// epilogue, or one that also stores new keys and values into their cache pages (nn.Linear as in
// src/minigpt_infer/model.py:43-44,96-101; the cache write of src/minigpt_infer/cache/paged.py:125-137).
//
// One kernel template, five tile shapes.  What bounds a tile kernel on this machine is the traffic
// between LDS and the MFMA units: a wave that owns R x C outputs reads (R + C) * 32 operand values
// from LDS for R * C * 32 multiply-adds, so a wave's tile is as large as the problem allows while
// it still gives every compute unit work: 256 x 256 outputs per workgroup (eight waves of
// 128 x 64) for large problems, down to 32 x 32 (four waves of 16 x 16) for a prompt portion of a
// hundred tokens.  A step along k is 64 long.
//
// The workgroup stages its slice of the activations and of W in LDS twice over.  A row of a slice
// is 128 bytes, eight chunks of 16; chunk c of row r lies at position c ^ (r & 7) of its row.  With
// that, the 16 rows x 4 chunks that an MFMA operand read (ds_read_b128) touches are served at the
// full 256 bytes per clock; rows padded by 16 bytes, the usual remedy, take twice as long on this
// LDS (measured with SQ_LDS_BANK_CONFLICT), and unpadded rows four times.
//
// Two steps' worth of loads are in flight: while step s is multiplied, the chunks of step s + 1
// (loaded during step s - 1) go into the other LDS buffer and those of step s + 2 are sent for,
// both spread between the MFMAs, because LDS takes writes at half the rate of reads and all at
// once they would hold every wave up.  MFMA operands are read from LDS two groups of MFMAs ahead
// of their use.  W is the first MFMA operand, so a lane ends up with four neighbouring output
// columns of one row and stores them as one vector.
//
// Tiles are numbered so that the workgroups that run at the same time on an XCD (which has an L2
// of its own) form a block of a few row tiles by a few column tiles, whose operands that L2 holds.
//
// Five further variants (DIRECT) send the slices from memory straight into LDS
// (global_load_lds_dwordx4) instead of through registers: three or four stages for a long inner
// size, 128 x 192 tiles for wide outputs under many rows, and four or six stages of 32 x 32 tiles for
// the rows of a decode step under a large matrix; see the kernel, choose_direct and launch_any.  Four more, for
// many rows, also let the workgroup's two halves read and multiply in turn (linear_mfma_halves_kernel, choose_large).
#include "common.h"
#include <type_traits>
#include "launchers.h"

typedef __attribute__((__vector_size__(8 * sizeof(short)))) short bf16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

#define MM_EPI_NONE 0
#define MM_EPI_GELU 1
#define MM_EPI_RESIDUAL 2
#define MM_EPI_QKV 3   // store, and scatter the key and value columns into their cache pages
#define MM_EPI_RELU2 5 // max(v, 0)^2
#define MM_EPI_XIELU 4 // a_p v^2 + v / 2 for v > 0, a_n (exp(v) - 1 - v) + v / 2 else, (a_p, a_n) from MfmaScatter::epi_coef

__device__ __forceinline__ float mfma_xielu(float v, float a_p, float a_n) {
  return v > 0.f ? fmaf(a_p * v, v, 0.5f * v) : fmaf(a_n, (__expf(v) - 1.0f) - v, 0.5f * v);
}

// where the key and value columns of a fused QKV product go (src/minigpt_infer/cache/paged.py:125-137)
struct MfmaScatter {
  bf16_t* kpool;
  bf16_t* vpool;
  const int* slot_mapping;  // per row: page * page_size + offset, or -1 for a padded row
  int q_width, kv_width, head_dim, n_kv_head, page_size;
  // Rows in groups that each multiply a matrix of their own (experts): row r belongs to group
  // r / group_rows, whose matrix is w + row_expert[group] * w_stride (a negative entry: the group is
  // not in use); row_valid[r] < 0 marks padding at the end of a group.  Null: one matrix for all rows.
  const int* row_expert = nullptr;
  const int* row_valid = nullptr;
  int group_rows = 0;
  long w_stride = 0;
  const float* epi_coef = nullptr;   // MM_EPI_XIELU: the two coefficients
};

// The bias of the four neighbouring output columns oc..oc+3 a lane holds.
__device__ __forceinline__ void mfma_bias4(const float* __restrict__ bias, int oc, int n_out, bool vec, float b4[4]) {
  b4[0] = b4[1] = b4[2] = b4[3] = 0.f;
  if (!bias) return;
  if (vec) {
    const float4 t = *reinterpret_cast<const float4*>(bias + oc);
    b4[0] = t.x; b4[1] = t.y; b4[2] = t.z; b4[3] = t.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) b4[e] = oc + e < n_out ? bias[oc + e] : 0.f;
  }
}

// Stores the four columns oc..oc+3 of row n: bias, activation, then a plain store, an add into
// the residual stream, or a store that also puts the four values at cache_dst (a key's or value's
// place in its cache page; null for query columns and rows without a slot).
// `vec`: the four columns can go as one aligned vector.
template <int EPI, typename OT>
__device__ __forceinline__ void mfma_store4(const f32x4_t& a, const float b4[4], OT* __restrict__ out, long ldo,
                                            int n, int oc, int n_out, bool vec, bf16_t* cache_dst, float a_p = 0.f,
                                            float a_n = 0.f) {
  OT* orow = out + (long)n * ldo;
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = a[e] + b4[e];
    if (EPI == MM_EPI_GELU) v[e] = gelu_tanh_fast(v[e]);
    if (EPI == MM_EPI_RELU2) v[e] = relu_squared(v[e]);
    if (EPI == MM_EPI_XIELU) v[e] = mfma_xielu(v[e], a_p, a_n);
  }
  if (vec && sizeof(OT) == 4) {
    float4* dst = reinterpret_cast<float4*>(orow + oc);
    if (EPI == MM_EPI_RESIDUAL) {
      const float4 old = *dst;
      *dst = make_float4(old.x + v[0], old.y + v[1], old.z + v[2], old.w + v[3]);
    } else {
      *dst = make_float4(v[0], v[1], v[2], v[3]);
    }
  } else if (vec && EPI != MM_EPI_RESIDUAL) {
    uint2 pk;
    pk.x = pack_bf16x2(v[0], v[1]);
    pk.y = pack_bf16x2(v[2], v[3]);
    *reinterpret_cast<uint2*>(orow + oc) = pk;
    // the four columns lie in one head (the launcher checks that sizes are multiples of 4)
    if (EPI == MM_EPI_QKV && cache_dst) *reinterpret_cast<uint2*>(cache_dst) = pk;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int o = oc + e;
      if (o >= n_out) continue;
      if (EPI == MM_EPI_RESIDUAL) {
        orow[o] = from_float<OT>(to_float<OT>(orow[o]) + v[e]);
      } else {
        orow[o] = from_float<OT>(v[e]);
      }
    }
  }
}

// Deals the workgroup ids out so that an XCD's workgroups (ids that agree modulo 8 go to the same
// XCD, which has an L2 of its own) are neighbours in tile order.
__device__ __forceinline__ int mfma_xcd_tile_id(int pid, int total) {
  const int per_xcd = (total + 7) >> 3, tall = (total & 7) ? (total & 7) : 8;
  const int xcd = pid & 7, local = pid >> 3;
  return xcd < tall ? xcd * per_xcd + local : tall * per_xcd + (xcd - tall) * (per_xcd - 1) + local;
}

namespace {

constexpr int MM_BK = 64;
constexpr int MM_LD = MM_BK;       // LDS row stride in elements: 128 bytes, eight 16-byte chunks
constexpr int MM_GROUP = 4;         // row tiles per block of tiles

// What becomes of a workgroup's sums: bias, activation, and the stores.  acc[i][j] of a lane: four neighbouring columns of one
// row, out[row0 + wr + j*16 + (lane & 15)][col0 + wc + i*16 + (lane >> 4)*4 + e].  lds: LDS_ELEMS elements that nobody needs any
// more once every wave is here.
template <int WTM, int WTN, int WVM, int WVN, int T, int LDS_ELEMS, int EPI, typename OT>
__device__ __forceinline__ void mfma_epilogue(f32x4_t (&acc)[WTN][WTM], bf16_t* lds, const float* __restrict__ bias,
                                              OT* __restrict__ out, long ldo, int n_rows, int n_out, int row0, int col0, int wr,
                                              int wc, const MfmaScatter& sc) {
  constexpr int BM = WVM * WTM * 16, BN = WVN * WTN * 16;
  const int tid = threadIdx.x, lane = tid & 63, lrow = lane & 15;
  // the activation's coefficients, read once (a store in between would make the compiler read them again)
  float xa_p = 0.f, xa_n = 0.f;
  if (EPI == MM_EPI_XIELU) {
    xa_p = sc.epi_coef[0];
    xa_n = sc.epi_coef[1];
  }
  // lane holds out[row0 + wr + j*16 + (lane & 15)][col0 + wc + i*16 + (lane >> 4)*4 + e], e = 0..3
  const bool vec = (n_out & 3) == 0 && (ldo & 3) == 0 && (((size_t)out | (size_t)bias) & 15) == 0;
  // bfloat16 outputs go through LDS (the staged operands are done with): a lane's four columns of
  // sixteen different rows would be sixteen 8-byte pieces per store; from LDS a thread stores 16
  // bytes and a row's threads a whole stretch of the row, and a key's or value's eight channels
  // go to their cache page the same way.
  constexpr int LDT = BN + 8;   // row stride of the tile in LDS
  // the whole tile at once if it fits, else the rows of one row of waves at a time
  constexpr int STAGE_ROWS = BM * LDT <= LDS_ELEMS ? BM : BM / WVM;
  constexpr bool CAN_STAGE = sizeof(OT) == 2 && STAGE_ROWS * LDT <= LDS_ELEMS;
  if (CAN_STAGE && EPI != MM_EPI_RESIDUAL && (n_out & 7) == 0 && (ldo & 7) == 0 && (((size_t)out) & 15) == 0 &&
      (EPI != MM_EPI_QKV || ((sc.q_width | sc.kv_width | sc.head_dim) & 7) == 0)) {
    bf16_t* tile = lds;
    for (int part = 0; part < BM / STAGE_ROWS; ++part) {
      __syncthreads();   // the staged operands, or the part before this one, are done with
      if (wr / STAGE_ROWS == part) {
#pragma unroll
        for (int i = 0; i < WTN; ++i) {
          const int tc = wc + i * 16 + (lane >> 4) * 4, oc = col0 + tc;
          float b4[4];
          mfma_bias4(bias, oc < n_out ? oc : 0, n_out, (((size_t)bias) & 15) == 0, b4);
#pragma unroll
          for (int j = 0; j < WTM; ++j) {
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              v[e] = acc[i][j][e] + b4[e];
              if (EPI == MM_EPI_GELU) v[e] = gelu_tanh_fast(v[e]);
              if (EPI == MM_EPI_RELU2) v[e] = relu_squared(v[e]);
              if (EPI == MM_EPI_XIELU) v[e] = mfma_xielu(v[e], xa_p, xa_n);
            }
            uint2 pk;
            pk.x = pack_bf16x2(v[0], v[1]);
            pk.y = pack_bf16x2(v[2], v[3]);
            *reinterpret_cast<uint2*>(&tile[(wr - part * STAGE_ROWS + j * 16 + lrow) * LDT + tc]) = pk;
          }
        }
      }
      __syncthreads();
      constexpr int CPR = BN / 8;   // 16-byte chunks per tile row
      for (int c = tid; c < STAGE_ROWS * CPR; c += T) {
        const int row = c / CPR, tc = (c % CPR) * 8;
        const int n = row0 + part * STAGE_ROWS + row, oc = col0 + tc;
        if (n >= n_rows || oc >= n_out) continue;
        const uint4 v8 = *reinterpret_cast<const uint4*>(&tile[row * LDT + tc]);
        *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(out) + (long)n * ldo + oc) = v8;
        if (EPI == MM_EPI_QKV && oc >= sc.q_width) {
          // the chunk's eight columns lie in one head
          const int slot = sc.slot_mapping[n];
          if (slot >= 0) {
            const int page = slot / sc.page_size, off = slot - page * sc.page_size;
            const int cq = oc - sc.q_width;  // column among keys then values
            const bool is_v = cq >= sc.kv_width;
            const int cc = is_v ? cq - sc.kv_width : cq;
            const int hh = cc / sc.head_dim, d = cc - hh * sc.head_dim;
            const long dst = (((long)page * sc.n_kv_head + hh) * sc.page_size + off) * sc.head_dim + d;
            *reinterpret_cast<uint4*>((is_v ? sc.vpool : sc.kpool) + dst) = v8;
          }
        }
      }
    }
    return;
  }
  // A key or value at (row n, column c of head hh, channel d) goes to
  // ((page * n_kv_head + hh) * page_size + offset) * head_dim + d of its pool, page and offset from
  // the row's slot: the row's part and the column's part of that are worked out once each.
  long cache_row[WTM];
  if (EPI == MM_EPI_QKV) {
#pragma unroll
    for (int j = 0; j < WTM; ++j) {
      const int n = row0 + wr + j * 16 + lrow;
      const int slot = n < n_rows ? sc.slot_mapping[n] : -1;
      const int page = slot / sc.page_size, off = slot - page * sc.page_size;
      cache_row[j] = slot < 0 ? -1 : ((long)page * sc.n_kv_head * sc.page_size + off) * sc.head_dim;
    }
  }
#pragma unroll
  for (int i = 0; i < WTN; ++i) {
    const int oc = col0 + wc + i * 16 + (lane >> 4) * 4;
    if (oc >= n_out) continue;
    float b4[4];
    mfma_bias4(bias, oc, n_out, vec, b4);
    bf16_t* cache_col = nullptr;
    if (EPI == MM_EPI_QKV && oc >= sc.q_width) {
      const int c = oc - sc.q_width;  // column among keys then values
      const bool is_v = c >= sc.kv_width;
      const int cc = is_v ? c - sc.kv_width : c;
      const int hh = cc / sc.head_dim, d = cc - hh * sc.head_dim;
      cache_col = (is_v ? sc.vpool : sc.kpool) + (long)hh * sc.page_size * sc.head_dim + d;
    }
#pragma unroll
    for (int j = 0; j < WTM; ++j) {
      const int n = row0 + wr + j * 16 + lrow;
      if (n >= n_rows) continue;
      bf16_t* cache_dst = nullptr;
      if (EPI == MM_EPI_QKV && cache_col && cache_row[j] >= 0) cache_dst = cache_col + cache_row[j];
      if (EPI == MM_EPI_XIELU)
        mfma_store4<EPI, OT>(acc[i][j], b4, out, ldo, n, oc, n_out, vec, cache_dst, xa_p, xa_n);
      else
        mfma_store4<EPI, OT>(acc[i][j], b4, out, ldo, n, oc, n_out, vec, cache_dst);
    }
  }
}

// The second chain of sums, if there is one, onto the first.
template <int CHAINS, int WTN, int WTM>
__device__ __forceinline__ void mfma_join_chains(f32x4_t (&chain)[CHAINS][WTN][WTM]) {
  if constexpr (CHAINS == 2) {
#pragma unroll
    for (int i = 0; i < WTN; ++i)
#pragma unroll
      for (int j = 0; j < WTM; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) chain[0][i][j][e] += chain[1][i][j][e];
  }
}

// WTM x WTN: 16-wide tiles per wave along the rows of the activations and along the rows of W;
// WVM x WVN: waves in a workgroup along the same.
// AHEAD: steps whose chunks are on their way from memory beyond the one that is being put into LDS
// (1: the schedule described above).  With few tiles of few rows over a large matrix that has to
// come from memory, a step's MFMAs are over long before the chunks of the step after next arrive
// (a 64 x 64 tile: 8 MFMAs a wave and step against a microsecond or more), and the product takes
// a memory round trip every two steps; more steps in flight, each in registers of its own, take that
// wait apart.
// KG: wave groups that share a tile (1 or 2).  With 2, the workgroup has twice the waves: group 0
// multiplies the first half (32) of every step along k and group 1 the second, each wave over the same
// part of the tile as its twin in the other group, and the twins' sums meet in LDS once, after the last
// step (float32 outputs only: the epilogue that stores them has no barrier, so group 1 is done then).
// For few tiles of 64 x 64 under a long inner size: a compute unit that has one such tile has four
// waves, too few to cover each other's waits for LDS and the barrier.
// CHAINS: 2 = an element's sum is two chains, over the first and over the second halves of the steps, added at the end: what two
// wave groups make (the same bits), with the accumulators of both in one wave.
// FOLD: > 0 = chains of that many steps, each added to the chains before it (with operands on their way in registers without a
// branch: where control flow joins the compiler waits for every load in flight).
template <int WTM, int WTN, int WVM, int WVN, int EPI, typename OT, int AHEAD = 1, int KG = 1, int DIRECT = 0, int CHAINS = 1,
          int FOLD = 0>
__global__ __launch_bounds__(64 * WVM * WVN * KG) void linear_mfma_kernel(
    const bf16_t* __restrict__ act, long lda, const bf16_t* __restrict__ w,
    const float* __restrict__ bias, OT* __restrict__ out, long ldo, int n_rows, int n_out, int k_dim,
    int k_parts, long part_stride, MfmaScatter sc) {
  static_assert(KG == 1 || (KG == 2 && sizeof(OT) == 4 && AHEAD == 1), "two wave groups: float32 outputs");
  static_assert(DIRECT == 0 || (DIRECT >= 2 && AHEAD == 1 && KG == 1), "slices straight into LDS: two stages or more");
  static_assert(CHAINS == 1 || (CHAINS == 2 && KG == 1), "two wave groups are two chains already");
  static_assert(FOLD == 0 || (CHAINS == 1 && KG == 1), "one way of keeping chains short");
  constexpr int T = 64 * WVM * WVN * KG;
  constexpr int STAGES = DIRECT > 0 ? DIRECT : 2;   // slices of a step that LDS holds
  constexpr int HALVES = (MM_BK / 32) / KG;   // halves of a step along k that a wave multiplies
  constexpr int BM = WVM * WTM * 16, BN = WVN * WTN * 16;
  constexpr int TPR = MM_BK / 8;  // threads per staged row (16 bytes each)
  constexpr int RPP = T / TPR;      // rows per staging pass
  constexpr int PA = BM / RPP, PW = BN / RPP;
  static_assert(DIRECT > 0 || (BM % RPP == 0 && BN % RPP == 0), "tile rows must be whole staging passes");
  static_assert(RPP % 8 == 0 && MM_BK == 64 && BM % 8 == 0 && BN % 8 == 0, "rows of eight chunks, swizzled in eights");
  extern __shared__ __align__(16) bf16_t lds[];
  bf16_t* const as_base = lds;                           // [STAGES][BM * MM_LD]
  bf16_t* const ws_base = lds + STAGES * BM * MM_LD;   // [STAGES][BN * MM_LD]

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = KG == 1 ? 0 : wave_all / (WVM * WVN);     // this wave's group: which half of a step it multiplies
  const int wave = KG == 1 ? wave_all : wave_all - kg * (WVM * WVN);
  const int row_tiles = (n_rows + BM - 1) / BM, col_tiles = (n_out + BN - 1) / BN;
  int row_tile, col_tile, part;
  {
    // with the inner size split into k_parts, part p of every tile comes before part p + 1 of any
    const int tiles = row_tiles * col_tiles;
    const int wid = mfma_xcd_tile_id(blockIdx.x, gridDim.x);
    part = wid / tiles;
    const int id = wid - part * tiles;
    const int per_group = MM_GROUP * col_tiles;
    const int group = id / per_group, in_group = id - group * per_group;
    const int first = group * MM_GROUP;
    const int rows_here = row_tiles - first < MM_GROUP ? row_tiles - first : MM_GROUP;
    row_tile = first + in_group % rows_here;
    col_tile = in_group / rows_here;
  }
  const int row0 = row_tile * BM, col0 = col_tile * BN;
  if (sc.row_expert) {
    // (the launcher has seen to it that a tile's rows lie in one group; padding comes last in a group)
    const int e = sc.row_expert[row0 / sc.group_rows];
    if (e < 0 || sc.row_valid[row0] < 0) return;   // the whole workgroup, before any barrier
    w += (long)e * sc.w_stride;
  }
  // this workgroup's stretch of the inner size (all of it unless the product is split), in whole steps
  const int k_per = (((k_dim + MM_BK - 1) / MM_BK + k_parts - 1) / k_parts) * MM_BK;
  const int k_begin = part * k_per;
  const int k_len = k_dim - k_begin < k_per ? k_dim - k_begin : k_per;
  out += part * part_stride;
  if (part != 0) bias = nullptr;  // of a product split along k, the first stretch's sums carry the bias (if any is given)
  const int wr = (wave / WVN) * (WTM * 16), wc = (wave % WVN) * (WTN * 16);
  const int lrow = lane & 15;

  const int srow = tid / TPR, sk = (tid % TPR) * 8;
  const int s_lds = srow * MM_LD + (((tid % TPR) ^ (srow & 7)) * 8);  // where this thread's chunk goes (RPP % 8 == 0)
  const bf16x8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  // What a thread stages per step: PA chunks of the activations' slice and PW of W's, each 16 bytes.
  constexpr int ITEMS = PA + PW;
  bf16x8_t gv[AHEAD][ITEMS];
  // rows past the end are read from the last row: their results are never stored
  const bf16_t* gp[ITEMS];
#pragma unroll
  for (int p = 0; p < PA; ++p) {
    const int r = row0 + srow + p * RPP;
    gp[p] = act + (long)(r < n_rows ? r : n_rows - 1) * lda + k_begin + sk;
  }
#pragma unroll
  for (int p = 0; p < PW; ++p) {
    const int r = col0 + srow + p * RPP;
    gp[PA + p] = w + (long)(r < n_out ? r : n_out - 1) * k_dim + k_begin + sk;
  }
  // A chunk that lies beyond the stretch's end (in its last, partial step) is read from the stretch's start instead
  // and counts as zero when it is stored: the select then waits for no load.
  // (set: which of the AHEAD sets of registers; a constant wherever these are called)
  auto load_item = [&](int p, int step, int set = 0) {
    const int k0 = step * MM_BK;
    gv[set][p] = *reinterpret_cast<const bf16x8_t*>(gp[p] + (k0 + sk + 8 <= k_len ? k0 : -sk));
  };
  auto store_item = [&](int p, int step, int buf, int set = 0) {
    bf16_t* dst = p < PA ? as_base + buf * (BM * MM_LD) + p * RPP * MM_LD
                         : ws_base + buf * (BN * MM_LD) + (p - PA) * RPP * MM_LD;
    *reinterpret_cast<bf16x8_t*>(dst + s_lds) = step * MM_BK + sk + 8 <= k_len ? gv[set][p] : zero8;
  };

  f32x4_t chain[CHAINS][WTN][WTM];  // [..][column tile of W][row tile of activations]
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int i = 0; i < WTN; ++i)
#pragma unroll
      for (int j = 0; j < WTM; ++j) chain[c][i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  auto& acc = chain[0];
  [[maybe_unused]] f32x4_t folded[WTN][WTM];
  if constexpr (FOLD > 0) {
#pragma unroll
    for (int i = 0; i < WTN; ++i)
#pragma unroll
      for (int j = 0; j < WTM; ++j) folded[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }

  const int k_steps = (k_len + MM_BK - 1) / MM_BK;
  const int c0 = ((lane >> 4) ^ (lrow & 7)) * 8;  // this lane's chunk of an operand row, first half of a step

  // One step along k.  Its 2 * WTM groups of MFMAs (one row tile of the activations against the
  // wave's WTN column tiles, for one half of the step) read their operands from LDS two groups
  // ahead of their use, so that a read's latency hides behind the MFMAs of the groups before it.
  // Spread between the groups, the thread puts the next step's chunks (loaded during the step
  // before this one) into the other LDS buffer and sends for those of the step after: LDS takes
  // writes at half the rate of reads, and all at once they would hold every wave up.
  // store_next / load_after: a compile-time yes or no; set: the registers that hold step s + 1 and
  // take step s + 1 + AHEAD
  auto k_step = [&](int s, auto store_next, auto load_after, auto set_c) {
    constexpr int set = decltype(set_c)::value;
    const int buf = DIRECT > 0 ? s % STAGES : s & 1;
    const bf16_t* as = as_base + buf * (BM * MM_LD) + (wr + lrow) * MM_LD;
    const bf16_t* ws = ws_base + buf * (BN * MM_LD) + (wc + lrow) * MM_LD;
    constexpr int GROUPS = HALVES * WTM;
    bf16x8_t wf[HALVES][WTN], af[3];
    // the second half's chunk is 4 further, which the swizzle turns into a flip of bit 5 of the offset
    // (with two wave groups a wave has one half only: its group's)
    const int h0 = kg * 32;
    auto read_a = [&](int g) {
      return *reinterpret_cast<const bf16x8_t*>(as + (g % WTM) * 16 * MM_LD + (c0 ^ (KG == 1 ? (g / WTM) * 32 : h0)));
    };
#pragma unroll
    for (int i = 0; i < WTN; ++i) wf[0][i] = *reinterpret_cast<const bf16x8_t*>(ws + i * 16 * MM_LD + (c0 ^ h0));
    if (WTM == 1 && HALVES == 2) {  // the second half's groups start at once
#pragma unroll
      for (int i = 0; i < WTN; ++i) wf[1][i] = *reinterpret_cast<const bf16x8_t*>(ws + i * 16 * MM_LD + (c0 ^ 32));
    }
    af[0] = read_a(0);
    af[1] = read_a(1);
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      if (g + 2 < GROUPS) af[(g + 2) % 3] = read_a(g + 2);
      if (WTM >= 2 && g % WTM == WTM - 2 && g / WTM + 1 < HALVES) {
#pragma unroll
        for (int i = 0; i < WTN; ++i)
          wf[g / WTM + 1][i] = *reinterpret_cast<const bf16x8_t*>(ws + i * 16 * MM_LD + (c0 ^ ((g / WTM + 1) * 32)));
      }
#pragma unroll
      for (int p = g * ITEMS / GROUPS; p < (g + 1) * ITEMS / GROUPS; ++p) {
        if (decltype(store_next)::value) store_item(p, s + 1, buf ^ 1, set);
        if (decltype(load_after)::value) load_item(p, s + 1 + AHEAD, set);
      }
      // the compiler's scheduler would move each read down to its use again
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < WTN; ++i) {
        f32x4_t& sum = chain[g / WTM % CHAINS][i][g % WTM];
        sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[g / WTM][i], af[g % 3], sum, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (FOLD > 0) {
      const bool ends = s % FOLD == FOLD - 1;
      if (DIRECT == 0 || ends) {
#pragma unroll
        for (int i = 0; i < WTN; ++i)
#pragma unroll
          for (int j = 0; j < WTM; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              folded[i][j][e] += ends ? acc[i][j][e] : 0.f;
              acc[i][j][e] = ends ? 0.f : acc[i][j][e];
            }
      }
    }
    if (decltype(store_next)::value) __syncthreads();  // the other buffer's readers finished before the last barrier
  };
  using yes = std::integral_constant<bool, true>;
  using no = std::integral_constant<bool, false>;
  using set0 = std::integral_constant<int, 0>;

  if constexpr (DIRECT > 0) {
    // The slices go from memory straight into LDS (global_load_lds_dwordx4: a wave's load puts its 64 lanes'
    // 16 bytes side by side, 1 KB, which is 8 rows of a slice).  The lane that fills position p of row r
    // fetches the chunk that belongs there, p ^ (r & 7).  No registers hold operands on their way and no
    // wave spends instructions on LDS stores; a compute unit also takes in more bytes a microsecond this
    // way than through registers.  STAGES slices of a step in LDS, STAGES - 1 steps on their way; a
    // step's loads are issued behind the barrier that says every wave has read the stage they overwrite.
    // The inner size is whole steps here (the launcher sees to it): nothing can be zeroed on its way.
    constexpr int WAVES = T / 64;
    constexpr int GROUPS_A = BM / 8, GROUPS = (BM + BN) / 8;
    // loads per wave and step: the same for every wave (each counts its own on their way)
    static_assert(GROUPS % WAVES == 0, "the groups of eight rows go round among the waves");
    constexpr int LPW = GROUPS / WAVES;
    constexpr int D = STAGES - 1;
    static_assert((D - 1) * LPW < 64, "the counter of loads in flight");
    typedef __attribute__((address_space(1))) const void* global_ptr_t;
    typedef __attribute__((address_space(3))) void* lds_ptr_t;
    const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
    const bf16_t* dp[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int g = wave_all + i * WAVES;   // 8 rows of the activations' slice, or of W's
      if (g < GROUPS_A) {
        const int r = row0 + g * 8 + lr;
        dp[i] = act + (long)(r < n_rows ? r : n_rows - 1) * lda + k_begin + lc;
      } else {
        const int r = col0 + (g - GROUPS_A) * 8 + lr;
        dp[i] = w + (long)(r < n_out ? r : n_out - 1) * k_dim + k_begin + lc;
      }
    }
    auto issue = [&](int step) {
      const int st = step % STAGES;
#pragma unroll
      for (int i = 0; i < LPW; ++i) {
        const int g = wave_all + i * WAVES;
        bf16_t* dst = g < GROUPS_A ? as_base + st * (BM * MM_LD) + g * (8 * MM_LD)
                                   : ws_base + st * (BN * MM_LD) + (g - GROUPS_A) * (8 * MM_LD);
        __builtin_amdgcn_global_load_lds((global_ptr_t)(dp[i] + step * MM_BK), (lds_ptr_t)dst, 16, 0, 0);
      }
    };
    // waits until at most `steps_behind` steps' loads of this wave are still on their way, then for every wave
    auto arrive = [&](int steps_behind) {
#define MM_WAIT_CASE(N) \
  case N: asm volatile("s_waitcnt vmcnt(%0)" ::"n"((N < D ? N : 0) * LPW) : "memory"); break;
      switch (steps_behind) {
        MM_WAIT_CASE(0) MM_WAIT_CASE(1) MM_WAIT_CASE(2) MM_WAIT_CASE(3) MM_WAIT_CASE(4) MM_WAIT_CASE(5) MM_WAIT_CASE(6)
        default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
      }
#undef MM_WAIT_CASE
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    static_assert(D <= 7, "arrive() knows up to six steps behind the one waited for");
#pragma unroll
    for (int j = 0; j < D; ++j)
      if (j < k_steps) issue(j);
    int s = 0;
    for (; s + D < k_steps; ++s) {
      arrive(D - 1);
      issue(s + D);
      k_step(s, no{}, no{}, set0{});
    }
    for (; s < k_steps; ++s) {   // the last steps: nothing more to send for
      arrive(k_steps - 1 - s);
      k_step(s, no{}, no{}, set0{});
    }
  } else {
    // The first two steps' chunks are sent for together, the first step's into registers of their own
    // (free before the loop needs them for MFMA operands): one trip to memory before the first MFMA
    // instead of two, which is a fifth of the whole kernel when the inner size is a few steps long.
    {
      bf16x8_t first[ITEMS];
  #pragma unroll
      for (int p = 0; p < ITEMS; ++p) first[p] = *reinterpret_cast<const bf16x8_t*>(gp[p] + (sk + 8 <= k_len ? 0 : -sk));
      if (AHEAD > 1 || k_steps > 1) {
  #pragma unroll
        for (int j = 1; j <= AHEAD; ++j)
  #pragma unroll
          for (int p = 0; p < ITEMS; ++p) load_item(p, j, j - 1);
      }
  #pragma unroll
      for (int p = 0; p < ITEMS; ++p) {
        bf16_t* dst = p < PA ? as_base + p * RPP * MM_LD : ws_base + (p - PA) * RPP * MM_LD;
        *reinterpret_cast<bf16x8_t*>(dst + s_lds) = sk + 8 <= k_len ? first[p] : zero8;
      }
    }
    __syncthreads();
    int s = 0;
    if constexpr (AHEAD == 1) {
      for (; s + 2 < k_steps; ++s) k_step(s, yes{}, yes{}, set0{});
      if (s + 1 < k_steps) k_step(s++, yes{}, no{}, set0{});
      k_step(s, no{}, no{}, set0{});
    } else {
      // Step s + 1 lies in set s mod AHEAD: the sets take turns, AHEAD steps a round, in whole rounds
      // and without a branch (where control flow joins the compiler waits for every load in flight):
      // a step beyond the last multiplies the zeros that stand in for chunks beyond the stretch's
      // end, and its loads read the stretch's start.
      auto round = [&](auto... set_c) { ((k_step(s, yes{}, yes{}, set_c), ++s), ...); };
      while (s < k_steps) {
        if constexpr (AHEAD == 2) round(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
        else if constexpr (AHEAD == 3) round(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{},
                                             std::integral_constant<int, 2>{});
        else round(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{},
                   std::integral_constant<int, 3>{});
      }
    }
  }

  if constexpr (KG == 2) {
    // the two groups' sums of the same part of the tile meet: group 1 hands its over through LDS (the
    // staged operands are done with) and is finished; group 0 adds them, first half of k first
    static_assert(WVM * WVN * WTN * WTM * 64 * 16 <= 2 * (BM + BN) * MM_LD * (int)sizeof(bf16_t), "the sums fit the LDS");
    f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
    __syncthreads();
    if (kg == 1) {
#pragma unroll
      for (int i = 0; i < WTN; ++i)
#pragma unroll
        for (int j = 0; j < WTM; ++j) red[((wave * WTN + i) * WTM + j) * 64 + lane] = acc[i][j];
    }
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int i = 0; i < WTN; ++i)
#pragma unroll
      for (int j = 0; j < WTM; ++j) {
        const f32x4_t t = red[((wave * WTN + i) * WTM + j) * 64 + lane];
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] += t[e];
      }
  }
  mfma_join_chains(chain);
  if constexpr (FOLD > 0) {
#pragma unroll
    for (int i = 0; i < WTN; ++i)
#pragma unroll
      for (int j = 0; j < WTM; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] = folded[i][j][e] + acc[i][j][e];
  }

  mfma_epilogue<WTM, WTN, WVM, WVN, T, STAGES * (BM + BN) * MM_LD, EPI, OT>(acc, lds, bias, out, ldo, n_rows, n_out, row0,
                                                                            col0, wr, wc, sc);
}

// The large tiles with the two halves of the workgroup out of step: 128 or 256 rows x 256 columns, eight waves of
// (WTM * 16) x 64, slices straight into LDS as in the DIRECT variants above.
//
// With all waves in step, each SIMD's two waves read their operands at the same time and then multiply at the same time, and
// the matrix units idle while the LDS works and the other way round (a step of 256 x 256 x 64 took 2.1 us for 0.9 us of
// MFMAs).  Here a step is cut into phases of 32 MFMAs a wave (64 of its rows), each a slot of reading and a slot of multiplying
// with a barrier between, and waves 4 to 7 (one on every SIMD) run one slot behind waves 0 to 3: in every slot one wave of a
// SIMD multiplies, at raised priority, while the other reads the operands of its next phase and sends for slices.
//
// (Four phases of 16 MFMAs took 163 us for 4,096 rows 6400 -> 1600, where two take 136; at full occupancy, 4,096 columns, both
// 160: the clock gives way.)
// With 256 rows a step has two phases (the upper and the lower 64 rows of a wave) and LDS two stages.  W and the upper rows
// have been read by both halves once the second half is through its first phase's reading: those of step s + 2 are sent for in
// the second phase of step s; the lower rows of step s + 1 in its first phase.  With 128 rows a step is one phase, LDS has
// three stages, and step s + 2 goes where step s - 1 was.  A wave waits for its own loads at the end of the slot behind which
// the first half begins to read what they bring; younger loads stay on their way.
//
// CHAINS as in the kernel above (two sets of accumulators are too many for 256 rows).
template <int WTM, int WTN, int EPI, typename OT, int CHAINS = 1>
__global__ __launch_bounds__(512, 2) void linear_mfma_halves_kernel(const bf16_t* __restrict__ act, long lda,
                                                                 const bf16_t* __restrict__ w, const float* __restrict__ bias,
                                                                 OT* __restrict__ out, long ldo, int n_rows, int n_out, int k_dim,
                                                                 MfmaScatter sc) {
  static_assert((WTM == 4 || WTM == 8) && (WTN == 3 || WTN == 4), "128 or 256 rows, 192 or 256 columns");
  static_assert(CHAINS == 1 || (CHAINS == 2 && WTM == 4), "accumulators");
  constexpr int WVM = 2, WVN = 4, T = 512;
  constexpr int BM = WVM * WTM * 16, BN = WVN * WTN * 16, STAGES = WTM == 8 ? 2 : 3;
  constexpr int LW = BN / 64;                 // a wave's loads of W's slice: 8 rows each; 2 of 64 (WTM = 8: upper, lower) rows a half
  extern __shared__ __align__(16) bf16_t lds[];
  bf16_t* const as_base = lds;
  bf16_t* const ws_base = lds + STAGES * BM * MM_LD;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row_tiles = (n_rows + BM - 1) / BM, col_tiles = (n_out + BN - 1) / BN;
  int row_tile, col_tile;
  {
    const int id = mfma_xcd_tile_id(blockIdx.x, gridDim.x);
    const int per_group = MM_GROUP * col_tiles;
    const int group = id / per_group, in_group = id - group * per_group;
    const int first = group * MM_GROUP;
    const int rows_here = row_tiles - first < MM_GROUP ? row_tiles - first : MM_GROUP;
    row_tile = first + in_group % rows_here;
    col_tile = in_group / rows_here;
  }
  const int row0 = row_tile * BM, col0 = col_tile * BN;
  if (sc.row_expert) {
    const int e = sc.row_expert[row0 / sc.group_rows];
    if (e < 0 || sc.row_valid[row0] < 0) return;   // the whole workgroup, before any barrier
    w += (long)e * sc.w_stride;
  }
  const int half = wave >> 2;
  const int wr = half * (WTM * 16), wc = (wave & 3) * (WTN * 16), lrow = lane & 15;
  const int k_steps = k_dim / MM_BK;

  typedef __attribute__((address_space(1))) const void* global_ptr_t;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
  // eight rows of the activations' slice: those numbered 16 h + 8 p + wave are rows wave * 8 .. of half h's part p (of 64 rows)
  constexpr int PARTS = WTM / 4;
  const bf16_t* ap[PARTS][2];
  const bf16_t* wp[LW];
#pragma unroll
  for (int p = 0; p < PARTS; ++p)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int r = row0 + (PARTS * 8 * h + 8 * p + wave) * 8 + lr;
      ap[p][h] = act + (long)(r < n_rows ? r : n_rows - 1) * lda + lc;
    }
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int r = col0 + (wave + 8 * i) * 8 + lr;
    wp[i] = w + (long)(r < n_out ? r : n_out - 1) * k_dim + lc;
  }
  auto issue_a = [&](int step, int st, int p) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(ap[p][h] + step * MM_BK),
                                       (lds_ptr_t)(as_base + st * (BM * MM_LD) + (PARTS * 8 * h + 8 * p + wave) * (8 * MM_LD)),
                                       16, 0, 0);
  };
  auto issue_w = [&](int step, int st) {
#pragma unroll
    for (int i = 0; i < LW; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(wp[i] + step * MM_BK),
                                       (lds_ptr_t)(ws_base + st * (BN * MM_LD) + (wave + 8 * i) * (8 * MM_LD)), 16, 0, 0);
  };

  f32x4_t chain[CHAINS][WTN][WTM];
#pragma unroll
  for (int c = 0; c < CHAINS; ++c)
#pragma unroll
    for (int i = 0; i < WTN; ++i)
#pragma unroll
      for (int j = 0; j < WTM; ++j) chain[c][i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int c0 = ((lane >> 4) ^ (lrow & 7)) * 8;
  bf16x8_t af[2][4], wf[2][WTN];   // [half of the step][row or column tile]
  auto read_a = [&](int st, int j0) {
    const bf16_t* p = as_base + st * (BM * MM_LD) + (wr + j0 * 16 + lrow) * MM_LD;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) af[h][j] = *reinterpret_cast<const bf16x8_t*>(p + j * 16 * MM_LD + (c0 ^ (h * 32)));
  };
  auto read_w = [&](int st) {
    const bf16_t* p = ws_base + st * (BN * MM_LD) + (wc + lrow) * MM_LD;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < WTN; ++i) wf[h][i] = *reinterpret_cast<const bf16x8_t*>(p + i * 16 * MM_LD + (c0 ^ (h * 32)));
  };
  auto multiply = [&](int j0) {
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < WTN; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          f32x4_t& sum = chain[h % CHAINS][i][j0 + j];
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][i], af[h][j], sum, 0, 0, 0);
        }
    __builtin_amdgcn_s_setprio(0);
  };
  // the end of a slot; what a wave has read has arrived
  auto slot_end = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // at most `YOUNGER` of this wave's loads are still on their way; none, towards the end, where fewer have been sent for
  constexpr int YOUNGER = WTM == 8 ? LW + 4 : LW + 2;
  auto arrived = [&](bool sent) {
    if (sent) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(YOUNGER) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };

#pragma unroll
  for (int s = 0; s < 2; ++s)
    if (s < k_steps) {
      issue_w(s, s);
      issue_a(s, s, 0);
      if (WTM == 8 && s == 0) issue_a(0, 0, PARTS - 1);
    }
  arrived(k_steps > 1);
  slot_end();
  if (half == 1) slot_end();
  for (int s = 0, st = 0; s < k_steps; ++s) {
    const bool next = s + 1 < k_steps, more = s + 2 < k_steps;
    read_w(st);
    read_a(st, 0);
    if constexpr (WTM == 8) {
      if (next) issue_a(s + 1, st ^ 1, 1);
      if (half == 1) arrived(next);
      slot_end();
      multiply(0);
      if (half == 0) arrived(next);
      slot_end();
      read_a(st, 4);
      if (more) {
        issue_w(s + 2, st);
        issue_a(s + 2, st, 0);
      }
      if (half == 1) arrived(more);
      slot_end();
      multiply(4);
      if (half == 0) arrived(more);
      slot_end();
    } else {
      if (more) {
        const int far = st == 0 ? 2 : st - 1;
        issue_w(s + 2, far);
        issue_a(s + 2, far, 0);
      }
      if (half == 1) arrived(more);
      slot_end();
      multiply(0);
      if (half == 0) arrived(more);
      slot_end();
    }
    st = st + 1 == STAGES ? 0 : st + 1;
  }
  if (half == 0) slot_end();   // as many barriers as the other half
  mfma_join_chains(chain);
  mfma_epilogue<WTM, WTN, WVM, WVN, T, STAGES * (BM + BN) * MM_LD, EPI, OT>(chain[0], lds, bias, out, ldo, n_rows, n_out, row0,
                                                                            col0, wr, wc, sc);
}

template <int WTM, int WTN, int EPI, typename OT, int CHAINS>
int launch_halves_one(const void* act, long lda, const void* w, const float* bias, void* out, long ldo, int n_rows, int n_out,
                      int k_dim, const MfmaScatter& sc, hipStream_t stream) {
  constexpr int BM = 32 * WTM, BN = 64 * WTN;
  constexpr size_t lds_bytes = (WTM == 8 ? 2ul : 3ul) * (BM + BN) * MM_LD * sizeof(bf16_t);
  auto kernel = linear_mfma_halves_kernel<WTM, WTN, EPI, OT, CHAINS>;
  static bool allowed = false;
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  const long tiles = (long)((n_rows + BM - 1) / BM) * ((n_out + BN - 1) / BN);
  if (tiles > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kernel, dim3((unsigned int)tiles), dim3(512), lds_bytes, stream, (const bf16_t*)act, lda, (const bf16_t*)w,
                     bias, (OT*)out, ldo, n_rows, n_out, k_dim, sc);
  return mgpt_last_error();
}

template <int WTM, int WTN, int CHAINS = 1>
int launch_halves(const void* act, long lda, const void* w, const float* bias, void* out, int out_dtype, long ldo, int n_rows,
                  int n_out, int k_dim, int epilogue, const MfmaScatter& sc, hipStream_t stream) {
#define MM_LAUNCH(E, OT) return launch_halves_one<WTM, WTN, E, OT, CHAINS>(act, lda, w, bias, out, ldo, n_rows, n_out, k_dim, sc, stream)
  if (epilogue == MM_EPI_NONE && out_dtype == MGPT_F32) MM_LAUNCH(MM_EPI_NONE, float);
  if (epilogue == MM_EPI_RESIDUAL && out_dtype == MGPT_F32) MM_LAUNCH(MM_EPI_RESIDUAL, float);
  if constexpr (CHAINS == 1) {
    if (epilogue == MM_EPI_NONE && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_NONE, bf16_t);
    if (epilogue == MM_EPI_GELU && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_GELU, bf16_t);
    if (epilogue == MM_EPI_RELU2 && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_RELU2, bf16_t);
    if (epilogue == MM_EPI_XIELU && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_XIELU, bf16_t);
    if (epilogue == MM_EPI_QKV && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_QKV, bf16_t);
  }
#undef MM_LAUNCH
  return MGPT_ERR_BAD_DTYPE;
}
// Few rows (NT slices of 16) under a large matrix: a workgroup owns all rows x NC slices of 16 columns, its four waves take the inner
// size 64 at a time in turn, and their sums meet in LDS in wave order.  Each wave brings its slices of W and of the rows straight
// into LDS, eight rows of 128 bytes a load, STAGES steps of its own on their way, and waits for nobody: no barrier before the last
// step.  What bounds it is the matrix's way from memory (16 rows 1600 -> 6400, 20.5 MB: 6.4 us, 3.2 TB/s with the launch; the 32 x 32
// tiles 7.8, whose barriers hold a step's four waves to the slowest load, on 200 of the 256 compute units); at 32 rows the rows' own, which
// every workgroup reads again.  More stages than these give nothing.  The rows go through LDS because with operands loaded into
// registers the compiler waits for all loads in flight where the loop closes.
// An element's sum is a chain a step of 64, those of a wave added in order, then the waves': error of 16 rows 6400 -> 1600 against 64
// bits, relative to the sums' norm, 1.1e-7 (decode kernel 2.4e-7, one chain 5.1e-7), 1600 -> 4800 0.77e-7 (1.2e-7, 2.4e-7).
template <int NT, int NC, int EPI, typename OT, int STAGES>
__global__ __launch_bounds__(256) void linear_mfma_rows_kernel(const bf16_t* __restrict__ act, long lda, const bf16_t* __restrict__ w,
                                                               const float* __restrict__ bias, OT* __restrict__ out, long ldo,
                                                               int n_rows, int n_out, int k_dim, int k_parts, long part_stride,
                                                               MfmaScatter sc) {
  constexpr int SLICE = 16 * MM_BK, SLICES = NC + NT;   // elements of 16 rows of a step; W's slices, then the rows'
  constexpr int LOADS = 2 * SLICES;                     // of a wave and step
  static_assert((STAGES - 1) * LOADS < 64, "the counter of loads in flight");
  static_assert(NT * NC <= 4, "a wave a tile of 16 x 16 behind the last step");
  typedef __attribute__((address_space(1))) const void* global_ptr_t;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  extern __shared__ __align__(16) bf16_t lds[];         // [4 waves][STAGES][SLICES][SLICE]
  __shared__ f32x4_t sums[4][NT * NC][64];
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col0 = blockIdx.x * (16 * NC), part = blockIdx.y;
  const int all_steps = k_dim / MM_BK, per = (all_steps + k_parts - 1) / k_parts;
  const int k_begin = part * per * MM_BK, steps = all_steps - part * per < per ? all_steps - part * per : per;
  const int own = steps > wave ? (steps - wave + 3) / 4 : 0;   // of this wave
  out += part * part_stride;
  if (part != 0) bias = nullptr;   // (the first stretch's sums carry it)
  // this lane's part of a load: row 8 i + lane / 8, chunk (lane % 8) ^ (row % 8)
  const int lr = lane >> 3, lc = ((lane & 7) ^ lr) * 8;
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    // (columns and rows past the end: the last one's sums, never stored)
    const int c = col0 + 8 * i + lr, r = 8 * (i - 2 * NC) + lr;
    src[i] = (i < 2 * NC ? w + (long)(c < n_out ? c : n_out - 1) * k_dim : act + (long)(r < n_rows ? r : n_rows - 1) * lda) +
             k_begin + wave * MM_BK + lc;
  }
  bf16_t* const staged = lds + wave * (STAGES * SLICES * SLICE);
  auto load = [&](int s, int st) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(src[i] + s * (4 * MM_BK)),
                                       (lds_ptr_t)(staged + st * (SLICES * SLICE) + i * (SLICE / 2)), 16, 0, 0);
  };
  auto arrive = [&](int behind) {   // waits until the loads of at most `behind` steps are on their way
#define MM_WAIT_CASE(N) \
  case N: asm volatile("s_waitcnt vmcnt(%0)" ::"n"((N < STAGES ? N : 0) * LOADS) : "memory"); break;
    switch (behind) {
      MM_WAIT_CASE(1) MM_WAIT_CASE(2) MM_WAIT_CASE(3)
      default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    }
#undef MM_WAIT_CASE
  };
  static_assert(STAGES <= 4, "arrive() knows up to three steps behind the one waited for");
  // what this wave's tile needs behind the last step: its bias, where its rows' keys and values go, and what the sums are added to
  const int n = (wave % NT) * 16 + li, oc = col0 + (wave / NT % NC) * 16 + lg * 4;
  const bool vec = (n_out & 3) == 0 && (ldo & 3) == 0 && (((size_t)out | (size_t)bias) & 15) == 0;
  float b4[4];
  mfma_bias4(bias, oc < n_out ? oc : 0, n_out, vec, b4);
  int slot = -1;
  if (EPI == MM_EPI_QKV) slot = sc.slot_mapping[n < n_rows ? n : 0];
  float4 added = {0.f, 0.f, 0.f, 0.f};
  if (EPI == MM_EPI_RESIDUAL && vec && wave < NT * NC && n < n_rows && oc < n_out)
    added = *reinterpret_cast<const float4*>(out + (long)n * ldo + oc);
#pragma unroll
  for (int s = 0; s < STAGES; ++s)
    if (s < own) load(s, s);
  f32x4_t acc[NC][NT];
#pragma unroll
  for (int i = 0; i < NC; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  const int at0 = li * MM_BK + ((lg ^ (li & 7)) * 8), at1 = at0 ^ 32;
  for (int s = 0, st = 0; s < own; ++s) {
    arrive(own - 1 - s < STAGES - 1 ? own - 1 - s : STAGES - 1);
    const bf16_t* slice = staged + st * (SLICES * SLICE);
    bf16x8_t op[SLICES][2];
#pragma unroll
    for (int j = 0; j < SLICES; ++j) {
      op[j][0] = *reinterpret_cast<const bf16x8_t*>(slice + j * SLICE + at0);
      op[j][1] = *reinterpret_cast<const bf16x8_t*>(slice + j * SLICE + at1);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // read before the stage is loaded again
    if (s + STAGES < own) load(s + STAGES, st);
    // a chain a step, added to those before it: chains are short whatever the inner size
    f32x4_t sum[NC][NT];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(op[i][h], op[NC + j][h],
                                                              h == 0 ? (f32x4_t){0.f, 0.f, 0.f, 0.f} : sum[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][j][e] += sum[i][j][e];
    st = st + 1 < STAGES ? st + 1 : 0;
  }
#pragma unroll
  for (int i = 0; i < NC; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) sums[wave][i * NT + j][lane] = acc[i][j];
  __syncthreads();
  if (wave >= NT * NC || n >= n_rows || oc >= n_out) return;
  f32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    v[e] = (sums[0][wave][lane][e] + sums[1][wave][lane][e]) + (sums[2][wave][lane][e] + sums[3][wave][lane][e]);
  if constexpr (EPI == MM_EPI_RESIDUAL) {
    if (vec) {
      *reinterpret_cast<float4*>(out + (long)n * ldo + oc) =
          make_float4(added.x + (v[0] + b4[0]), added.y + (v[1] + b4[1]), added.z + (v[2] + b4[2]), added.w + (v[3] + b4[3]));
      return;
    }
  }
  bf16_t* cache_dst = nullptr;
  if (EPI == MM_EPI_QKV && oc >= sc.q_width && slot >= 0) {
    const int page = slot / sc.page_size, off = slot - page * sc.page_size;
    const int c = oc - sc.q_width;   // column among keys then values
    const bool is_v = c >= sc.kv_width;
    const int cc = is_v ? c - sc.kv_width : c;
    const int hh = cc / sc.head_dim, d = cc - hh * sc.head_dim;
    cache_dst = (is_v ? sc.vpool : sc.kpool) + (((long)page * sc.n_kv_head + hh) * sc.page_size + off) * sc.head_dim + d;
  }
  mfma_store4<EPI, OT>(v, b4, out, ldo, n, oc, n_out, vec, cache_dst);
}

template <int WTM, int WTN, int WVM, int WVN, int EPI, typename OT, int AHEAD, int KG = 1, int DIRECT = 0, int CHAINS = 1, int FOLD = 0>
int launch_one(const void* act, long lda, const void* w, const float* bias, void* out, long ldo, int n_rows,
               int n_out, int k_dim, int k_parts, long part_stride, const MfmaScatter& sc, hipStream_t stream) {
  static_assert(AHEAD >= 1 && AHEAD <= 4, "sets of staging registers");
  constexpr int BM = WVM * WTM * 16, BN = WVN * WTN * 16;
  constexpr size_t lds_bytes = (DIRECT > 0 ? DIRECT : 2ul) * (BM + BN) * MM_LD * sizeof(bf16_t);
  static_assert(lds_bytes <= 160 * 1024, "a workgroup's LDS");
  auto kernel = linear_mfma_kernel<WTM, WTN, WVM, WVN, EPI, OT, AHEAD, KG, DIRECT, CHAINS, FOLD>;
  static bool allowed = false;  // more LDS than a kernel gets without asking
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  const long tiles = (long)((n_rows + BM - 1) / BM) * ((n_out + BN - 1) / BN) * k_parts;
  if (tiles > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;
  hipLaunchKernelGGL(kernel, dim3((unsigned int)tiles), dim3(64 * WVM * WVN * KG), lds_bytes, stream,
                     (const bf16_t*)act, lda, (const bf16_t*)w, bias, (OT*)out, ldo, n_rows, n_out, k_dim, k_parts,
                     part_stride, sc);
  return mgpt_last_error();
}

template <int WTM, int WTN, int WVM, int WVN, int AHEAD = 1, int DIRECT = 0, int CHAINS = 1>
int launch_shape(const void* act, long lda, const void* w, const float* bias, void* out, int out_dtype, long ldo,
                 int n_rows, int n_out, int k_dim, int epilogue, int k_parts, long part_stride,
                 const MfmaScatter& sc, hipStream_t stream) {
#define MM_LAUNCH(E, OT)                                                                                            \
  return launch_one<WTM, WTN, WVM, WVN, E, OT, AHEAD, 1, DIRECT, CHAINS>(act, lda, w, bias, out, ldo, n_rows, n_out, k_dim, \
                                                                         k_parts, part_stride, sc, stream)
  if (epilogue == MM_EPI_NONE && out_dtype == MGPT_F32) MM_LAUNCH(MM_EPI_NONE, float);
  if (epilogue == MM_EPI_RESIDUAL && out_dtype == MGPT_F32) MM_LAUNCH(MM_EPI_RESIDUAL, float);
  if constexpr (CHAINS == 1) {
    if (epilogue == MM_EPI_NONE && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_NONE, bf16_t);
    if (epilogue == MM_EPI_GELU && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_GELU, bf16_t);
    if (epilogue == MM_EPI_RELU2 && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_RELU2, bf16_t);
    if (epilogue == MM_EPI_XIELU && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_XIELU, bf16_t);
    if (epilogue == MM_EPI_QKV && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_QKV, bf16_t);
  }
#undef MM_LAUNCH
  return MGPT_ERR_BAD_DTYPE;
}

template <int NT, int NC, int EPI, typename OT, int STAGES>
int launch_rows_one(const void* act, long lda, const void* w, const float* bias, void* out, long ldo, int n_rows, int n_out, int k_dim,
                    int k_parts, long part_stride, const MfmaScatter& sc, hipStream_t stream) {
  constexpr size_t lds_bytes = 4ul * STAGES * (NC + NT) * 16 * MM_BK * sizeof(bf16_t), sums_bytes = 4ul * NT * NC * 64 * 16;
  static_assert(lds_bytes + sums_bytes <= 160 * 1024, "a workgroup's LDS");
  auto kernel = linear_mfma_rows_kernel<NT, NC, EPI, OT, STAGES>;
  static bool allowed = false;  // more LDS than a kernel gets without asking
  if (!allowed) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds_bytes);
    if (e != hipSuccess) return (int)e;
    allowed = true;
  }
  hipLaunchKernelGGL(kernel, dim3((n_out + 16 * NC - 1) / (16 * NC), k_parts), dim3(256), lds_bytes, stream, (const bf16_t*)act, lda,
                     (const bf16_t*)w, bias, (OT*)out, ldo, n_rows, n_out, k_dim, k_parts, part_stride, sc);
  return mgpt_last_error();
}

template <int NT, int NC, int STAGES>
int launch_rows(const void* act, long lda, const void* w, const float* bias, void* out, int out_dtype, long ldo, int n_rows,
                int n_out, int k_dim, int epilogue, int k_parts, long part_stride, const MfmaScatter& sc, hipStream_t stream) {
#define MM_LAUNCH(E, OT)                                                                                                  \
  return launch_rows_one<NT, NC, E, OT, STAGES>(act, lda, w, bias, out, ldo, n_rows, n_out, k_dim, k_parts, part_stride, sc, stream)
  if (epilogue == MM_EPI_NONE && out_dtype == MGPT_F32) MM_LAUNCH(MM_EPI_NONE, float);
  if (epilogue == MM_EPI_RESIDUAL && out_dtype == MGPT_F32) MM_LAUNCH(MM_EPI_RESIDUAL, float);
  if (epilogue == MM_EPI_NONE && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_NONE, bf16_t);
  if (epilogue == MM_EPI_GELU && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_GELU, bf16_t);
  if (epilogue == MM_EPI_RELU2 && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_RELU2, bf16_t);
  if (epilogue == MM_EPI_QKV && out_dtype == MGPT_BF16) MM_LAUNCH(MM_EPI_QKV, bf16_t);
#undef MM_LAUNCH
  return MGPT_ERR_BAD_DTYPE;
}

// The 64 x 64 tile with two wave groups (float32 outputs: plain, or added into the residual stream).
int launch_two_groups(const void* act, long lda, const void* w, const float* bias, void* out, int out_dtype, long ldo,
                      int n_rows, int n_out, int k_dim, int epilogue, int k_parts, long part_stride,
                      const MfmaScatter& sc, hipStream_t stream) {
  if (out_dtype != MGPT_F32) return MGPT_ERR_BAD_DTYPE;
  if (epilogue == MM_EPI_NONE)
    return launch_one<2, 2, 2, 2, MM_EPI_NONE, float, 1, 2>(act, lda, w, bias, out, ldo, n_rows, n_out, k_dim, k_parts,
                                                          part_stride, sc, stream);
  if (epilogue == MM_EPI_RESIDUAL)
    return launch_one<2, 2, 2, 2, MM_EPI_RESIDUAL, float, 1, 2>(act, lda, w, bias, out, ldo, n_rows, n_out, k_dim,
                                                              k_parts, part_stride, sc, stream);
  return MGPT_ERR_BAD_DTYPE;
}

// Tile shapes, largest first: rows x columns of a workgroup's tile.
constexpr int MM_SHAPES = 5;
constexpr int MM_TILE_ROWS[MM_SHAPES] = {256, 128, 128, 64, 32};
constexpr int MM_TILE_COLS[MM_SHAPES] = {256, 256, 64, 64, 32};
constexpr int MM_MAX_PARTS = 8;
constexpr int MM_FOLD = 2;   // steps of a chain where chains are kept short
constexpr int MM_AHEAD = 4;  // steps on their way from memory in the variant for few tiles over a large matrix
// Shape ids from MM_DIRECT_FIRST on: the variants whose slices go from memory straight into LDS, by tile
// (rows x columns), waves and stages: 32 x 32 (four waves of 16 x 16) and 64 x 64 (four of 32 x 32) with four
// stages, 128 x 64 (eight of 32 x 32) with three, 128 x 192 (eight of 64 x 48) with two, 32 x 32 with six; then the
// variants with the halves out of step.
constexpr int MM_DIRECT_FIRST = MM_SHAPES + 3;
constexpr int MM_DIRECT_VARIANTS = 9;
constexpr int MM_DIRECT_ROWS[MM_DIRECT_VARIANTS] = {32, 64, 128, 128, 32, 256, 128, 256, 128};
constexpr int MM_DIRECT_COLS[MM_DIRECT_VARIANTS] = {32, 64, 64, 192, 32, 256, 256, 192, 192};
constexpr int MM_DIRECT_HALVES = 5;     // the first of the four variants with the halves out of step: 256 x 256, 128 x 256,
                                        // 256 x 192, 128 x 192
// then the same variants with two chains of sums (float32 outputs; those of 128 x 64 and of 128 rows out of step have them)
constexpr int MM_CHAINS_FIRST = MM_DIRECT_FIRST + MM_DIRECT_VARIANTS;
constexpr bool MM_HAS_CHAINS[MM_DIRECT_VARIANTS] = {false, false, true, false, false, false, true, false, true};
constexpr int MM_ROWS = MM_CHAINS_FIRST + MM_DIRECT_VARIANTS;   // the kernel for few rows, 16 columns a workgroup, then 32
constexpr int MM_SHAPE_IDS = MM_ROWS + 2;
constexpr int MM_ROWS_MAX = 32;

long tiles_of(int shape, int n_rows, int n_out) {
  return (long)((n_rows + MM_TILE_ROWS[shape] - 1) / MM_TILE_ROWS[shape]) *
         ((n_out + MM_TILE_COLS[shape] - 1) / MM_TILE_COLS[shape]);
}

// The largest tile that still fills the machine's 256 compute units.  The two largest shapes run
// one workgroup per unit, so what counts for them is also how full their last round is.
int choose_shape(int n_rows, int n_out) {
  // Few rows under a wide output (the head of a decode step, 50k columns): the product is a pass over
  // the matrix, and a tile taller than the rows only makes each workgroup's share of that pass
  // larger.  Measured at 50304 x 512 (and alike at inner sizes 768 and 1600): 32 rows take 11.4 us
  // with 32 x 32 tiles and 17.9 with 256 x 256, 64 rows 13.9 with 64 x 64 and 19.3, 128 rows 17.5
  // with 128 x 256 and 22.4; from 256 rows on the largest tile is the fastest again.
  if (n_rows <= 32 && tiles_of(4, n_rows, n_out) >= 256) return 4;
  if (n_rows <= 64 && tiles_of(3, n_rows, n_out) >= 256) return 3;
  if (n_rows <= 128 && tiles_of(1, n_rows, n_out) >= 160) return 1;
  for (int shape = 0; shape < 2; ++shape) {
    const long t = tiles_of(shape, n_rows, n_out);
    const long rounds = (t + 255) / 256;
    if (t >= (shape == 0 ? 160 : 140) && 10 * t >= 7 * rounds * 256) return shape;
  }
  // 128 x 64 tiles only where their last round of 256 is well filled: 384 of them (2,048 rows under 1,536
  // columns) leave half the compute units with two tiles and half with one, and 768 tiles of 64 x 64
  // take 8.4 us where they take 9.2; 512 (under 2,048 columns) take 10.3 against 10.6
  {
    const long t = tiles_of(2, n_rows, n_out);
    if (t >= 300 && 100 * t >= 85 * ((t + 255) / 256) * 256) return 2;
  }
  if (tiles_of(3, n_rows, n_out) >= 192) return 3;
  return 4;
}

// Whether a product of few rows goes to the kernel that has nothing but them and 16 or 32 columns a workgroup, rather than to the decode
// kernel (from the matrix packed for it) or the 32 x 32 tiles.  us in a graph, matrices from memory, those two / here, where the
// better one is: 1600 -> 4800 6.5 / 5.3 at 1 row, 7.6 / 5.7 at 8, 9.0 / 6.0 at 16, 7.7 / 7.1 at 32; 1600 -> 6400 9.2 / 6.4 at 16, 7.9 / 7.4
// at 32; 1600 -> 1600 4.0 / 3.8, 4.8 / 4.1, 5.1 / 4.4, 5.8 / 5.2
// (into the residual rows of a decode step at 32 rows 6.1 / 5.9); 2048 -> 2048 4.7 / 4.5 at 4, 7.6 / 7.1 at 32; 2688 -> 1024 4.8 / 4.1, 7.1 /
// 6.3; 5440 -> 2048 9.9 / 7.8, 14.4 / 10.2; 768 -> 2304 3.2 / 3.0 at 8, 4.6 / 3.4 at 32.
bool rows_take(int n_rows, int n_out, int k_dim) {
  const long elements = (long)n_out * k_dim;
  if (n_rows < 1 || n_rows > MM_ROWS_MAX || k_dim % MM_BK != 0 || n_out < 768 || n_out > 8192) return false;
  // Small matrices are a launch and one trip to memory either way (1024 -> 1024 2.6 / 2.8, 768 -> 768 2.6 / 2.7, 512 -> 3072 2.6 / 2.8 at 1
  // row), and rows of 2,048 bytes and multiples come from few of the memory's channels at a time, which a packed matrix does not
  // (2048 -> 1024 3.6 / 3.7, 4.3 / 4.9; 1024 -> 2048 3.8 / 3.9 at 32).  The decode kernel's time grows with the rows, this one's hardly: with
  // few of them the lines are further up.  896 -> 1792 3.05 / 3.24 at 4 rows, into float32 rows, 3.28 / 3.26 at 12; 768 -> 2304 3.12 / 3.17 at
  // 3, 3.21 / 3.18 at 6, 896 -> 2304 3.26 / 3.33 at 6, 3.35 / 3.31 at 8; 896 -> 3072 3.10 / 3.22 at 1, 3.32 / 3.28 at 4; 1600 -> 1024 3.54 /
  // 3.66 at 4, 3.85 / 3.68 at 12; 1792 -> 1280 3.50 / 3.60 at 1; 2048 -> 4096 5.37 / 5.58 at 1, 5.76 / 5.69 at 4; 2048 -> 7168 7.8 / 8.0 and
  // 2048 -> 8192 8.7 / 8.9 at 1.
  if (elements < (k_dim % 1024 == 0 ? 4000000 : 1500000)) return false;
  if (k_dim < 768 && n_rows < 8) return false;
  if (k_dim < 1024 && n_rows < (n_out <= 2048 ? 12 : n_out <= 2560 ? (k_dim < 832 ? 4 : 8) : n_out <= 4096 ? 3 : 1)) return false;
  if (elements < 2400000 && n_out < 1536 && n_rows < 6) return false;
  if (k_dim == 2048 && (n_out <= 4096 || n_out == 7168) && n_rows < 3) return false;
  if (n_out > 7168 && n_rows < 4) return false;
  // A long inner size under few columns before it is cut (rows_parts): 64 workgroups at most, each with a long chain of steps (6144 -> 768
  // 6.5 / 7.0 at 1 row, 8192 -> 1024 8.1 / 8.6 at 4).
  if (n_out <= 1024 && k_dim >= 6144 && (long)n_rows * k_dim < (k_dim % 8192 == 0 ? 65536 : 30000)) return false;
  // Large matrices with rows of 4,096 bytes and multiples: 6144 -> 7168 (44 million) 18.5 / 20.2 at 1 row, 20.4 / 20.2 at 6; 8192 -> 6400 (52)
  // 24.9 / 26.1 at 4, 26.7 / 26.0 at 8; 8192 -> 8128 (67) 30.6 / 32.5 at 8, equal at 12; 16384 -> 4096 32.9 / 35.4 at 16, 39.2 / 35.8 at 17,
  // 16384 -> 1536 15.6 / 15.9 at 8.  Not under 257 to 320 tiles of columns, which the decode kernel takes in two rounds (8192 -> 5120 21.9 / 21.5).
  if (k_dim % 2048 == 0 && (n_out <= 4096 || n_out > 5120) && n_rows * 2500000L <= elements - 36000000) return false;
  if (k_dim >= 16384 && n_out > 1024 && n_rows <= (n_out > 3072 ? 16 : 12)) return false;
  // Two tiles of rows read again by every workgroup, where the 32 x 32 tiles fill the chip: 8192 -> 4800 21.9 / 22.2 at 17, 22.6 / 24.2 at 32,
  // 7680 -> 4800 22.0 / 22.1 at 24, 22.7 / 23.9 at 32; 10240 -> 4096 23.8 / 24.6 at 32.
  if (n_rows > 16 && n_out > 4096 && n_out <= 5120 && (k_dim % 2048 == 0 ? k_dim >= 8192 : (long)n_rows * k_dim >= 215000)) return false;
  if (n_rows > 28 && n_out > 2560 && n_out <= 4096 && k_dim >= 10240) return false;
  return true;
}

// Into how many stretches such a product's inner size is cut (choose_split's reasons): every 16 columns read all rows again, and a
// wave's steps are a chain.  us with the sums added up and into float32 rows, whole / cut: 6400 -> 1600 8.2 / 8.0 at 1 row, 9.3 / 8.6 at 8,
// 14.2 / 10.6 at 32 (in four, 32 columns a workgroup); 5440 -> 2048 8.6 / 9.0 at 8, 9.7 / 9.2 at 16, 12.3 / 10.5 at 32; 2688 -> 1024 5.9 / 6.3
// at 16, 7.2 / 6.7 at 32; 8192 -> 2048 12.8 / 13.4 at 16, 15.9 / 12.5 at 32; 5120 -> 1024 7.9 / 7.2 at 8 (in four).  With more than 128 tiles of
// columns the stretches are more workgroups than the chip takes at once: 2048 -> 2304 6.2 / 8.4 at 32, 4096 -> 2560 9.6 / 11.3; and rows of
// 16,384 bytes in stretches come from fewer of the memory's channels still: 8192 -> 1536 9.4 / 10.7 at 4, 11.0 / 10.9 at 12.
int rows_parts(int n_rows, int n_out, int k_dim) {
  const int tiles = (n_out + 15) / 16;
  if (tiles > 160 || (tiles > 128 && k_dim < 5120) || k_dim / MM_BK < 32) return 1;
  if (k_dim % 8192 == 0 && tiles > 64 && n_rows <= 12) return 1;
  const bool many = (long)n_rows * k_dim >= (tiles <= 64 && k_dim >= 5120 ? 30000 : 50000), lengthy = k_dim >= 5120 && tiles <= 100;
  if (tiles <= 64 || n_rows > 16) return many ? 4 : (tiles > 64 && lengthy ? 2 : 1);
  return (many || lengthy) && (k_dim % 1024 != 0 || tiles < 128) ? 2 : 1;
}

// 32 columns a workgroup: where 16 are more workgroups than compute units, and half as many read the rows half as often (in four
// stretches, 16 / 32 columns: 6400 -> 1088 11.2 / 10.0 at 32 rows, 4096 -> 1152 8.0 / 7.7 at 17; 6400 -> 768 8.4 with 16).
bool rows_wide(int n_rows, int n_out, int parts) {
  const int tiles = (n_out + 15) / 16;
  return parts > 1 ? parts == 4 && n_rows > 16 && tiles > 64 : tiles > 256;
}

// Whether the inner size is split into stretches, and then with which tile shape and into how many
// (parts == 1: not at all, and the shape is the one chosen by the tiles alone).  A long inner size
// with few tiles leaves most compute units idle for a long time: then several workgroups share a
// tile, each writes the sum over its stretch to the caller's buffer, and a second kernel adds the
// sums in the order of k (so the result does not depend on which workgroup ran when) and applies
// the epilogue.  That costs a pass over parts x the output, so it is done only for an inner size of
// at least 32 steps whose unsplit product would not fill the compute units; every stretch is at
// least 8 steps long; 64 x 64 tiles if they and the stretches together fill the units, else 32 x 32.
// The QKV epilogue is never split.
void choose_split(int n_rows, int n_out, int k_dim, int epilogue, int* shape, int* parts) {
  *shape = choose_shape(n_rows, n_out);
  *parts = 1;
  const int steps = (k_dim + MM_BK - 1) / MM_BK;
  // "would not fill the units": counted in 64 x 64 tiles for a very long inner size, where the many
  // 32 x 32 tiles that would fill them take far longer than 64 x 64 tiles with stretches
  if (epilogue == MM_EPI_QKV || (n_out & 3) != 0 || steps < 32 || tiles_of(steps >= 64 ? 3 : 4, n_rows, n_out) >= 256)
    return;
  for (int sh = 3; sh <= 4; ++sh) {
    const long t = tiles_of(sh, n_rows, n_out);
    int p = 1;
    while (p < MM_MAX_PARTS && t * p * 2 <= 640 && steps / (p * 2) >= 8) p *= 2;
    if (p > 1 && (t * p >= 256 || sh == 4)) {
      *shape = sh;
      *parts = p;
      return;
    }
  }
}

// drops stretches that would be empty (the stretch length is rounded up to whole steps)
int used_parts(int k_dim, int parts) {
  const int steps = (k_dim + MM_BK - 1) / MM_BK;
  const int per = (steps + parts - 1) / parts;
  return (steps + per - 1) / per;
}

// out[n, o] = sum over the stretches' sums, in their order, + bias, with the epilogue
template <int EPI, typename OT>
__global__ __launch_bounds__(256) void linear_mfma_join_kernel(const float* __restrict__ partials, int k_parts,
                                                               const float* __restrict__ bias, OT* __restrict__ out,
                                                               long ldo, int n_rows, int n_out,
                                                               const float* __restrict__ epi_coef) {
  const int quads = n_out >> 2;
  const long idx = (long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long)n_rows * quads) return;
  const int row = (int)(idx / quads), oc = (int)(idx - (long)row * quads) * 4;
  const float* p = partials + (long)row * n_out + oc;
  const long part_stride = (long)n_rows * n_out;
  float4 v = *reinterpret_cast<const float4*>(p);
  for (int s = 1; s < k_parts; ++s) {
    const float4 t = *reinterpret_cast<const float4*>(p + s * part_stride);
    v.x += t.x; v.y += t.y; v.z += t.z; v.w += t.w;
  }
  if (bias) {
    const bool al = (((size_t)bias) & 15) == 0;
    if (al) {
      const float4 b4 = *reinterpret_cast<const float4*>(bias + oc);
      v.x += b4.x; v.y += b4.y; v.z += b4.z; v.w += b4.w;
    } else {
      v.x += bias[oc]; v.y += bias[oc + 1]; v.z += bias[oc + 2]; v.w += bias[oc + 3];
    }
  }
  if (EPI == MM_EPI_GELU) {
    v.x = gelu_tanh_fast(v.x); v.y = gelu_tanh_fast(v.y); v.z = gelu_tanh_fast(v.z); v.w = gelu_tanh_fast(v.w);
  }
  if (EPI == MM_EPI_RELU2) {
    v.x = relu_squared(v.x); v.y = relu_squared(v.y); v.z = relu_squared(v.z); v.w = relu_squared(v.w);
  }
  if (EPI == MM_EPI_XIELU) {
    const float a_p = epi_coef[0], a_n = epi_coef[1];
    v.x = mfma_xielu(v.x, a_p, a_n); v.y = mfma_xielu(v.y, a_p, a_n); v.z = mfma_xielu(v.z, a_p, a_n); v.w = mfma_xielu(v.w, a_p, a_n);
  }
  OT* orow = out + (long)row * ldo + oc;
  const float r[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (EPI == MM_EPI_RESIDUAL) orow[e] = from_float<OT>(to_float<OT>(orow[e]) + r[e]);
    else orow[e] = from_float<OT>(r[e]);
  }
}

int launch_join(const float* partials, int k_parts, const float* bias, void* out, int out_dtype, long ldo,
                int n_rows, int n_out, int epilogue, hipStream_t stream, const float* epi_coef = nullptr) {
  const long work = (long)n_rows * (n_out >> 2);
  dim3 grid((unsigned int)((work + 255) / 256));
#define MM_JOIN(E, OT)                                                                                  \
  hipLaunchKernelGGL((linear_mfma_join_kernel<E, OT>), grid, dim3(256), 0, stream, partials, k_parts, \
                     bias, (OT*)out, ldo, n_rows, n_out, epi_coef)
  if (epilogue == MM_EPI_NONE && out_dtype == MGPT_BF16) MM_JOIN(MM_EPI_NONE, bf16_t);
  else if (epilogue == MM_EPI_NONE && out_dtype == MGPT_F32) MM_JOIN(MM_EPI_NONE, float);
  else if (epilogue == MM_EPI_GELU && out_dtype == MGPT_BF16) MM_JOIN(MM_EPI_GELU, bf16_t);
  else if (epilogue == MM_EPI_RELU2 && out_dtype == MGPT_BF16) MM_JOIN(MM_EPI_RELU2, bf16_t);
  else if (epilogue == MM_EPI_XIELU && out_dtype == MGPT_BF16) MM_JOIN(MM_EPI_XIELU, bf16_t);
  else if (epilogue == MM_EPI_RESIDUAL && out_dtype == MGPT_F32) MM_JOIN(MM_EPI_RESIDUAL, float);
  else return MGPT_ERR_BAD_DTYPE;
#undef MM_JOIN
  return mgpt_last_error();
}

bool shapes_ok(const void* act, long lda, const void* w, const void* out, long ldo, int n_rows, int n_out, int k_dim) {
  return act && w && out && n_rows >= 0 && n_out >= 0 && k_dim > 0 && (k_dim % 16) == 0 && lda >= k_dim &&
         (lda % 8) == 0 && ldo >= n_out;
}

// whole steps along k, and operands aligned for 16-byte loads: what the variants that load straight into LDS need
bool direct_ok(const void* act, const void* w, int k_dim) {
  return (k_dim % MM_BK) == 0 && ((((size_t)act) | ((size_t)w)) & 15) == 0;
}

long direct_tiles(int variant, int n_rows, int n_out) {
  return (long)((n_rows + MM_DIRECT_ROWS[variant] - 1) / MM_DIRECT_ROWS[variant]) *
         ((n_out + MM_DIRECT_COLS[variant] - 1) / MM_DIRECT_COLS[variant]);
}

// 64 x 64 tiles under a long inner size (16 steps and more a workgroup), float32 out: two wave groups
// a tile.  [2048 x 2048 -> 512] 12.9 us against 14.4, [1024 x 2048 -> 512] 12.2 / 13.4, [2048 x 3072 ->
// 768] 24.2 / 25.5, [8192 x 2048 -> 512] 33.9 / 35.3; at 8 steps ([2048 x 512 -> 512]) nothing.
// (alone in a graph the variant is ahead at 256 tiles too, 12.9 us against 14.4; inside the 2,048-token
// prefill step it is not, 0.599-0.607 ms against 0.596-0.602 in turns on one box: more than a tile a unit)
bool two_groups_pay(int steps, long tiles) { return steps >= 16 && tiles > 256; }

// The shape id for a product of a prompt portion (128 rows and more) whose slices can go straight into
// LDS and that gains by it, or -1: the rules further down decide.  Which products gain was measured inside
// the prefill step, one product of the layer changed at a time (alone in a graph of its own, with its
// operands in the L2 from the launch before, every such variant is 10-20 % ahead of the register path, and
// most of that is not there in the step):
// - a long inner size (32 steps and more: the second feed-forward product).  Through registers two steps are
//   on their way, or the inner size is split over workgroups and a second kernel adds the parts; here three
//   or four stages hold as many steps, with no registers spent on them.  Prefill steps of 256 to 2,048
//   tokens: width 512 -3 %, width 768 -1 to -10 %, width 1600 at 2,048 tokens -7 %.
// - a wide output under many rows: tiles of 128 x 192 where a round of them costs less than a round of
//   256 x 256 (qkv and first feed-forward product at 8,192 tokens, widths 512 to 1600: -2 to -5 % of the step).
// - many rows (512 and more) under an inner size of 12 steps and more: the variant that takes least by a model of rounds of
//   workgroups (choose_large below).
int choose_medium(int n_rows, int n_out, int k_dim) {
  if (k_dim / MM_BK >= 32) {
    const long t128 = direct_tiles(2, n_rows, n_out), t64 = direct_tiles(1, n_rows, n_out);
    if (t128 > 520) return -1;
    if (t128 >= 190) return MM_DIRECT_FIRST + 2;
    return MM_DIRECT_FIRST + (t64 >= 190 ? 1 : 0);
  }
  // (measured from 1,536 columns up; under 512 columns at 8,192 rows those tiles lose 2 % of the step)
  const long wide = direct_tiles(3, n_rows, n_out), largest = tiles_of(0, n_rows, n_out);
  if (n_out < 1536 || wide < 190) return -1;
  // a tile's cost: its outputs, times a factor that falls with its size, times the rounds of 256 tiles
  const double cost_wide = (double)((wide + 255) / 256) * 128 * 192 * 0.78;
  const double cost_largest = (double)((largest + 255) / 256) * 256 * 256 * 0.72;
  if (largest >= 160 && cost_largest <= cost_wide) return -1;
  return MM_DIRECT_FIRST + 3;
}

// Of the large variants the one that takes least: rounds of as many workgroups as the chip holds, each steps x us a step + us for
// its fill and epilogue, and behind them 0.68 us a million outputs (added to float32 rows, which are read and written: 1.28).  The numbers
// are fits to 417 products of 512 to 12,288 rows, inner sizes 768 to 6,400 and 640 to 10,880 columns (each variant alone in a graph,
// three sets of operands in turn): half of the predictions are within 2 %, 95 of 100 within 7.  The choice takes up to 5 % longer
// than the best variant, up to 4 % longer than the rules above without it, and 7 % less than those in the mean.  Two workgroups of
// the variants with less LDS share a compute unit, and each is faster where it has one to itself.
// Those rules / now, in turn, us: 4,096 rows 1600 -> 4800 69 / 68, 1600 -> 6400 87 / 81, 1600 -> 1600 added to float32 rows 40 / 35,
// 6400 -> 1600 107 / 100; 3,300 rows 2048 -> 10880 165 / 133; 1,500 rows 1600 -> 4800 35 / 28; 12,000 rows 3072 -> 768 102 / 75.
// At full occupancy (4,096 rows 6400 -> 4096) the 256 x 256 tile reaches 1,340 TFLOP/s, the register path's 1,180; the clock is
// down to 1.95 GHz there, the matrix units are busy 65 % of the cycles.
//
// Lines: from 512 rows, 12 steps and 140 tiles on (smaller tiles, or a split, use more of the chip below).  From 32 steps on 128 x 64
// tiles keep to the range that they have above, and 128 x 192 lose what they gain by sharing a unit (12,288 rows 6400 -> 1600
// 288 us, 128 x 256 271).  Beyond 16,384 columns (the head over many tokens) memory counts for more than rounds: 256 x 256 from
// 1,000 rows on, below only where their last row of tiles is more than half full and the inner size long, else the rules above
// (rules above / 256 x 256, us, 768 -> 50304: 600 rows 73 / 88, 720 85 / 93, 850 96 / 119, 1,024 150 / 130, 2,048 304 / 264;
// 1600 -> 50304: 512 rows 109 / 104, 720 164 / 157, 850 198 / 202, 1,300 296 / 271, 4,096 750 / 724).
//
// Grouped rows (experts) count with their padding, which comes last in a group and in the call: the XCDs take equal stretches of all
// tiles, so those that got the used ones take the time (counted by used tiles the choice was 8 % slower in the mean of 224 products
// of 512 to 24,000 pairs for 8 to 64 experts, and up to 54 %; counted as here it is 8 % faster than the rules above).  Where a
// group's second half is padding, the two workgroups that share a unit leave it to one of them: 128 x 192 then win by up to 14 %
// what would be a tie (16 experts 1024 -> 2048, 512 pairs: 23.9 us, 256 x 192 26.5).
int choose_large(int n_rows, int n_out, int k_dim, bool added, bool grouped, bool chains, double* least) {
  const int steps = k_dim / MM_BK;
  if (n_rows < 512 || n_out < 512 || steps < 12) return -1;
  if (n_out > 16384) {
    const bool full = (n_rows + 255) / 256 * 2 == (n_rows + 127) / 128 && (steps >= 20 || n_rows == 512);
    return n_rows >= 1000 || full ? MM_DIRECT_FIRST + MM_DIRECT_HALVES : -1;
  }
  struct Cost { int variant, per_unit; double step, step_alone, round, round_added; };
  const Cost costs[] = {{2, 2, 0.56, 0.355, 0.3, 0.3},
                        {3, 2, steps >= 32 ? 1.2 : 1.09, 0.71, 0.2, 2.2},
                        {MM_DIRECT_HALVES, 1, 1.37, 1.30, 0.3, 7.0},
                        {MM_DIRECT_HALVES + 1, 1, 0.825, 0.76, 0.7, 3.9},
                        {MM_DIRECT_HALVES + 2, 1, 1.09, 1.05, 0.55, 6.4},
                        {MM_DIRECT_HALVES + 3, 1, 0.72, 0.645, 0.7, 2.8}};
  const double outputs = 1e-6 * n_rows * n_out, behind = added ? 4.6 + 1.28 * outputs : 3.6 + 0.68 * outputs;
  int best = -1;
  for (const Cost& c : costs) {
    const long tiles = direct_tiles(c.variant, n_rows, n_out), at_once = 256L * c.per_unit;
    if (tiles < 140 || (chains && !MM_HAS_CHAINS[c.variant])) continue;
    if (steps >= 32 && c.variant == 2 && tiles > 520) continue;
    if (steps >= 48 && c.variant == 3) continue;
    const long rest = tiles % at_once;
    const double round = added ? c.round_added : c.round;
    double t = behind + (double)(tiles / at_once) * (steps * c.step + round);
    if (rest > 0) t += steps * (rest <= 256 ? c.step_alone : c.step) + round;
    if (grouped && c.variant == 3 && tiles <= 2 * at_once) t *= 0.95;
    if (best < 0 || t < *least) best = c.variant, *least = t;
  }
  return best < 0 ? -1 : (chains ? MM_CHAINS_FIRST : MM_DIRECT_FIRST) + best;
}

// Float32 outputs that would go to the 64 x 64 tiles with two wave groups have their sums as two chains there; a large variant
// in their place makes the same two: single chains, twice as long, are further from the sums in 64 bits (2,048 rows 1600 -> 1600
// 1.08e-7 of the sums' norm, two chains 0.80e-7; 3,000 rows 6400 -> 1600 3.42e-7 / 2.39e-7).  The second set of accumulators costs
// up to 3 % (3,500 rows 5120 -> 1280 62 us instead of 61, with two wave groups 93).
//
// The 64 x 64 tiles themselves take 6.7 us and 0.19 us a step and round of 256 of them, several sharing a compute unit: less than a
// large variant with one workgroup in its second round (1,600 rows 1280 -> 1280, 500 of them 14.1 us, 260 of 128 x 64 16.7).  With
// four stages, under 32 steps and more, two on a unit take 0.39 us a step (64 x 64 / 128 x 64, us: 600 rows 2048 -> 2048 15.6 / 16.3,
// 1,300 rows 4096 -> 1024 28.0 / 29.0; 850 rows 5120 -> 1280 38.6 / 34.1).
int choose_direct(int n_rows, int n_out, int k_dim, bool f32, bool added, bool grouped) {
  if (n_rows < 128 || (k_dim % MM_BK) != 0) return -1;
  const int medium = choose_medium(n_rows, n_out, k_dim), steps = k_dim / MM_BK;
  const bool small = medium < 0 && choose_shape(n_rows, n_out) == 3;
  const long tiles = tiles_of(3, n_rows, n_out);
  double least = 0.0;
  const int large = choose_large(n_rows, n_out, k_dim, added, grouped, f32 && small && two_groups_pay(steps, tiles), &least);
  if (small && 6.7 + (double)((tiles + 255) / 256) * (0.19 * steps + (added ? 1.2 : 0.35)) < least) return medium;
  if (medium == MM_DIRECT_FIRST + 1 && (added ? 4.2 : 3.2) + 0.39 * steps < least) return medium;
  return large >= 0 ? large : medium;
}

// shape < 0: chosen by the size.  k_parts: 0 = chosen by the size, together with the shape, if
// `partials` holds enough floats (else unsplit; with a given shape unsplit too), 1 = unsplit,
// more = that many stretches (refused if the buffer is too small).
// leave_parts: the stretches' sums stay in `partials` ([parts][n_rows][n_out], the first with the
// bias), no second kernel joins them; *leave_parts gets the number of parts, 0 if the product is not split.
int launch_any(int shape, int k_parts, const void* act, long lda, const void* w, const float* bias, void* out,
               int out_dtype, long ldo, int n_rows, int n_out, int k_dim, int epilogue, float* partials,
               long partials_floats, const MfmaScatter& sc, hipStream_t stream, int* leave_parts = nullptr) {
  if (n_rows == 0 || n_out == 0) return MGPT_OK;
  if (!act || !w || !out || (epilogue == MM_EPI_XIELU && !sc.epi_coef)) return MGPT_ERR_NULL;
  if (!shapes_ok(act, lda, w, out, ldo, n_rows, n_out, k_dim)) return MGPT_ERR_BAD_SHAPE;
  // shapes MM_SHAPES and MM_SHAPES + 1: the two smallest tiles with more steps on their way from memory
  int ahead = 0;  // 0: chosen below
  bool two_groups = false;  // the 64 x 64 tile with two wave groups (shape MM_SHAPES + 2)
  int direct = -1;  // which of the variants whose slices go straight into LDS (-1: through registers)
  bool chains = false;  // two chains of sums
  if (shape < 0 && k_parts <= 1 && !leave_parts) {
    const int chosen = direct_ok(act, w, k_dim) ? choose_direct(n_rows, n_out, k_dim, out_dtype == MGPT_F32, epilogue == MM_EPI_RESIDUAL,
                                                              sc.row_expert != nullptr)
                                              : -1;
    if (chosen >= 0) shape = chosen, k_parts = 1;
  }
  bool rows = false, rows_32 = false;  // the kernel for few rows, with 32 columns a workgroup
  if (shape >= MM_ROWS) {
    if (shape >= MM_SHAPE_IDS || n_rows > MM_ROWS_MAX || sc.row_expert || !direct_ok(act, w, k_dim)) return MGPT_ERR_BAD_SHAPE;
    rows = true;
    rows_32 = shape == MM_ROWS + 1;
    shape = 3;   // (the rules below for the other variants do not apply)
    ahead = 1;
  } else if (shape >= MM_DIRECT_FIRST) {
    if (shape >= MM_SHAPE_IDS || !direct_ok(act, w, k_dim)) return MGPT_ERR_BAD_SHAPE;
    chains = shape >= MM_CHAINS_FIRST;
    direct = shape - (chains ? MM_CHAINS_FIRST : MM_DIRECT_FIRST);
    if (chains && (!MM_HAS_CHAINS[direct] || out_dtype != MGPT_F32)) return MGPT_ERR_BAD_SHAPE;
    if (direct >= MM_DIRECT_HALVES && k_parts > 1) return MGPT_ERR_BAD_SHAPE;   // (these are not split)
    shape = 3;   // (the rules below for the other variants do not apply)
    ahead = 1;
  } else if (shape == MM_SHAPES + 2) {
    shape = 3;
    ahead = 1;
    two_groups = true;
  } else if (shape >= MM_SHAPES && shape < MM_SHAPES + 2) {
    shape -= 2;
    ahead = MM_AHEAD;
  } else if (shape >= 0) {
    ahead = 1;
  }
  const bool forced = k_parts > 1;
  if (shape < 0 && k_parts == 0 && partials) {
    choose_split(n_rows, n_out, k_dim, epilogue, &shape, &k_parts);
    if (k_parts > 1 && (long)used_parts(k_dim, k_parts) * n_rows * n_out > partials_floats) shape = -1, k_parts = 1;
  }
  if (shape < 0) shape = choose_shape(n_rows, n_out);
  if (shape >= MM_SHAPES) return MGPT_ERR_BAD_SHAPE;
  if (k_parts == 0) k_parts = 1;
  if (ahead == 0) {
    // Few small tiles over a long enough stretch: the workgroups are too few to hide a trip to
    // memory behind one another.  Measured over matrices that come from memory, 32 x 32 tiles, 40-64
    // rows: [4800 x 1600] 9.8-10.0 us against 10.8, [6400 x 1600] 10.7-11.9 against 15.6, [1600 x 1600]
    // 8.4 against 10.3 (and 8.6 / 10.5 at 136 rows, 250 tiles), [4096 x 1024] 6.3 against 7.6; with more
    // than two such workgroups a compute unit nothing is gained ([4800 x 1600] at 136 rows, 750 tiles:
    // 12.8 against 11.7).
    const int steps = (k_dim + MM_BK - 1) / MM_BK;
    ahead = (shape == 4 && steps / k_parts >= 12 && tiles_of(4, n_rows, n_out) * k_parts <= 512) ? MM_AHEAD : 1;
    // The same with the slices straight into LDS, where the operands allow it: the steps on their way need no
    // registers, so there can be more of them (six stages while a compute unit has one such workgroup, four
    // with more).  Decode steps of 12 layers of width 1600, in turns with the variant above on one box: 24 rows
    // 0.774 -> 0.740 ms, 32 rows 0.795 -> 0.762, 64 rows 1.000 -> 0.949 (with six stages there 0.970).
    // Under fewer than 20 steps four stages are enough (310 rows 768 -> 768 with the LayerNorm behind it: 8.1 us with six, 7.7).
    if (ahead == MM_AHEAD && direct_ok(act, w, k_dim)) {
      direct = tiles_of(4, n_rows, n_out) * k_parts <= 256 && steps >= 20 ? 4 : 0;
      ahead = 1;
    }
    // Prompt portions of a few hundred rows under an inner size of 20 to 31 steps (longer ones have their rule above): 64 x 64 tiles
    // with four stages from 160 tiles on, up to one a compute unit.  Over inner sizes 1,280 to 1,920, outputs 768 to 4,800 and 128 to
    // 1,024 rows they take 9 to 22 % less than 32 or 64 wide tiles through registers, alone in a graph (400 rows 1600 -> 1600 12.9 /
    // 10.3 us); with the LayerNorm behind them 400 rows 17.2 / 15.3, 520 rows 18.0 / 15.8, 310 rows (125 tiles) 13.3 / 15.1.
    if (direct < 0 && n_rows >= 128 && k_parts == 1 && steps >= 20 && (shape == 3 || shape == 4) && direct_ok(act, w, k_dim)) {
      const long t64 = tiles_of(3, n_rows, n_out);
      if (t64 >= 160 && t64 <= 256) direct = 1, ahead = 1;
    }
  }
  if (k_parts > 1) {
    k_parts = used_parts(k_dim, k_parts > MM_MAX_PARTS ? MM_MAX_PARTS : k_parts);
    const bool fits = partials && (long)k_parts * n_rows * n_out <= partials_floats &&
                      (((size_t)partials) & 15) == 0 && (n_out & 3) == 0 && epilogue != MM_EPI_QKV;
    if (!fits) {
      if (forced) return MGPT_ERR_BAD_SHAPE;
      k_parts = 1;
    }
  }
  const bool split = k_parts > 1;
  // Up to 32 rows under a narrow output and a long inner size (64 under matrices of less than 6 million elements), where these tiles
  // stand in for the decode kernel, whose sums are 16 chains: chains of two steps.  Error of 16 rows 6400 -> 1600 against 64 bits, relative to the sums' norm: decode kernel
  // 1.35e-7, eight stretches of one chain 1.84e-7, of short ones 1.02e-7; 6.5 and 6.8 us.
  const bool fold = !forced && split && shape == 4 && n_rows <= ((long)n_out * k_dim < 6000000 ? 64 : 32) && n_out < 4096 && k_dim > 4096;
  if (two_groups) {
    // forced: what this kernel stores must be float32, plain or added into the residual stream (the sums of
    // a split product are)
    const int dt_here = split ? MGPT_F32 : out_dtype, epi_here = split ? MM_EPI_NONE : epilogue;
    if (dt_here != MGPT_F32 || (epi_here != MM_EPI_NONE && epi_here != MM_EPI_RESIDUAL)) return MGPT_ERR_BAD_SHAPE;
  } else if (shape == 3 && ahead == 1 && direct < 0 && !rows) {
    const int steps_here = ((k_dim + MM_BK - 1) / MM_BK + k_parts - 1) / k_parts;
    const int dt_here = split ? MGPT_F32 : out_dtype, epi_here = split ? MM_EPI_NONE : epilogue;
    two_groups = two_groups_pay(steps_here, tiles_of(3, n_rows, n_out) * k_parts) && dt_here == MGPT_F32 &&
                 (epi_here == MM_EPI_NONE || epi_here == MM_EPI_RESIDUAL);
  }
  if (leave_parts) {
    *leave_parts = split ? k_parts : 0;
    if (!split) return MGPT_OK;  // nothing launched: the caller takes another way
  }
  void* dst = split ? (void*)partials : out;
  const float* b = (split && !leave_parts) ? nullptr : bias;
  const int dt = split ? MGPT_F32 : out_dtype, epi = split ? MM_EPI_NONE : epilogue;
  const long ld = split ? n_out : ldo, stride = split ? (long)n_rows * n_out : 0;
#define MM_ARGS act, lda, w, b, dst, dt, ld, n_rows, n_out, k_dim, epi, k_parts, stride, sc, stream
  int rc = MGPT_ERR_BAD_SHAPE;
#define MM_FOLD_ARGS act, lda, w, b, dst, ld, n_rows, n_out, k_dim, k_parts, stride, sc, stream
#define MM_HALVES_ARGS act, lda, w, b, dst, dt, ld, n_rows, n_out, k_dim, epi, sc, stream
  if (fold) {
    rc = direct == 4   ? launch_one<1, 1, 2, 2, MM_EPI_NONE, float, 1, 1, 6, 1, MM_FOLD>(MM_FOLD_ARGS)
         : direct == 0 ? launch_one<1, 1, 2, 2, MM_EPI_NONE, float, 1, 1, 4, 1, MM_FOLD>(MM_FOLD_ARGS)
         : ahead > 1   ? launch_one<1, 1, 2, 2, MM_EPI_NONE, float, MM_AHEAD, 1, 0, 1, MM_FOLD>(MM_FOLD_ARGS)
                       : launch_one<1, 1, 2, 2, MM_EPI_NONE, float, 1, 1, 0, 1, MM_FOLD>(MM_FOLD_ARGS);
  } else if (rows) {
    if (n_rows <= 16) rc = rows_32 ? launch_rows<1, 2, 3>(MM_ARGS) : launch_rows<1, 1, 4>(MM_ARGS);
    else rc = rows_32 ? launch_rows<2, 2, 2>(MM_ARGS) : launch_rows<2, 1, 3>(MM_ARGS);
  } else if (direct >= 0 && chains) {
    switch (direct) {
      case 2: rc = launch_shape<2, 2, 4, 2, 1, 3, 2>(MM_ARGS); break;
      case 6: rc = launch_halves<4, 4, 2>(MM_HALVES_ARGS); break;
      case 8: rc = launch_halves<4, 3, 2>(MM_HALVES_ARGS); break;
      default: break;
    }
  } else if (direct >= 0) {
    switch (direct) {
      case 0: rc = launch_shape<1, 1, 2, 2, 1, 4>(MM_ARGS); break;
      case 1: rc = launch_shape<2, 2, 2, 2, 1, 4>(MM_ARGS); break;
      case 2: rc = launch_shape<2, 2, 4, 2, 1, 3>(MM_ARGS); break;
      case 3: rc = launch_shape<4, 3, 2, 4, 1, 2>(MM_ARGS); break;
      case 4: rc = launch_shape<1, 1, 2, 2, 1, 6>(MM_ARGS); break;
      case 5: rc = launch_halves<8, 4>(MM_HALVES_ARGS); break;
      case 6: rc = launch_halves<4, 4>(MM_HALVES_ARGS); break;
      case 7: rc = launch_halves<8, 3>(MM_HALVES_ARGS); break;
      case 8: rc = launch_halves<4, 3>(MM_HALVES_ARGS); break;
      default: break;
    }
  } else
  switch (shape) {
    case 0: rc = launch_shape<8, 4, 2, 4>(MM_ARGS); break;  // 256 x 256, eight waves of 128 x 64
    case 1: rc = launch_shape<4, 4, 2, 4>(MM_ARGS); break;  // 128 x 256, eight waves of 64 x 64
    case 2: rc = launch_shape<4, 2, 2, 2>(MM_ARGS); break;  // 128 x 64, four waves of 64 x 32
    case 3:  // 64 x 64, four waves of 32 x 32 (or eight, in two groups)
      rc = two_groups ? launch_two_groups(MM_ARGS)
                      : ahead > 1 ? launch_shape<2, 2, 2, 2, MM_AHEAD>(MM_ARGS) : launch_shape<2, 2, 2, 2>(MM_ARGS);
      break;
    case 4:  // 32 x 32, four waves of 16 x 16
      rc = ahead > 1 ? launch_shape<1, 1, 2, 2, MM_AHEAD>(MM_ARGS) : launch_shape<1, 1, 2, 2>(MM_ARGS);
      break;
  }
#undef MM_HALVES_ARGS
#undef MM_FOLD_ARGS
#undef MM_ARGS
  if (rc != MGPT_OK || !split || leave_parts) return rc;
  return launch_join(partials, k_parts, bias, out, out_dtype, ldo, n_rows, n_out, epilogue, stream, sc.epi_coef);
}

}  // namespace

// A product of up to 32 rows in whole steps of 64: 0 where the kernel that has nothing but them and a few columns a workgroup is not the
// fastest, else its shape for mgpt_linear_mfma_shape + 256 x the stretches of the inner size.
extern "C" int mgpt_linear_mfma_rows_plan(int n_rows, int n_out, int k_dim, int epilogue) {
  if (!rows_take(n_rows, n_out, k_dim)) return 0;
  const int parts = epilogue == MM_EPI_QKV || (n_out & 3) != 0 ? 1 : used_parts(k_dim, rows_parts(n_rows, n_out, k_dim));
  return MM_ROWS + (rows_wide(n_rows, n_out, parts) ? 1 : 0) + 256 * parts;
}

// How many floats of scratch the product would use if it were split along its inner size (0: it
// would not be split).  The caller brings that buffer to mgpt_linear_mfma.
extern "C" long mgpt_linear_mfma_partials(int n_rows, int n_out, int k_dim, int epilogue) {
  if (n_rows <= 0 || n_out <= 0 || k_dim <= 0) return 0;
  int shape, parts;
  choose_split(n_rows, n_out, k_dim, epilogue, &shape, &parts);
  return parts > 1 ? (long)used_parts(k_dim, parts) * n_rows * n_out : 0;
}

// The first half of a split product alone: partials[p][n][o] = the sum over stretch p of the inner
// size (+ bias[o] in p = 0), p < mgpt_linear_mfma_partials(n_rows, n_out, k_dim, residual epilogue) /
// (n_rows * n_out), for a caller that adds the parts up itself (a pending residual: fused_decode.h).
// MGPT_ERR_BAD_SHAPE, with nothing launched, if the product would not be split or the buffer is too small.
extern "C" int mgpt_linear_mfma_parts(const void* act, long lda, const void* w, const float* bias, float* partials,
                                      long partials_floats, int n_rows, int n_out, int k_dim, hipStream_t stream) {
  if (!partials) return MGPT_ERR_NULL;
  MfmaScatter sc = {};
  int parts = 0;
  const int rc = launch_any(-1, 0, act, lda, w, bias, partials, MGPT_F32, n_out, n_rows, n_out, k_dim, MM_EPI_RESIDUAL,
                            partials, partials_floats, sc, stream, &parts);
  if (rc != MGPT_OK) return rc;
  return parts > 1 ? MGPT_OK : MGPT_ERR_BAD_SHAPE;
}

// The same with the shape and the number of stretches given (mgpt_linear_mfma_shape).
extern "C" int mgpt_linear_mfma_shape_parts(int shape, int k_parts, const void* act, long lda, const void* w, const float* bias,
                                            float* partials, long partials_floats, int n_rows, int n_out, int k_dim,
                                            hipStream_t stream) {
  if (!partials) return MGPT_ERR_NULL;
  if (shape < 0 || shape >= MM_SHAPE_IDS || k_parts <= 1 || k_parts != used_parts(k_dim, k_parts)) return MGPT_ERR_BAD_SHAPE;
  MfmaScatter sc = {};
  int parts = 0;
  const int rc = launch_any(shape, k_parts, act, lda, w, bias, partials, MGPT_F32, n_out, n_rows, n_out, k_dim, MM_EPI_RESIDUAL,
                            partials, partials_floats, sc, stream, &parts);
  if (rc != MGPT_OK) return rc;
  return parts > 1 ? MGPT_OK : MGPT_ERR_BAD_SHAPE;
}

// Which variant whose slices go straight into LDS an unsplit product of 128 and more rows goes to (a shape id as for
// mgpt_linear_mfma_shape, for operands aligned to 16 bytes), or -1: one of those through registers, or one of the smallest tiles.
extern "C" int mgpt_linear_mfma_choice(int n_rows, int n_out, int k_dim, int out_dtype, int epilogue, int grouped) {
  return choose_direct(n_rows, n_out, k_dim, out_dtype == MGPT_F32, epilogue == MM_EPI_RESIDUAL, grouped != 0);
}

// act: [n_rows, k_dim] bfloat16 with row stride lda (a multiple of 8, 16-byte aligned base);
// w: [n_out, k_dim] dense bfloat16; out: [n_rows, n_out] with row stride ldo.  k_dim must be a
// multiple of 16.  partials: scratch of partials_floats floats (16-byte aligned) or null; with it
// a long inner size over few tiles is split (mgpt_linear_mfma_partials says how much that needs).
// Refuses other layouts with MGPT_ERR_BAD_SHAPE.
extern "C" int mgpt_linear_mfma(const void* act, long lda, const void* w, const float* bias, void* out,
                                int out_dtype, long ldo, int n_rows, int n_out, int k_dim, int epilogue,
                                float* partials, long partials_floats, hipStream_t stream) {
  if (epilogue == MM_EPI_QKV) return MGPT_ERR_BAD_SHAPE;  // mgpt_linear_mfma_qkv brings the pools
  MfmaScatter sc = {};
  return launch_any(-1, 0, act, lda, w, bias, out, out_dtype, ldo, n_rows, n_out, k_dim, epilogue, partials,
                    partials_floats, sc, stream);
}

// The same product with the xIELU activation behind it (bfloat16 out): coef = float32 (a_p, a_n), the coefficients of
// v^2 for v > 0 and of (exp(v) - 1 - v) for v <= 0, beside v / 2 in both.
extern "C" int mgpt_linear_mfma_xielu(const void* act, long lda, const void* w, const float* bias, void* out,
                                      long ldo, int n_rows, int n_out, int k_dim, const float* coef, float* partials,
                                      long partials_floats, hipStream_t stream) {
  if (!coef) return MGPT_ERR_NULL;
  MfmaScatter sc = {};
  sc.epi_coef = coef;
  return launch_any(-1, 0, act, lda, w, bias, out, MGPT_BF16, ldo, n_rows, n_out, k_dim, MM_EPI_XIELU, partials,
                    partials_floats, sc, stream);
}

// The same product with the tile shape given (0 = 256 x 256, 1 = 128 x 256, 2 = 128 x 64,
// 3 = 64 x 64, 4 = 32 x 32, 5 and 6 = 64 x 64 and 32 x 32 with four steps on their way from memory,
// 7 = 64 x 64 with two wave groups a tile (float32 outputs), 8 to 12 = the slices straight into LDS: 32 x 32 and
// 64 x 64 with four stages, 128 x 64 with three, 128 x 192 with two, 32 x 32 with six (an inner size of whole steps of 64 and operands
// aligned to 16 bytes, else refused), 13 to 16 = the halves out of step, 256 x 256, 128 x 256, 256 x 192, 128 x 192 (the same
// conditions, and never split), 19, 23 and 25 = 10, 14 and 16 with two chains of sums (float32 outputs), 26 and 27 = up to 32 rows
// with 16 and 32 columns a workgroup (the conditions of 8, not with xIELU); negative: chosen) and the number of stretches of the inner size given
// (k_parts as for launch_any above), instead of chosen by the size: for tests and measurements.
extern "C" int mgpt_linear_mfma_shape(int shape, int k_parts, const void* act, long lda, const void* w,
                                      const float* bias, void* out, int out_dtype, long ldo, int n_rows,
                                      int n_out, int k_dim, int epilogue, float* partials, long partials_floats,
                                      hipStream_t stream) {
  if (epilogue == MM_EPI_QKV || shape >= MM_SHAPE_IDS || k_parts < 0) return MGPT_ERR_BAD_SHAPE;
  MfmaScatter sc = {};
  return launch_any(shape, k_parts, act, lda, w, bias, out, out_dtype, ldo, n_rows, n_out, k_dim, epilogue,
                    partials, partials_floats, sc, stream);
}

// Rows in groups of group_rows (256) that each multiply a matrix of their own: out[r] = act[r] W_e^T with
// e = row_expert[r / group_rows] (negative: nothing is computed for the group) and W_e = w + e * w_stride;
// row_valid[r] < 0 marks the padding that ends a group, and a tile that starts in it is skipped.  bfloat16 or
// float32 out, no bias, no epilogue or (bfloat16 out) the squared relu, the inner size never split.
extern "C" int mgpt_linear_mfma_grouped(const void* act, long lda, const void* w, long w_stride, const int* row_expert,
                                        const int* row_valid, int group_rows, void* out, int out_dtype, long ldo,
                                        int n_rows, int n_out, int k_dim, int epilogue, hipStream_t stream) {
  if (!row_expert || !row_valid) return MGPT_ERR_NULL;
  if (epilogue != MM_EPI_NONE && epilogue != MM_EPI_RELU2) return MGPT_ERR_BAD_SHAPE;
  // every tile shape's rows (32 to 256) divide a group
  if (group_rows != 256 || (n_rows % group_rows) != 0 || w_stride < (long)n_out * k_dim || (w_stride & 7) != 0)
    return MGPT_ERR_BAD_SHAPE;
  MfmaScatter sc = {};
  sc.row_expert = row_expert;
  sc.row_valid = row_valid;
  sc.group_rows = group_rows;
  sc.w_stride = w_stride;
  return launch_any(-1, 1, act, lda, w, nullptr, out, out_dtype, ldo, n_rows, n_out, k_dim, epilogue, nullptr, 0, sc,
                    stream);
}

// The fused QKV product of a step with prompt portions: out[n] = act[n] W^T + bias in bfloat16, and
// the key and value columns (after the first q_width) of every row with a slot also go into the
// cache pools [pages, n_kv_head, page_size, head_dim].  Refuses (MGPT_ERR_BAD_SHAPE) sizes that
// are no multiples of 4 and outputs that are not aligned for 8-byte stores.  shape: as for
// mgpt_linear_mfma_shape, or negative to have it chosen.
extern "C" int mgpt_linear_mfma_qkv(const void* act, long lda, const void* w, const float* bias, void* out,
                                    long ldo, int n_rows, int n_out, int k_dim, void* kpool, void* vpool,
                                    const int* slot_mapping, int q_width, int kv_width, int head_dim,
                                    int n_kv_head, int page_size, int shape, hipStream_t stream) {
  if (!kpool || !vpool || !slot_mapping) return MGPT_ERR_NULL;
  if (head_dim <= 0 || (head_dim % 4) != 0 || (q_width % 4) != 0 || q_width + 2 * kv_width != n_out ||
      kv_width != n_kv_head * head_dim || page_size <= 0 || (n_out % 4) != 0 || (ldo % 4) != 0 ||
      (((size_t)out | (size_t)bias) & 15) != 0 || (shape >= MM_SHAPES + 2 && shape < MM_DIRECT_FIRST) ||
      shape >= MM_SHAPE_IDS)
    return MGPT_ERR_BAD_SHAPE;
  MfmaScatter sc = {(bf16_t*)kpool, (bf16_t*)vpool, slot_mapping, q_width, kv_width, head_dim, n_kv_head, page_size};
  return launch_any(shape, 1, act, lda, w, bias, out, MGPT_BF16, ldo, n_rows, n_out, k_dim, MM_EPI_QKV, nullptr, 0, sc,
                    stream);
}
