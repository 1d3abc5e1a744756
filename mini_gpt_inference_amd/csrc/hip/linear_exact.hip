// out[n, o] = sum_k A[n, k] W[o, k] (+ bias[o]) with an optional GELU-tanh, squared-relu or residual-add epilogue, all in
// 32 bits on the matrix cores (v_mfma_f32_16x16x4_f32: float32 products and sums): the product of the true 32-bit path
// (reference: src/minigpt_infer/model.py:43-44,96-101).
//
// The order of an element's sum depends on nothing but k, so that a token's logits are the same bits however the tokens
// were cut into steps: k is cut into blocks of 256; a block's sum runs over groups of 16 k from zero, a group as four
// matrix instructions of which the i-th takes k = i, 4 + i, 8 + i, 12 + i (what a lane loads as one 16-byte piece serves
// all four); the blocks' sums are added up in order, then the bias.  What is missing to a group counts as zeros.  All
// kernels below keep to that, whatever their tiles, and whether one wave has all blocks of an element or each wave some.
#include "common.h"
#include "launchers.h"
#include "linear_exact.h"

#define EPI_NONE 0
#define EPI_GELU 1
#define EPI_RESIDUAL 2  // out += result
#define EPI_QKV 3       // out = result; key and value columns also into their pages
#define EPI_RELU2 5     // max(result, 0)^2

#define EX_BLOCK 256    // k of a block
#define EX_GROUP 16     // k of a group

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float ex_f4;

template <int EPI>
__device__ __forceinline__ float ex_epilogue(float v, float old) {
  if (EPI == EPI_GELU) return gelu_tanh(v);
  if (EPI == EPI_RELU2) return relu_squared(v);
  if (EPI == EPI_RESIDUAL) return old + v;
  return v;
}

// Where a key or value column c >= q_width of token row r goes, or null (a padded row).
__device__ __forceinline__ float* ex_page_row(const ExactScatter& sc, int r, int c) {
  const int slot = sc.slot_mapping[r];
  if (slot < 0) return nullptr;
  c -= sc.q_width;
  float* pool = c < sc.kv_width ? sc.kpool : sc.vpool;
  if (c >= sc.kv_width) c -= sc.kv_width;
  const int page = slot / sc.page_size, h = c / sc.head_dim;
  return pool + ((long)(page * (sc.kv_width / sc.head_dim) + h) * sc.page_size + (slot - page * sc.page_size)) * sc.head_dim +
         (c - h * sc.head_dim);
}

// Four k of a row from k on; those at or beyond k_dim count as zero.  VEC: rows are 16-byte aligned and k_dim is a multiple
// of 4.
template <bool VEC>
__device__ __forceinline__ ex_f4 ex_load(const float* __restrict__ row, int k, int k_dim) {
  ex_f4 v = {0.f, 0.f, 0.f, 0.f};
  if (VEC) {
    if (k < k_dim) v = *reinterpret_cast<const ex_f4*>(row + k);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float x = row[k + i < k_dim ? k + i : k_dim - 1];   // (no branch between the loads)
      v[i] = k + i < k_dim ? x : 0.f;
    }
  }
  return v;
}

// Many rows: a workgroup of four waves per tile of 32 T rows x 32 T columns, a wave 16 T x 16 T of them; steps of 32 k
// through two buffers of LDS (STAGES == 0; else that many), rows of 128 bytes whose 16-byte pieces are XORed with the row's low
// bits.  The matrix cores' float32 rate (a sixteenth of bfloat16's) is what bounds it, with T = 4 from about 256 tiles on.
//
// STAGES > 0: the slices go from memory straight into LDS (global_load_lds_dwordx4: a wave's load brings 8 rows of 128 bytes,
// the lane that fills piece p of row r fetching piece p ^ (r & 7)), STAGES - 1 steps on their way, for inner sizes of whole
// steps: through registers one step is on its way, and a workgroup that is alone on its compute unit waits for memory every step.
// Before / now, us: 1,201 rows 2048 -> 512 54.6 / 46.4, 512 -> 50304 588 / 562; 2,000 rows 768 -> 768 34.3 / 31.8, 3072 -> 768
// 121.7 / 108.4; 600 rows 5120 -> 1280 128.8 / 108.3; 5,000 rows 1600 -> 6400 859 / 828 (124 TFLOP/s).  Eight waves a tile instead
// of four: the same.
#define EX_BK 32
template <int T, int EPI, bool VEC, int STAGES>
__global__ __launch_bounds__(256) void linear_exact_tile_kernel(
    const float* __restrict__ A, long lda, const float* __restrict__ W, const float* __restrict__ bias,
    float* __restrict__ out, long ldo, int n_rows, int n_out, int k_dim, int row_tiles, int vec_out, ExactScatter sc) {
  constexpr int B = 32 * T;                          // rows and columns of the tile
  constexpr int PIECES = B * EX_BK / 4 / 256;        // 16-byte pieces of one operand's slice that a thread stages
  extern __shared__ __align__(16) float ex_lds[];    // [buffers][2 B][EX_BK]: rows of activations, then of W
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = (int)(blockIdx.x % row_tiles) * B, col0 = (int)(blockIdx.x / row_tiles) * B;
  const int wr = (wave & 1) * 16 * T, wc = (wave >> 1) * 16 * T;
  const int l16 = lane & 15, lk = lane >> 4;

  // rows past the end are read from the last one: their results are never stored
  constexpr int ROW = EX_BK / 4, STEP = 256 / ROW;   // pieces of a row, rows that 256 threads stage at a time
  const int srow = tid / ROW, sp = tid % ROW;        // this thread's piece of a slice: row srow + STEP p
  const float* ap[PIECES];
  const float* wp[PIECES];
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const int r = row0 + srow + STEP * p, c = col0 + srow + STEP * p;
    ap[p] = A + (long)(r < n_rows ? r : n_rows - 1) * lda;
    wp[p] = W + (long)(c < n_out ? c : n_out - 1) * k_dim;
  }
  const int s_lds = srow * EX_BK + ((sp ^ (srow & 7)) << 2);
  [[maybe_unused]] ex_f4 ga[PIECES], gw[PIECES];
  auto load = [&](int k0) {
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      ga[p] = ex_load<VEC>(ap[p], k0 + 4 * sp, k_dim);
      gw[p] = ex_load<VEC>(wp[p], k0 + 4 * sp, k_dim);
    }
  };
  auto store = [&](int buf) {
    float* dst = ex_lds + buf * (2 * B * EX_BK) + s_lds;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      *reinterpret_cast<ex_f4*>(dst + STEP * p * EX_BK) = ga[p];
      *reinterpret_cast<ex_f4*>(dst + (B + STEP * p) * EX_BK) = gw[p];
    }
  };

  ex_f4 acc[T][T], sum[T][T];                        // [column tile][row tile]: the block's sum, the blocks' sum
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j) acc[i][j] = sum[i][j] = (ex_f4){0.f, 0.f, 0.f, 0.f};

  // the step at k0, whose slices lie in buffer buf
  auto multiply = [&](int k0, int buf) {
    const float* as = ex_lds + buf * (2 * B * EX_BK) + (wr + l16) * EX_BK;
    const float* ws = ex_lds + buf * (2 * B * EX_BK) + (B + wc + l16) * EX_BK;
#pragma unroll
    for (int g = 0; g < EX_BK / EX_GROUP; ++g) {
      const int piece = ((4 * g + lk) ^ (l16 & 7)) << 2;
      ex_f4 af[T], wf[T];
#pragma unroll
      for (int t = 0; t < T; ++t) {
        af[t] = *reinterpret_cast<const ex_f4*>(as + t * 16 * EX_BK + piece);
        wf[t] = *reinterpret_cast<const ex_f4*>(ws + t * 16 * EX_BK + piece);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
          for (int j = 0; j < T; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][e], af[j][e], acc[i][j], 0, 0, 0);
    }
    if (((k0 + EX_BK) & (EX_BLOCK - 1)) == 0 || k0 + EX_BK >= k_dim) {
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = (ex_f4){0.f, 0.f, 0.f, 0.f};
        }
    }
  };
  if constexpr (STAGES > 0) {
    constexpr int LOADS = 2 * B / 8 / 4;             // of a wave and step: 8 rows each, the activations' first
    constexpr int D = STAGES - 1;
    typedef __attribute__((address_space(1))) const void* global_ptr_t;
    typedef __attribute__((address_space(3))) void* lds_ptr_t;
    const int lr = lane >> 3, lc = ((lane & 7) ^ lr) << 2;
    const float* dp[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int r = (wave + 4 * i) * 8 + lr;
      if (i < LOADS / 2) dp[i] = A + (long)(row0 + r < n_rows ? row0 + r : n_rows - 1) * lda + lc;
      else dp[i] = W + (long)(col0 + r - B < n_out ? col0 + r - B : n_out - 1) * k_dim + lc;
    }
    auto issue = [&](int k0, int buf) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i)
        __builtin_amdgcn_global_load_lds((global_ptr_t)(dp[i] + k0),
                                         (lds_ptr_t)(ex_lds + buf * (2 * B * EX_BK) + (wave + 4 * i) * (8 * EX_BK)), 16, 0, 0);
    };
    const int steps = k_dim / EX_BK;
#pragma unroll
    for (int j = 0; j < D; ++j)
      if (j < steps) issue(j * EX_BK, j);
    for (int s = 0, buf = 0; s < steps; ++s) {
      // this wave's loads of step s have arrived (D - 1 younger steps may be on their way), then everybody's; nobody reads
      // the buffer of step s - 1 any more, which is where step s + D goes
      if (s + D <= steps) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * LOADS) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      if (s + D < steps) issue((s + D) * EX_BK, buf == 0 ? STAGES - 1 : buf - 1);
      multiply(s * EX_BK, buf);
      buf = buf + 1 == STAGES ? 0 : buf + 1;
    }
  } else {
    load(0);
    store(0);
    __syncthreads();
    for (int k0 = 0, buf = 0; k0 < k_dim; k0 += EX_BK, buf ^= 1) {
      const bool more = k0 + EX_BK < k_dim;
      if (more) load(k0 + EX_BK);
      // (the lines of multiply once more: called, the compiler lays this loop out otherwise, 2 % slower with 64 x 64 tiles and up to
      // 15 % with 128 x 128)
      const float* as = ex_lds + buf * (2 * B * EX_BK) + (wr + l16) * EX_BK;
      const float* ws = ex_lds + buf * (2 * B * EX_BK) + (B + wc + l16) * EX_BK;
#pragma unroll
      for (int g = 0; g < EX_BK / EX_GROUP; ++g) {
        const int piece = ((4 * g + lk) ^ (l16 & 7)) << 2;
        ex_f4 af[T], wf[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
          af[t] = *reinterpret_cast<const ex_f4*>(as + t * 16 * EX_BK + piece);
          wf[t] = *reinterpret_cast<const ex_f4*>(ws + t * 16 * EX_BK + piece);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int i = 0; i < T; ++i)
#pragma unroll
            for (int j = 0; j < T; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][e], af[j][e], acc[i][j], 0, 0, 0);
      }
      if (((k0 + EX_BK) & (EX_BLOCK - 1)) == 0 || !more) {
#pragma unroll
        for (int i = 0; i < T; ++i)
#pragma unroll
          for (int j = 0; j < T; ++j) {
            sum[i][j] += acc[i][j];
            acc[i][j] = (ex_f4){0.f, 0.f, 0.f, 0.f};
          }
      }
      if (more) store(buf ^ 1);
      __syncthreads();
    }
  }

  // a lane has four consecutive columns of a row
#pragma unroll
  for (int j = 0; j < T; ++j) {
    const int r = row0 + wr + 16 * j + l16;
    if (r >= n_rows) continue;
#pragma unroll
    for (int i = 0; i < T; ++i) {
      const int c = col0 + wc + 16 * i + 4 * lk;
      float* dst = out + (long)r * ldo + c;
      if (vec_out && c + 4 <= n_out) {
        ex_f4 v = sum[i][j];
        if (bias) v += *reinterpret_cast<const ex_f4*>(bias + c);
        ex_f4 old = {0.f, 0.f, 0.f, 0.f};
        if (EPI == EPI_RESIDUAL) old = *reinterpret_cast<const ex_f4*>(dst);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = ex_epilogue<EPI>(v[e], old[e]);
        *reinterpret_cast<ex_f4*>(dst) = v;
        if (EPI == EPI_QKV && c >= sc.q_width) {       // four columns of one head: all sizes are multiples of 4
          if (float* at = ex_page_row(sc, r, c)) *reinterpret_cast<ex_f4*>(at) = v;
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < n_out) {
            float v = sum[i][j][e];
            if (bias) v += bias[c + e];
            dst[e] = v = ex_epilogue<EPI>(v, EPI == EPI_RESIDUAL ? dst[e] : 0.f);
            if (EPI == EPI_QKV && c + e >= sc.q_width) {
              if (float* at = ex_page_row(sc, r, c + e)) *at = v;
            }
          }
      }
    }
  }
}

// Few rows, or a product whose tiles would leave compute units idle: a workgroup per 16 rows x 16 columns, each of its
// waves on blocks of its own (wave w: blocks w, w + waves, ...), operands straight from memory; the blocks' sums meet in
// LDS and are added up in order.  Four groups of a block are loaded while the four before are multiplied.  Nothing is
// shared between waves, so beyond a few dozen rows its loads bound it, at 26 to 33 TFLOP/s.
//
// SHORT: inner sizes of up to 192, whose last groups are not there at all, not even as zeros to add (16 rows with an inner size
// of 64 / 37: 4.2 / 6.1 us with those zeros, 3.4 / 3.5 without; the test costs longer ones 0.15 us).
template <int EPI, bool VEC, bool SHORT>
__global__ __launch_bounds__(1024) void linear_exact_rows_kernel(
    const float* __restrict__ A, long lda, const float* __restrict__ W, const float* __restrict__ bias,
    float* __restrict__ out, long ldo, int n_rows, int n_out, int k_dim, int row_tiles, ExactScatter sc) {
  constexpr int N = 256;                             // elements of the tile
  constexpr int U = 4;                               // groups on their way
  extern __shared__ __align__(16) float ex_lds[];    // [waves][N]
  const int tid = threadIdx.x, lane = tid & 63, waves = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = (int)(blockIdx.x % row_tiles) * 16, col0 = (int)(blockIdx.x / row_tiles) * 16;
  const int l16 = lane & 15, lk = lane >> 4;
  const int blocks = (k_dim + EX_BLOCK - 1) / EX_BLOCK;
  const int lr = row0 + l16, lc = col0 + l16;
  const float* ap = A + (long)(lr < n_rows ? lr : n_rows - 1) * lda;
  const float* wp = W + (long)(lc < n_out ? lc : n_out - 1) * k_dim;

  // element e of the tile: row e / 16, column e % 16; a thread adds up e = tid, tid + threads, ...
  float total[N / 64] = {0.f, 0.f, 0.f, 0.f};
  for (int b0 = 0; b0 < blocks; b0 += waves) {
    const int b = b0 + wave;
    ex_f4 acc = {0.f, 0.f, 0.f, 0.f};
    if (b < blocks) {
      const int kb = b * EX_BLOCK + 4 * lk;
      ex_f4 af[2][U], wf[2][U];
      auto load = [&](int set, int k) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          wf[set][u] = ex_load<VEC>(wp, k + u * EX_GROUP, k_dim);
          af[set][u] = ex_load<VEC>(ap, k + u * EX_GROUP, k_dim);
        }
      };
      load(0, kb);
#pragma unroll
      for (int q = 0; q < EX_BLOCK / EX_GROUP / U; ++q) {
        if (SHORT && q && q * U * EX_GROUP >= k_dim) break;
        if (q + 1 < EX_BLOCK / EX_GROUP / U) load((q + 1) & 1, kb + (q + 1) * U * EX_GROUP);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[q & 1][u][e], af[q & 1][u][e], acc, 0, 0, 0);
      }
    }
    if (b0) __syncthreads();                         // the round before has been added up
    *reinterpret_cast<ex_f4*>(ex_lds + wave * N + l16 * 16 + 4 * lk) = acc;
    __syncthreads();
    const int here = blocks - b0 < waves ? blocks - b0 : waves;
#pragma unroll
    for (int m = 0; m < N / 64; ++m) {
      const int e = tid + m * (waves << 6);
      if (e < N)
        for (int w = 0; w < here; ++w) total[m] += ex_lds[w * N + e];
    }
  }
#pragma unroll
  for (int m = 0; m < N / 64; ++m) {
    const int e = tid + m * (waves << 6);
    const int r = row0 + (e >> 4), c = col0 + (e & 15);
    if (e < N && r < n_rows && c < n_out) {
      float* dst = out + (long)r * ldo + c;
      float v = total[m];
      if (bias) v += bias[c];
      *dst = v = ex_epilogue<EPI>(v, EPI == EPI_RESIDUAL ? *dst : 0.f);
      if (EPI == EPI_QKV && c >= sc.q_width) {
        if (float* at = ex_page_row(sc, r, c)) *at = v;
      }
    }
  }
}

// Few rows with an output so narrow that workgroups of 16 x 16 outputs leave compute units idle while each brings the whole
// inner size by itself: a workgroup has one block of k, whose sum goes to memory, sums[block][row][column]; whoever reads the
// result next adds the blocks up in order (a LayerNorm: mgpt_layernorm_parts).  A wave has 16 columns and R tiles of 16 rows;
// the rows' slice (R x 16 KB) is shared through LDS, all of a wave's slice of W (16 KB) is on its way at once.  What bounds
// it is what a compute unit takes in, about 50 KB a us.  us with the LayerNorm behind it, rows kernel and LayerNorm / here:
// 1 row 3072 -> 768 12.8 / 8.7, 16 rows 16.7 / 9.0, 64 rows 17.8 / 14.0; 6400 -> 1600 23 / 16, 30 / 17, 56 / 27; 16 rows
// 2048 -> 512 13.0 / 8.1, 768 -> 768 8.7 / 8.1; 1 row 1024 -> 1024 7.7 / 8.2, 512 -> 512 6.5 / 7.5.
template <int R, bool VEC>
__global__ __launch_bounds__(256) void linear_exact_parts_kernel(const float* __restrict__ A, long lda,
                                                                 const float* __restrict__ W, float* __restrict__ sums,
                                                                 int n_rows, int n_out, int k_dim, int row_tiles) {
  constexpr int GROUPS = EX_BLOCK / EX_GROUP;
  extern __shared__ __align__(16) float ex_lds[];    // [16 R][EX_BLOCK], 16-byte pieces XORed with the row's low bits
  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y, row0 = (int)(blockIdx.x % row_tiles) * 16 * R, col0 = ((int)(blockIdx.x / row_tiles) * 4 + wave) * 16;
  const int lc = col0 + l16, kb = b * EX_BLOCK;
  const float* wp = W + (long)(lc < n_out ? lc : n_out - 1) * k_dim;
  ex_f4 ga[4 * R], wf[GROUPS];
#pragma unroll
  for (int p = 0; p < 4 * R; ++p) {                  // a wave a row: 64 pieces
    const int r = row0 + 4 * p + wave;
    ga[p] = ex_load<VEC>(A + (long)(r < n_rows ? r : n_rows - 1) * lda, kb + 4 * lane, k_dim);
  }
#pragma unroll
  for (int u = 0; u < GROUPS; ++u) wf[u] = ex_load<VEC>(wp, kb + u * EX_GROUP + 4 * lk, k_dim);
#pragma unroll
  for (int p = 0; p < 4 * R; ++p) {
    const int r = 4 * p + wave;
    *reinterpret_cast<ex_f4*>(ex_lds + r * EX_BLOCK + ((lane ^ (r & 7)) << 2)) = ga[p];
  }
  __builtin_amdgcn_s_waitcnt(0xc07f);                // lgkmcnt(0): W may still be on its way
  __builtin_amdgcn_s_barrier();
  ex_f4 acc[R];
#pragma unroll
  for (int t = 0; t < R; ++t) acc[t] = (ex_f4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < GROUPS; ++u) {
    ex_f4 af[R];
#pragma unroll
    for (int t = 0; t < R; ++t)
      af[t] = *reinterpret_cast<const ex_f4*>(ex_lds + (16 * t + l16) * EX_BLOCK + (((4 * u + lk) ^ (l16 & 7)) << 2));
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int t = 0; t < R; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[u][e], af[t][e], acc[t], 0, 0, 0);
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int r = row0 + 16 * t + l16;
    if (r < n_rows && col0 + 4 * lk < n_out)         // n_out is a multiple of 4
      *reinterpret_cast<ex_f4*>(sums + ((long)b * n_rows + r) * n_out + col0 + 4 * lk) = acc[t];
  }
}

struct ExactArgs {
  const float* A; long lda; const float* W; const float* bias; float* out; long ldo;
  int n_rows, n_out, k_dim;
  ExactScatter sc;
};

template <int T, int EPI, bool VEC, int STAGES>
static int launch_tile(const ExactArgs& a, hipStream_t stream) {
  constexpr int B = 32 * T, bytes = (STAGES > 0 ? STAGES : 2) * 2 * B * EX_BK * (int)sizeof(float);
  static_assert(bytes <= 64 * 1024, "what a kernel gets without asking");
  const int row_tiles = (a.n_rows + B - 1) / B, col_tiles = (a.n_out + B - 1) / B;
  if ((long)row_tiles * col_tiles > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;
  uintptr_t stored = reinterpret_cast<uintptr_t>(a.out) | reinterpret_cast<uintptr_t>(a.bias);
  if (EPI == EPI_QKV) stored |= reinterpret_cast<uintptr_t>(a.sc.kpool) | reinterpret_cast<uintptr_t>(a.sc.vpool);
  const int vec_out = a.ldo % 4 == 0 && (stored & 15) == 0 &&
                      (EPI != EPI_QKV || (a.sc.q_width % 4 == 0 && a.sc.head_dim % 4 == 0));
  hipLaunchKernelGGL((linear_exact_tile_kernel<T, EPI, VEC, STAGES>), dim3(row_tiles * col_tiles), dim3(256), bytes, stream, a.A, a.lda,
                     a.W, a.bias, a.out, a.ldo, a.n_rows, a.n_out, a.k_dim, row_tiles, vec_out,
                     a.sc);
  return mgpt_last_error();
}

template <int EPI, bool VEC>
static int launch_rows(const ExactArgs& a, hipStream_t stream) {
  const int row_tiles = (a.n_rows + 15) / 16, col_tiles = (a.n_out + 15) / 16;
  if ((long)row_tiles * col_tiles > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;
  const int blocks = (a.k_dim + EX_BLOCK - 1) / EX_BLOCK;
  const int rounds = (blocks + 15) / 16, waves = (blocks + rounds - 1) / rounds;
#define EX_ROWS_LAUNCH(SHORT)                                                                                              \
  hipLaunchKernelGGL((linear_exact_rows_kernel<EPI, VEC, SHORT>), dim3(row_tiles * col_tiles), dim3(64 * waves),          \
                     waves * 256 * (int)sizeof(float), stream, a.A, a.lda, a.W, a.bias, a.out, a.ldo, a.n_rows, a.n_out, \
                     a.k_dim, row_tiles, a.sc)
  if (a.k_dim <= 192) EX_ROWS_LAUNCH(true);
  else EX_ROWS_LAUNCH(false);
#undef EX_ROWS_LAUNCH
  return mgpt_last_error();
}

enum { EX_ROWS, EX_TILE64, EX_TILE128, EX_LDS32, EX_LDS64, EX_LDS128 };   // the last three: slices straight into LDS

// The kernel that takes least by what was measured (us; a call's fixed part is the same for all): the rows kernel by its
// rate, 34 TFLOP/s against these tiles, whose calls cost 2 us more; a tile kernel by the rounds of 256 workgroups that it needs, a
// round of 64 x 64 tiles 0.019 us a k (0.0225 alone on a compute unit), of 128 x 128 tiles 0.068.  Rows kernel / 64 / 128, us: 64 rows
// 768 -> 2304 12.1 / 22 / 60; 256 rows 32.9 / 23.3 / 61; 1,100 rows 116 / 48.7 / 63; 256 rows 3072 -> 768 41 / 78 / 223; 1,100 rows
// 512 -> 50304 1525 / 536 / 512.  The 64 x 64 FMA tiles that these kernels replace reached 10 to 15 TFLOP/s (1,100 rows
// 2048 -> 512: 163 us, here 54), the FMA kernel for few rows took 57 us for 16 rows 3072 -> 768 (here 14).
static int rows_or_tiles(int n_rows, int n_out, int k_dim) {
  if ((long)n_rows * n_out <= 380000) return EX_ROWS;   // less than one round of either tile (and no divisions on the host)
  const double k = k_dim, rows = 2.0 * n_rows * n_out * k / 34e6;
  auto rounds = [&](int b) {
    const long tiles = (long)((n_rows + b - 1) / b) * ((n_out + b - 1) / b);
    return (double)((tiles + 255) / 256);
  };
  const double r64 = rounds(64), t64 = r64 > 1 ? r64 * 0.019 * k : 0.0225 * k, t128 = rounds(128) * 0.068 * k;
  if (rows <= t64 && rows <= t128) return EX_ROWS;
  return t64 <= t128 ? EX_TILE64 : EX_TILE128;
}

// Whether tiles of 32 x 32 take the place of the kernel above (inner sizes of whole steps, aligned operands): several of their
// workgroups share a compute unit, so few tiles spread over the chip evenly.  us a k with one, two, three and n of them on a
// compute unit 0.010, 0.014, 0.019, 0.0065 n; the rows kernel at 29 TFLOP/s, a call of either costing the same.  Rows kernel or
// 64 x 64 tiles / here, us: 100 rows 768 -> 2304 15.7 / 13.8; 300 rows 768 -> 768 15.7 / 10.5, 3072 -> 768 51.9 / 33.6; 600 rows
// 512 -> 512 13.9 / 9.9, 5120 -> 1280 107 / 97; 1,201 rows 2048 -> 512 45.3 / 40.8; 400 rows 512 -> 2048 14.8 / 17.6 (not taken).
static bool small_tiles(int n_rows, int n_out, int k_dim) {
  if ((long)n_rows * n_out <= 145000) return false;   // the rows kernel takes less than one round of these
  const double k = k_dim, rows = 2.0 * n_rows * n_out * k / 29e6;
  auto per_unit = [&](int b) {
    const long tiles = (long)((n_rows + b - 1) / b) * ((n_out + b - 1) / b);
    return (double)((tiles + 255) / 256);
  };
  const double r64 = per_unit(64), t64 = r64 > 1 ? r64 * 0.019 * k : 0.0225 * k, t128 = per_unit(128) * 0.068 * k;
  const double n32 = per_unit(32), t32 = k * (n32 <= 1 ? 0.010 : n32 <= 2 ? 0.014 : n32 <= 3 ? 0.019 : 0.0065 * n32);
  return t32 < rows && t32 < t64 && t32 < t128;
}

// The kernel for a product; aligned: rows of both operands start 16 bytes apart at least, as loads straight into LDS want them
// beside an inner size of whole steps.  Tiles whose slices go straight into LDS come two to a compute unit (64 KB each), through
// registers up to five of 64 x 64.  So 64 x 64 tiles stay with the registers for short inner sizes where the chip has more than two
// each (7,000 rows 64 -> 3000 38.6 us, straight into LDS 46.0; 4,400 rows 128 -> 3000 41.4 / 44.2; 1,500 rows 96 -> 2000 11.5 / 12.1)
// and where there is one part round more (700 rows 256 -> 3000, 517 tiles, 19.8 / 20.6); 128 x 128 tiles where a second round is half
// full: its workgroups come two to a unit then, on the units that end first (4,000 rows 768 -> 3072, 768 tiles, 170 / 202; 3,800 rows
// 640 -> 3072 142 / 168; 7,000 rows 384 -> 1500 92 / 109; from inner sizes of about 1,152 on the units end far enough apart: 3,800 rows
// 1152 -> 3072 243 / 239, 1280 -> 3840 270 / 257).
static int exact_kernel(int n_rows, int n_out, int k_dim, bool aligned) {
  const int kernel = rows_or_tiles(n_rows, n_out, k_dim);
  if (!aligned || k_dim % EX_BK != 0) return kernel;
  if (small_tiles(n_rows, n_out, k_dim)) return EX_LDS32;
  if (kernel == EX_ROWS) return kernel;
  const int b = kernel == EX_TILE64 ? 64 : 128;
  const long tiles = (long)((n_rows + b - 1) / b) * ((n_out + b - 1) / b);
  if (kernel == EX_TILE64)
    return tiles > 512 && (k_dim <= 96 || (k_dim <= 384 && tiles <= 768) || (k_dim < 224 && tiles > 2048)) ? EX_TILE64 : EX_LDS64;
  return tiles > 640 && tiles <= 768 && k_dim >= 160 && k_dim < 1152 ? EX_TILE128 : EX_LDS128;
}

extern "C" int mgpt_linear_exact_kernel(int n_rows, int n_out, int k_dim, int aligned) {
  return exact_kernel(n_rows, n_out, k_dim, aligned != 0);
}

template <int EPI, bool VEC>
static int launch_kernel(const ExactArgs& a, int kernel, hipStream_t stream) {
  if constexpr (VEC) {
    if (kernel == EX_LDS32) return launch_tile<1, EPI, true, 6>(a, stream);
    if (kernel == EX_LDS64) return launch_tile<2, EPI, true, 4>(a, stream);
    if (kernel == EX_LDS128) return launch_tile<4, EPI, true, 2>(a, stream);
  }
  if (kernel == EX_ROWS) return launch_rows<EPI, VEC>(a, stream);
  return kernel == EX_TILE64 ? launch_tile<2, EPI, VEC, 0>(a, stream) : launch_tile<4, EPI, VEC, 0>(a, stream);
}

int mgpt_linear_exact_launch(const float* A, long lda, const float* W, const float* bias, float* out, long ldo, int n_rows,
                             int n_out, int k_dim, int epi, const ExactScatter& sc, hipStream_t stream) {
  const ExactArgs a = {A, lda, W, bias, out, ldo, n_rows, n_out, k_dim, sc};
  const bool vec = k_dim % 4 == 0 && lda % 4 == 0 && ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15) == 0;
  const int kernel = exact_kernel(n_rows, n_out, k_dim, vec);
#define EX_LAUNCH(E) return vec ? launch_kernel<E, true>(a, kernel, stream) : launch_kernel<E, false>(a, kernel, stream)
  if (epi == EPI_NONE) EX_LAUNCH(EPI_NONE);
  if (epi == EPI_GELU) EX_LAUNCH(EPI_GELU);
  if (epi == EPI_RELU2) EX_LAUNCH(EPI_RELU2);
  if (epi == EPI_RESIDUAL) EX_LAUNCH(EPI_RESIDUAL);
  if (epi == EPI_QKV && sc.kpool && sc.vpool && sc.slot_mapping) EX_LAUNCH(EPI_QKV);   // a plain product has no pages
#undef EX_LAUNCH
  return MGPT_ERR_BAD_SHAPE;
}

// The product whose key and value columns (kv_width each, behind q_width columns of queries) also go to the pools at
// slot_mapping[row] (a negative one: nowhere), [num_pages][kv_width / head_dim][page_size][head_dim].  The separate kernel
// that copied them took 4.6 us a layer of a decode step, which is what a kernel costs there.
extern "C" int mgpt_linear_exact_qkv(const float* A, long lda, const float* W, const float* bias, float* out, long ldo,
                                     int n_rows, int n_out, int k_dim, float* kpool, float* vpool, const int* slot_mapping,
                                     int q_width, int kv_width, int head_dim, int page_size, hipStream_t stream) {
  if (n_rows == 0 || n_out == 0) return MGPT_OK;
  if (!A || !W || !out || !kpool || !vpool || !slot_mapping) return MGPT_ERR_NULL;
  if (n_rows < 0 || n_out < 0 || k_dim <= 0 || lda < k_dim || ldo < n_out || q_width < 0 || head_dim <= 0 || page_size <= 0 ||
      kv_width <= 0 || kv_width % head_dim != 0 || q_width + 2 * kv_width != n_out)
    return MGPT_ERR_BAD_SHAPE;
  const ExactScatter sc = {kpool, vpool, slot_mapping, q_width, kv_width, head_dim, page_size};
  return mgpt_linear_exact_launch(A, lda, W, bias, out, ldo, n_rows, n_out, k_dim, EPI_QKV, sc, stream);
}

// sums[b][n][o] = the sum over block b (256 k) of A[n] W[o], dense float32 with n_out a multiple of 4, 16-byte aligned: what
// the product above adds up in the order of b, then the bias.
extern "C" int mgpt_linear_exact_parts(const float* A, long lda, const float* W, float* sums, int n_rows, int n_out, int k_dim,
                                       hipStream_t stream) {
  if (n_rows == 0 || n_out == 0) return MGPT_OK;
  if (!A || !W || !sums) return MGPT_ERR_NULL;
  if (n_rows < 0 || n_out < 0 || k_dim <= 0 || lda < k_dim || n_out % 4 != 0 || (reinterpret_cast<uintptr_t>(sums) & 15) != 0)
    return MGPT_ERR_BAD_SHAPE;
  const bool vec = k_dim % 4 == 0 && lda % 4 == 0 && ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(W)) & 15) == 0;
  // one tile of rows a workgroup while there is a compute unit for each (17 rows 3072 -> 768, 288 of them: 11.5 us, in
  // workgroups of two 10.2; 64 rows 2048 -> 512, 256 of them: 10.1 / 10.7), else two (four: 10 % less to 30 % more)
  const long ones = (((long)n_rows + 15) / 16) * (((long)n_out + 63) / 64) * (((long)k_dim + EX_BLOCK - 1) / EX_BLOCK);
  const int r16 = n_rows <= 16 || ones <= 256 ? 1 : 2;
  const long row_tiles = ((long)n_rows + 16 * r16 - 1) / (16 * r16), tiles = row_tiles * (((long)n_out + 63) / 64);
  const int blocks = (int)(((long)k_dim + EX_BLOCK - 1) / EX_BLOCK);
  if (tiles > 0x7fffffffL || blocks > 65535) return MGPT_ERR_TOO_LARGE;
#define EX_PARTS_LAUNCH(R, V)                                                                                                  \
  hipLaunchKernelGGL((linear_exact_parts_kernel<R, V>), dim3((unsigned int)tiles, blocks), dim3(256), R * 16 * EX_BLOCK * 4, \
                     stream, A, lda, W, sums, n_rows, n_out, k_dim, (int)row_tiles)
  if (r16 == 1) { if (vec) EX_PARTS_LAUNCH(1, true); else EX_PARTS_LAUNCH(1, false); }
  else { if (vec) EX_PARTS_LAUNCH(2, true); else EX_PARTS_LAUNCH(2, false); }
#undef EX_PARTS_LAUNCH
  return mgpt_last_error();
}
