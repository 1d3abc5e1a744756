// Token embedding (+ learned position rows) into the 32-bit residual stream,
// and LayerNorm with 32-bit statistics.
//
// embedding: x0[t] = tok_emb[id_t] + pos_emb[pos_t]   (reference: src/minigpt_infer/model.py:183)
// LayerNorm: y = (x - mean) / sqrt(var_biased + eps) * w (+ b) over the last dim
//            (reference: nn.LayerNorm at src/minigpt_infer/model.py:107,109,127)
#include "common.h"
#include "layernorm_sums.h"
#include "launchers.h"

template <typename WT>
__global__ void embed_kernel(const int* __restrict__ ids, const int* __restrict__ pos,
                             const WT* __restrict__ tok, const WT* __restrict__ postab,
                             float* __restrict__ x, int n_tokens, int width) {
  int n = blockIdx.x;
  if (n >= n_tokens) return;
  long id = ids[n];
  const WT* trow = tok + id * (long)width;
  const WT* prow = postab ? postab + (long)pos[n] * width : nullptr;
  float* xr = x + (long)n * width;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    float v = to_float<WT>(trow[c]);
    if (prow) v += to_float<WT>(prow[c]);
    xr[c] = v;
  }
}

extern "C" int mgpt_embed(const int* ids, const int* pos, const void* tok, const void* postab,
                          float* x, int n_tokens, int width, int table_dtype, hipStream_t stream) {
  if (n_tokens == 0) return MGPT_OK;
  if (!ids || !tok || !x || (postab && !pos)) return MGPT_ERR_NULL;
  if (n_tokens < 0 || width <= 0) return MGPT_ERR_BAD_SHAPE;
  int threads = width >= 256 ? 256 : 64;
  if (table_dtype == MGPT_F32) {
    hipLaunchKernelGGL(embed_kernel<float>, dim3(n_tokens), dim3(threads), 0, stream, ids, pos,
                       (const float*)tok, (const float*)postab, x, n_tokens, width);
  } else if (table_dtype == MGPT_BF16) {
    hipLaunchKernelGGL(embed_kernel<bf16_t>, dim3(n_tokens), dim3(threads), 0, stream, ids, pos,
                       (const bf16_t*)tok, (const bf16_t*)postab, x, n_tokens, width);
  } else {
    return MGPT_ERR_BAD_DTYPE;
  }
  return mgpt_last_error();
}

// One wave per row; four rows per workgroup.  A row of up to 64 * LN_CACHE values is read once
// and kept in registers.  First the mean; then, together, the centred sum of squares and what
// the mean lost to rounding (kept apart: the mean is a sum of two floats), so the variance is
// never a difference of large numbers and a row of nearly equal values far from zero stays exact.
// Wider rows take the same steps with the row re-read from cache.
#define LN_CACHE 16

template <typename OT>
__global__ void layernorm_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                 const float* __restrict__ b, OT* __restrict__ out,
                                 const int* __restrict__ rows, int n_rows, int width, float eps) {
  int lane = threadIdx.x & (MGPT_WAVE - 1);
  int row = blockIdx.x * (blockDim.x / MGPT_WAVE) + (threadIdx.x / MGPT_WAVE);
  if (row >= n_rows) return;
  long src = rows ? rows[row] : row;
  const float* xr = x + src * (long)width;
  OT* orow = out + (long)row * width;
  if (width <= MGPT_WAVE * LN_CACHE) {
    // the row, the gain and the bias are all asked for before anything is waited for
    float xv[LN_CACHE], gv[LN_CACHE], bv[LN_CACHE];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < LN_CACHE; ++i) {
      const int c = lane + i * MGPT_WAVE;
      const int cc = c < width ? c : 0;
      xv[i] = xr[cc];
      gv[i] = w[cc];
      bv[i] = b ? b[cc] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < LN_CACHE; ++i) {
      if (lane + i * MGPT_WAVE >= width) xv[i] = 0.f;
      s += xv[i];
    }
    const float mean = wave_sum(s) / (float)width;
    float e = 0.f, v2 = 0.f;
#pragma unroll
    for (int i = 0; i < LN_CACHE; ++i) {
      const float d = (lane + i * MGPT_WAVE < width) ? xv[i] - mean : 0.f;
      xv[i] = d;
      e += d;
      v2 = fmaf(d, d, v2);
    }
    const float corr = wave_sum(e) / (float)width;
    const float var = fmaxf(wave_sum(v2) / (float)width - corr * corr, 0.f);
    const float rstd = 1.0f / sqrtf(var + eps);
#pragma unroll
    for (int i = 0; i < LN_CACHE; ++i) {
      const int c = lane + i * MGPT_WAVE;
      if (c < width) orow[c] = from_float<OT>((xv[i] - corr) * rstd * gv[i] + bv[i]);
    }
    return;
  }
  float s = 0.f;
  for (int c = lane; c < width; c += MGPT_WAVE) s += xr[c];
  const float mean = wave_sum(s) / (float)width;
  float e = 0.f, v2 = 0.f;
  for (int c = lane; c < width; c += MGPT_WAVE) {
    const float d = xr[c] - mean;
    e += d;
    v2 = fmaf(d, d, v2);
  }
  const float corr = wave_sum(e) / (float)width;
  const float var = fmaxf(wave_sum(v2) / (float)width - corr * corr, 0.f);
  const float rstd = 1.0f / sqrtf(var + eps);
  for (int c = lane; c < width; c += MGPT_WAVE) {
    float y = ((xr[c] - mean) - corr) * rstd * w[c];
    if (b) y += b[c];
    orow[c] = from_float<OT>(y);
  }
}

// The same for widths that are multiples of 4 up to 64 * 4 * LN_VEC with 16-byte aligned rows: every
// lane loads and stores vectors of four (a row of 512 is two loads per lane instead of eight).
// LN_VEC is the number of such vectors a lane holds: the row's width / 256, rounded up to one of
// 1, 2, 3, 4, 6, 8 (rows up to 2048 wide), so that a row of 512 costs two loads and not four.
template <typename OT, int LN_VEC>
__global__ void layernorm_vec_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                     const float* __restrict__ b, OT* __restrict__ out,
                                     const int* __restrict__ rows, int n_rows, int width, float eps) {
  const int lane = threadIdx.x & (MGPT_WAVE - 1);
  const int row = blockIdx.x * (blockDim.x / MGPT_WAVE) + (threadIdx.x / MGPT_WAVE);
  if (row >= n_rows) return;
  const long src = rows ? rows[row] : row;
  const float4* xr = reinterpret_cast<const float4*>(x + src * (long)width);
  const float4* w4 = reinterpret_cast<const float4*>(w);
  const float4* b4 = reinterpret_cast<const float4*>(b);
  const int n4 = width >> 2;
  float4 xv[LN_VEC], gv[LN_VEC], bv[LN_VEC];
#pragma unroll
  for (int i = 0; i < LN_VEC; ++i) {
    const int c = lane + i * MGPT_WAVE;
    const int cc = c < n4 ? c : 0;
    xv[i] = xr[cc];
    gv[i] = w4[cc];
    bv[i] = b ? b4[cc] : make_float4(0.f, 0.f, 0.f, 0.f);
  }
  float mean, corr, rstd;
  layernorm_sums<LN_VEC, LN_VEC <= 4 ? 1 : 2>(xv, n4, width, eps, mean, corr, rstd);   // (5 and 7 vectors: 6 and 8 here)
  OT* orow = out + (long)row * width;
#pragma unroll
  for (int i = 0; i < LN_VEC; ++i) {
    const int c = lane + i * MGPT_WAVE;
    if (c >= n4) continue;
    const float y0 = (xv[i].x - corr) * rstd * gv[i].x + bv[i].x, y1 = (xv[i].y - corr) * rstd * gv[i].y + bv[i].y;
    const float y2 = (xv[i].z - corr) * rstd * gv[i].z + bv[i].z, y3 = (xv[i].w - corr) * rstd * gv[i].w + bv[i].w;
    if (sizeof(OT) == 4) {
      reinterpret_cast<float4*>(orow)[c] = make_float4(y0, y1, y2, y3);
    } else {
      uint2 pk;
      pk.x = pack_bf16x2(y0, y1);
      pk.y = pack_bf16x2(y2, y3);
      reinterpret_cast<uint2*>(orow)[c] = pk;
    }
  }
}

// The same for rows of 513 to 2,048 values where the rows are few: a workgroup a row, a vector of four a lane, W waves.  One
// wave a row has three to eight vectors a lane there, and their loads, sums and stores one behind the other.  The waves hand
// each other the row through LDS and each makes all of its sums, in the order of the kernel above: a row's result is the same
// bits in both, and so whatever the number of rows.  With many rows there are waves enough, and eight waves that make one
// row's sums eight times only cost.  us in a graph of such calls, a wave a row / here: bfloat16 outputs, 16 rows of 768
// 2.43 / 1.95, of 1,600 3.30 / 2.42, of 2,048 3.45 / 2.47; 200 rows of 1,600 3.41 / 2.61; 640 rows of 768 2.58 / 2.55;
// with masks on all vectors 640 rows of 1,600 3.57 / 4.30.  The line between them, 1,920 waves (two a SIMD, nearly), lies
// where the two meet: 640 rows of 768, 274 of 1,600, 240 of 2,048.  (Waves that each sum a part of the row and meet in LDS
// took 2.25 us for 16 rows of 1,600, but in an order of their own, which the 32-bit path then had to keep to with many rows
// as well: 4,096 rows of 768 took 6.2 us for 5.3.)
template <typename OT, int W>
__global__ __launch_bounds__(64 * W) void layernorm_shared_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                  const float* __restrict__ b, OT* __restrict__ out,
                                                                  const int* __restrict__ rows, int width, float eps) {
  __shared__ float4 row_s[64 * W];
  const int tid = threadIdx.x, lane = tid & (MGPT_WAVE - 1), n4 = width >> 2;
  const long src = rows ? rows[blockIdx.x] : (long)blockIdx.x;
  const int c = tid < n4 ? tid : 0;
  const float4 v = reinterpret_cast<const float4*>(x + src * (long)width)[c];
  const float4 g = reinterpret_cast<const float4*>(w)[c];
  const float4 o = b ? reinterpret_cast<const float4*>(b)[c] : make_float4(0.f, 0.f, 0.f, 0.f);
  row_s[tid] = v;
  __syncthreads();
  float4 xv[W];
#pragma unroll
  for (int i = 0; i < W; ++i) xv[i] = row_s[lane + i * MGPT_WAVE];
  float mean, corr, rstd;
  layernorm_sums<W, 1>(xv, n4, width, eps, mean, corr, rstd);
  if (tid >= n4) return;
  const float y0 = ((v.x - mean) - corr) * rstd * g.x + o.x, y1 = ((v.y - mean) - corr) * rstd * g.y + o.y;
  const float y2 = ((v.z - mean) - corr) * rstd * g.z + o.z, y3 = ((v.w - mean) - corr) * rstd * g.w + o.w;
  OT* orow = out + (long)blockIdx.x * width;
  if (sizeof(OT) == 4) reinterpret_cast<float4*>(orow)[tid] = make_float4(y0, y1, y2, y3);
  else reinterpret_cast<uint2*>(orow)[tid] = make_uint2(pack_bf16x2(y0, y1), pack_bf16x2(y2, y3));
}

// The kernel above for float32 rows that a product has left as sums over its blocks of k (linear_exact.hip): first
// x += ((sums[0] + sums[1]) + ...) + bias, in the order in which that product adds them up itself, so the same bits; the row
// goes back to `settled` if there is one (the rows' own place: nobody else reads them).  Without a gain that is all.
template <int W>
__global__ __launch_bounds__(64 * W) void layernorm_parts_kernel(const float* __restrict__ x, const float* __restrict__ sums,
                                                                 int n_parts, long part_stride, const float* __restrict__ add,
                                                                 const float* __restrict__ w, const float* __restrict__ b,
                                                                 float* __restrict__ out, const int* __restrict__ rows,
                                                                 int width, float eps, float* settled) {
  constexpr int AT_ONCE = 16;                       // sums on their way
  __shared__ float4 row_s[64 * W];
  const int tid = threadIdx.x, lane = tid & (MGPT_WAVE - 1), n4 = width >> 2;
  const long src = rows ? rows[blockIdx.x] : (long)blockIdx.x;
  const int c = tid < n4 ? tid : 0;
  const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
  const float4* part = reinterpret_cast<const float4*>(sums + src * (long)width) + c;
  float4 v = reinterpret_cast<const float4*>(x + src * (long)width)[c];
  const float4 more = add ? reinterpret_cast<const float4*>(add)[c] : zero;
  const float4 g = w ? reinterpret_cast<const float4*>(w)[c] : zero;
  const float4 o = b ? reinterpret_cast<const float4*>(b)[c] : zero;
  float4 total = zero;
  for (int p0 = 0; p0 < n_parts; p0 += AT_ONCE) {
    float4 t[AT_ONCE];
#pragma unroll
    for (int p = 0; p < AT_ONCE; ++p) t[p] = part[(p0 + p < n_parts ? p0 + p : p0) * (part_stride >> 2)];
#pragma unroll
    for (int p = 0; p < AT_ONCE; ++p)
      if (p0 + p < n_parts) {
        total.x += t[p].x; total.y += t[p].y; total.z += t[p].z; total.w += t[p].w;
      }
  }
  if (add) {
    total.x += more.x; total.y += more.y; total.z += more.z; total.w += more.w;
  }
  v.x += total.x; v.y += total.y; v.z += total.z; v.w += total.w;
  if (settled && tid < n4) reinterpret_cast<float4*>(settled + src * (long)width)[tid] = v;
  if (!w) return;
  row_s[tid] = v;
  __syncthreads();
  float4 xv[W];
#pragma unroll
  for (int i = 0; i < W; ++i) xv[i] = row_s[lane + i * MGPT_WAVE];
  float mean, corr, rstd;
  layernorm_sums<W, 1>(xv, n4, width, eps, mean, corr, rstd);
  if (tid >= n4) return;
  const float y0 = ((v.x - mean) - corr) * rstd * g.x + o.x, y1 = ((v.y - mean) - corr) * rstd * g.y + o.y;
  const float y2 = ((v.z - mean) - corr) * rstd * g.z + o.z, y3 = ((v.w - mean) - corr) * rstd * g.w + o.w;
  reinterpret_cast<float4*>(out + (long)blockIdx.x * width)[tid] = make_float4(y0, y1, y2, y3);
}

// Rows of 2,049 to 4,096 values: 16 waves a row, whose sums meet in LDS (16 rows of 4,096 with the 4-byte loads of the first
// kernel above 29 us, here 2.9; 4,096 rows 74 / 24).
template <typename OT>
__global__ __launch_bounds__(1024) void layernorm_row_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                             const float* __restrict__ b, OT* __restrict__ out,
                                                             const int* __restrict__ rows, int width, float eps) {
  constexpr int W = 16;
  __shared__ float red[W][2], red_sum[W];
  const int tid = threadIdx.x, wave = tid >> 6;
  const long src = rows ? rows[blockIdx.x] : (long)blockIdx.x;
  const bool in = 4 * tid < width;
  const int c = in ? tid : 0;
  float4 v = reinterpret_cast<const float4*>(x + src * (long)width)[c];
  const float4 g = reinterpret_cast<const float4*>(w)[c];
  const float4 o = b ? reinterpret_cast<const float4*>(b)[c] : make_float4(0.f, 0.f, 0.f, 0.f);
  const float s = wave_sum(in ? (v.x + v.y) + (v.z + v.w) : 0.f);
  if ((tid & 63) == 0) red_sum[wave] = s;
  __syncthreads();
  float mean = 0.f;
#pragma unroll
  for (int i = 0; i < W; ++i) mean += red_sum[i];
  mean /= (float)width;
  v.x -= mean; v.y -= mean; v.z -= mean; v.w -= mean;
  const float e = wave_sum(in ? (v.x + v.y) + (v.z + v.w) : 0.f);
  const float q = wave_sum(in ? fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))) : 0.f);
  if ((tid & 63) == 0) {
    red[wave][0] = e;
    red[wave][1] = q;
  }
  __syncthreads();
  float corr = 0.f, var = 0.f;
#pragma unroll
  for (int i = 0; i < W; ++i) {
    corr += red[i][0];
    var += red[i][1];
  }
  corr /= (float)width;
  const float rstd = 1.0f / sqrtf(fmaxf(var / (float)width - corr * corr, 0.f) + eps);
  if (!in) return;
  const float y0 = (v.x - corr) * rstd * g.x + o.x, y1 = (v.y - corr) * rstd * g.y + o.y;
  const float y2 = (v.z - corr) * rstd * g.z + o.z, y3 = (v.w - corr) * rstd * g.w + o.w;
  OT* orow = out + (long)blockIdx.x * width;
  if (sizeof(OT) == 4) reinterpret_cast<float4*>(orow)[tid] = make_float4(y0, y1, y2, y3);
  else reinterpret_cast<uint2*>(orow)[tid] = make_uint2(pack_bf16x2(y0, y1), pack_bf16x2(y2, y3));
}

// rows: optional gather list (n_rows entries) of source rows of x; out row i <- x row rows[i].
extern "C" int mgpt_layernorm(const float* x, const float* w, const float* b, void* out,
                              const int* rows, int n_rows, int width, float eps, int out_dtype,
                              hipStream_t stream) {
  if (n_rows == 0) return MGPT_OK;
  if (!x || !w || !out) return MGPT_ERR_NULL;
  if (n_rows < 0 || width <= 0) return MGPT_ERR_BAD_SHAPE;
  const int rows_per_block = 4;
  dim3 grid((n_rows + rows_per_block - 1) / rows_per_block), block(rows_per_block * MGPT_WAVE);
  const bool vec = (width % 4) == 0 && width <= 4096 &&
                   ((((size_t)x) | ((size_t)w) | ((size_t)b) | ((size_t)out)) & 15) == 0;
  const int need = (width / 4 + MGPT_WAVE - 1) / MGPT_WAVE;   // vectors of four per lane of one wave
#define LN_LAUNCH(OT, V) \
  hipLaunchKernelGGL((layernorm_vec_kernel<OT, V>), grid, block, 0, stream, x, w, b, (OT*)out, rows, n_rows, width, eps)
#define LN_SHARED(OT, W)                                                                                                 \
  hipLaunchKernelGGL((layernorm_shared_kernel<OT, W>), dim3(n_rows), dim3(64 * W), 0, stream, x, w, b, (OT*)out, rows, \
                     width, eps)
#define LN_PICK(OT)                                                                                                  \
  if (need <= 1) LN_LAUNCH(OT, 1);                                                                                   \
  else if (need <= 2) LN_LAUNCH(OT, 2);                                                                              \
  else if (need > 8)                                                                                                 \
    hipLaunchKernelGGL((layernorm_row_kernel<OT>), dim3(n_rows), dim3(1024), 0, stream, x, w, b, (OT*)out, rows, width,     \
                       eps);                                                                                         \
  else if ((long)n_rows * need <= 1920) {                                                                            \
    if (need <= 3) LN_SHARED(OT, 3);                                                                                 \
    else if (need <= 4) LN_SHARED(OT, 4);                                                                            \
    else if (need <= 5) LN_SHARED(OT, 5);                                                                            \
    else if (need <= 6) LN_SHARED(OT, 6);                                                                            \
    else if (need <= 7) LN_SHARED(OT, 7);                                                                            \
    else LN_SHARED(OT, 8);                                                                                           \
  } else if (need <= 3) LN_LAUNCH(OT, 3);                                                                            \
  else if (need <= 4) LN_LAUNCH(OT, 4);                                                                              \
  else if (need <= 6) LN_LAUNCH(OT, 6);                                                                              \
  else LN_LAUNCH(OT, 8)
  if (vec && out_dtype == MGPT_F32) {
    LN_PICK(float);
  } else if (vec && out_dtype == MGPT_BF16) {
    LN_PICK(bf16_t);
#undef LN_PICK
#undef LN_SHARED
#undef LN_LAUNCH
  } else if (out_dtype == MGPT_F32) {
    hipLaunchKernelGGL(layernorm_kernel<float>, grid, block, 0, stream, x, w, b, (float*)out, rows,
                       n_rows, width, eps);
  } else if (out_dtype == MGPT_BF16) {
    hipLaunchKernelGGL(layernorm_kernel<bf16_t>, grid, block, 0, stream, x, w, b, (bf16_t*)out,
                       rows, n_rows, width, eps);
  } else {
    return MGPT_ERR_BAD_DTYPE;
  }
  return mgpt_last_error();
}

// Rows left as sums over blocks by mgpt_linear_exact_parts (part_stride floats apart): out row i = LayerNorm of row rows[i] (or
// i) of x + the sums in order + add (null: none), and with `settled` (x itself, or rows of the same kind) that sum as well;
// w null: nothing but the sum.  Widths that are multiples of 4 up to 2,048, everything 16-byte aligned.
extern "C" int mgpt_layernorm_parts(const float* x, const float* sums, int n_parts, long part_stride, const float* add,
                                    const float* w, const float* b, float* out, const int* rows, int n_rows, int width,
                                    float eps, float* settled, hipStream_t stream) {
  if (n_rows == 0) return MGPT_OK;
  if (!x || !sums || (w ? !out : !settled)) return MGPT_ERR_NULL;
  const size_t together = (size_t)x | (size_t)sums | (size_t)add | (size_t)w | (size_t)b | (size_t)out | (size_t)settled;
  if (n_rows < 0 || n_parts <= 0 || width <= 0 || width % 4 != 0 || width > 2048 || part_stride % 4 != 0 || (together & 15) != 0 ||
      (rows && settled))
    return MGPT_ERR_BAD_SHAPE;
#define LP_LAUNCH(V)                                                                                                       \
  case V:                                                                                                                  \
    hipLaunchKernelGGL(layernorm_parts_kernel<V>, dim3(n_rows), dim3(64 * V), 0, stream, x, sums, n_parts, part_stride, add, w, \
                       b, out, rows, width, eps, settled);                                                                 \
    break
  switch ((width / 4 + MGPT_WAVE - 1) / MGPT_WAVE) {
    LP_LAUNCH(1); LP_LAUNCH(2); LP_LAUNCH(3); LP_LAUNCH(4); LP_LAUNCH(5); LP_LAUNCH(6); LP_LAUNCH(7); LP_LAUNCH(8);
  }
#undef LP_LAUNCH
  return mgpt_last_error();
}
