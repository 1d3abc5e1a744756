// Token embedding (+ learned position rows) into the 32-bit residual stream,
// and LayerNorm with 32-bit statistics.
//
// embedding: x0[t] = tok_emb[id_t] + pos_emb[pos_t]   (reference: src/minigpt_infer/model.py:183)
// LayerNorm: y = (x - mean) / sqrt(var_biased + eps) * w (+ b) over the last dim
//            (reference: nn.LayerNorm at src/minigpt_infer/model.py:107,109,127)
#include "common.h"
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
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < LN_VEC; ++i) {
    if (lane + i * MGPT_WAVE >= n4) xv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    s += (xv[i].x + xv[i].y) + (xv[i].z + xv[i].w);
  }
  const float mean = wave_sum(s) / (float)width;
  float e = 0.f, v2 = 0.f;
#pragma unroll
  for (int i = 0; i < LN_VEC; ++i) {
    const bool in = lane + i * MGPT_WAVE < n4;
    float* p = reinterpret_cast<float*>(&xv[i]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float d = in ? p[k] - mean : 0.f;
      p[k] = d;
      e += d;
      v2 = fmaf(d, d, v2);
    }
  }
  const float corr = wave_sum(e) / (float)width;
  const float var = fmaxf(wave_sum(v2) / (float)width - corr * corr, 0.f);
  const float rstd = 1.0f / sqrtf(var + eps);
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

// The same for rows of 513 to 4,096 values (multiples of 4, 16-byte aligned): a workgroup a row with a vector of four a lane, W
// waves, whose sums meet in LDS.  One wave a row has three to eight vectors a lane there, and their loads, sums and stores
// one behind the other (us in a graph of such calls, a wave a row / here: 32 rows of 768 2.87 / 2.49, of 1,600 3.70 / 2.71; of
// 4,096, which had 4-byte loads, 29.5 / 3.3; 512 rows of 1,600 3.97 / 3.47).  With many rows there are waves enough and the
// meeting only costs (1,024 rows of 1,600 4.23 / 4.50): bfloat16 outputs of more than 640 rows of up to 2,048 stay with the
// kernel above.  Float32 outputs, the 32-bit path's, always come here where it takes the row (4,096 rows of 768 5.6 / 6.6, beside
// products of hundreds): their sums run in one order whatever the number of rows.
template <typename OT, int W>
__global__ __launch_bounds__(64 * W) void layernorm_row_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                               const float* __restrict__ b, OT* __restrict__ out,
                                                               const int* __restrict__ rows, int width, float eps) {
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
#define LN_ROW(OT, W) \
  hipLaunchKernelGGL((layernorm_row_kernel<OT, W>), dim3(n_rows), dim3(64 * W), 0, stream, x, w, b, (OT*)out, rows, width, eps)
#define LN_PICK_WAVE(OT)                \
  if (need <= 3) LN_LAUNCH(OT, 3);      \
  else if (need <= 4) LN_LAUNCH(OT, 4); \
  else if (need <= 6) LN_LAUNCH(OT, 6); \
  else LN_LAUNCH(OT, 8)
#define LN_PICK_ROW(OT)               \
  if (need <= 3) LN_ROW(OT, 3);       \
  else if (need <= 4) LN_ROW(OT, 4);  \
  else if (need <= 5) LN_ROW(OT, 5);  \
  else if (need <= 6) LN_ROW(OT, 6);  \
  else if (need <= 7) LN_ROW(OT, 7);  \
  else if (need <= 8) LN_ROW(OT, 8);  \
  else LN_ROW(OT, 16)
  if (vec && out_dtype == MGPT_F32) {
    if (need <= 1) LN_LAUNCH(float, 1);
    else if (need <= 2) LN_LAUNCH(float, 2);
    else { LN_PICK_ROW(float); }
  } else if (vec && out_dtype == MGPT_BF16) {
    if (need <= 1) LN_LAUNCH(bf16_t, 1);
    else if (need <= 2) LN_LAUNCH(bf16_t, 2);
    else if (n_rows <= 640 || need > 8) { LN_PICK_ROW(bf16_t); }
    else { LN_PICK_WAVE(bf16_t); }
#undef LN_PICK_ROW
#undef LN_PICK_WAVE
#undef LN_ROW
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
