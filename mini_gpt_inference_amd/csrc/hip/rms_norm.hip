// Root-mean-square norms over float32 statistics.
//
//   unit(x) = x / sqrt(mean(x^2) + eps)
//
// rms_norm: out = [out +] mult * unit(x) * (offset + gain) [* act(gate)] (or, with the gate in front of the norm,
// unit(x * silu(gate)) in place of unit(x) and no gate behind), per segment: a row holds
// `groups` segments of `width` values (one for a norm over the row, one per head for a norm per
// head).  gain may be absent (a norm without a weight), offset is 1 for a gain stored as its
// distance from one.  Rows may be gathered (`rows`), and a second buffer may be cleared on the way
// (the buffer the next sublayer adds its output into).
//
// rms_post_norm: the step between two sublayers of a layer whose sublayers are normed on both
// sides, one workgroup a row:
//   y = sum_b coef * unit(y_b) * gain_b          (only with several branches; else y = y_0;
//                                                 join_unit = 0: sum_b coef * y_b * gain_b, a weighted sum)
//   x += mult * unit(y) * (offset + gain_post) (* scale_post, a scale per channel)
//   h = unit(x) * (offset + gain_next)           (if there is a next norm; without its gain, h = x if there is an h)
//   y_b = 0                                       (ready for the next sublayer's additions)
// Sums of squares are taken in float32 in a fixed order (lane-strided, then across the wave, then
// across the waves in order), so a row's result does not depend on the other rows of the step.
#include "common.h"
#include "dtype_io.h"
#include "launchers.h"

#define RMS_ACT_NONE 0
#define RMS_ACT_SILU 1
#define RMS_ACT_SIGMOID 2
#define RMS_ACT_SILU_FIRST 3      // the input is multiplied by silu(gate) before its root mean square is taken

__device__ __forceinline__ float rms_gate_act(float g, int act) {
  if (act == RMS_ACT_SILU) return g / (1.0f + expf(-g));
  if (act == RMS_ACT_SIGMOID) return 1.0f / (1.0f + expf(-g));
  return g;
}

// sum over the workgroup's threads (1, 2 or 4 waves), the same value in every thread; waves are added in order
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  if (blockDim.x == 64) return v;
  const int wave = threadIdx.x >> 6;
  __syncthreads();      // the scratch's readers of the call before are done
  if ((threadIdx.x & 63) == 0) scratch[wave] = v;
  __syncthreads();
  return blockDim.x == 128 ? scratch[0] + scratch[1] : (scratch[0] + scratch[1]) + (scratch[2] + scratch[3]);
}

// one workgroup per segment: a wave for a narrow one (a head), four for a wide one (a row of the model's width).
// PT > 0: a thread keeps its PT values of the segment in registers between the two passes (segments of up to
// PT * threads values), and everything that it reads is on its way before the first sum; PT = 0: the second pass reads them again.
// XT, GT, OT: the types of the input, the gate and the output.  What bounds few rows is the trips to memory: with types chosen at run
// time every value was waited for by itself, and gain and gate came behind the sum.  us in a graph, so / here: 8 rows of 1,024 3.4 / 2.7,
// with a gate 4.2 / 3.1, of 2,048 4.3 / 3.3, of 8,192 16.5 / 11.1; 4,075 rows of 1,024 8.8 / 7.1, of 8 gated heads of 128 14.0 / 11.7.  PT is close to
// the values there are: those beyond the segment's end are loads as well (4,096 rows of 1,280 14.0 / 17.5 with 16, 11.5 with 6).
template <int PT, typename XT, typename GT, typename OT>
__global__ __launch_bounds__(256) void rms_norm_kernel(
    const XT* x, long ldx, const int* __restrict__ rows,      // (out may be x: the norm in place)
    const float* __restrict__ gain, float offset, float eps, float mult, const GT* __restrict__ gate,
    long ldg, int gate_act, OT* out, long ldo, int accumulate,
    float* __restrict__ zero, long ldz, int zero_width, int n_rows, int groups, int x_gstride, int o_gstride,
    int width) {
  __shared__ float scratch[4];
  const long seg = blockIdx.x;
  const int row = (int)(seg / groups), g = (int)(seg - (long)row * groups);
  const int src = rows ? rows[row] : row;
  const long xb = (long)src * ldx + (long)g * x_gstride;
  const int step = blockDim.x;
  const long ob = (long)row * ldo + (long)g * o_gstride;
  const long gb = (long)row * ldg + (long)g * o_gstride;
  const bool gate_first = gate && gate_act == RMS_ACT_SILU_FIRST, gate_last = gate && !gate_first;
  auto finish = [&](int c, float v, float gain_c, float gate_c, float old) {
    if (gain) v *= offset + gain_c;
    if (gate_last) v *= rms_gate_act(gate_c, gate_act);
    if (accumulate) v += old;
    out[ob + c] = from_float<OT>(v);
  };
  float ss = 0.f;
  if constexpr (PT > 0) {
    XT xr[PT];
    GT gr[PT];
    OT old[PT];
    float gn[PT], xv[PT];
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      const int c = (int)threadIdx.x + u * step, cc = c < width ? c : width - 1;
      xr[u] = x[xb + cc];
    }
    if (gate) {
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        const int c = (int)threadIdx.x + u * step;
        gr[u] = gate[gb + (c < width ? c : width - 1)];
      }
    }
    if (gain) {
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        const int c = (int)threadIdx.x + u * step;
        gn[u] = gain[(long)g * width + (c < width ? c : width - 1)];
      }
    }
    if (accumulate) {
#pragma unroll
      for (int u = 0; u < PT; ++u) {
        const int c = (int)threadIdx.x + u * step;
        old[u] = out[ob + (c < width ? c : width - 1)];
      }
    }
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      float v = to_float<XT>(xr[u]);
      if (gate_first) v *= rms_gate_act(to_float<GT>(gr[u]), RMS_ACT_SILU);
      xv[u] = (int)threadIdx.x + u * step < width ? v : 0.f;
    }
#pragma unroll
    for (int u = 0; u < PT; ++u) ss = fmaf(xv[u], xv[u], ss);
    ss = block_sum(ss, scratch);
    const float r = mult / sqrtf(ss / (float)width + eps);
#pragma unroll
    for (int u = 0; u < PT; ++u) {
      const int c = (int)threadIdx.x + u * step;
      if (c < width) finish(c, xv[u] * r, gain ? gn[u] : 0.f, gate_last ? to_float<GT>(gr[u]) : 0.f, accumulate ? to_float<OT>(old[u]) : 0.f);
    }
  } else {
    auto input = [&](int c) {
      float v = to_float<XT>(x[xb + c]);
      if (gate_first) v *= rms_gate_act(to_float<GT>(gate[gb + c]), RMS_ACT_SILU);
      return v;
    };
    for (int c = threadIdx.x; c < width; c += step) {
      const float v = input(c);
      ss = fmaf(v, v, ss);
    }
    ss = block_sum(ss, scratch);
    const float r = mult / sqrtf(ss / (float)width + eps);
    for (int c = threadIdx.x; c < width; c += step)
      finish(c, input(c) * r, gain ? gain[(long)g * width + c] : 0.f, gate_last ? to_float<GT>(gate[gb + c]) : 0.f,
             accumulate ? to_float<OT>(out[ob + c]) : 0.f);
  }
  if (zero && g == 0)
    for (int c = threadIdx.x; c < zero_width; c += step) zero[(long)row * ldz + c] = 0.f;
}

extern "C" int mgpt_rms_norm(const void* x, int x_dtype, long ldx, const int* rows, const float* gain, float offset,
                             float eps, float mult, const void* gate, int gate_dtype, long ldg, int gate_act,
                             void* out, int out_dtype, long ldo, int accumulate, float* zero, long ldz,
                             int zero_width, int n_rows, int groups, int x_gstride, int o_gstride, int width,
                             hipStream_t stream) {
  if (n_rows == 0) return MGPT_OK;
  if (!x || !out) return MGPT_ERR_NULL;
  if (n_rows < 0 || groups <= 0 || width <= 0 || zero_width < 0) return MGPT_ERR_BAD_SHAPE;
  if (!dtype_ok(x_dtype) || !dtype_ok(out_dtype) || (gate && !dtype_ok(gate_dtype))) return MGPT_ERR_BAD_DTYPE;
  const long segs = (long)n_rows * groups;
  if (segs > 0x7fffffffL) return MGPT_ERR_TOO_LARGE;
  const int threads = width <= 256 ? 64 : (width <= 512 ? 128 : 256);
#define RN_LAUNCH(PT, XT, GT, OT)                                                                                  \
  hipLaunchKernelGGL((rms_norm_kernel<PT, XT, GT, OT>), dim3((unsigned)segs), dim3(threads), 0, stream, (const XT*)x, ldx, rows, \
                     gain, offset, eps, mult, (const GT*)gate, ldg, gate_act, (OT*)out, ldo, accumulate, zero, ldz, zero_width,  \
                     n_rows, groups, x_gstride, o_gstride, width)
#define RN_TYPES(PT)                                                                                               \
  do {                                                                                                             \
    if (x_dtype == MGPT_F32) {                                                                                     \
      if (gate_dtype == MGPT_F32) { if (out_dtype == MGPT_F32) RN_LAUNCH(PT, float, float, float); else RN_LAUNCH(PT, float, float, bf16_t); } \
      else { if (out_dtype == MGPT_F32) RN_LAUNCH(PT, float, bf16_t, float); else RN_LAUNCH(PT, float, bf16_t, bf16_t); }       \
    } else {                                                                                                       \
      if (gate_dtype == MGPT_F32) { if (out_dtype == MGPT_F32) RN_LAUNCH(PT, bf16_t, float, float); else RN_LAUNCH(PT, bf16_t, float, bf16_t); } \
      else { if (out_dtype == MGPT_F32) RN_LAUNCH(PT, bf16_t, bf16_t, float); else RN_LAUNCH(PT, bf16_t, bf16_t, bf16_t); }     \
    }                                                                                                              \
  } while (0)
  if (!gate) gate_dtype = out_dtype;
  const int per_thread = (width + threads - 1) / threads;
  if (per_thread <= 2) RN_TYPES(2);
  else if (per_thread <= 4) RN_TYPES(4);
  else if (per_thread <= 6) RN_TYPES(6);
  else if (per_thread <= 8) RN_TYPES(8);
  else if (per_thread <= 16) RN_TYPES(16);
  else RN_TYPES(0);
#undef RN_TYPES
#undef RN_LAUNCH
  return mgpt_last_error();
}

// sum over the workgroup's 256 threads, the same value in every thread; waves are added in order
__device__ __forceinline__ float block_sum_256(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();      // the scratch's readers of the call before are done
  if ((threadIdx.x & 63) == 0) scratch[wave] = v;
  __syncthreads();
  return (scratch[0] + scratch[1]) + (scratch[2] + scratch[3]);
}

#define RMS_MAX_BRANCHES 4

struct RmsBranches {
  float* y[RMS_MAX_BRANCHES];
  const float* gain[RMS_MAX_BRANCHES];
};

__global__ __launch_bounds__(256) void rms_post_norm_kernel(RmsBranches br, int n_branches, float coef, int join_unit,
                                                            float* __restrict__ x, const float* __restrict__ gain_post,
                                                            const float* __restrict__ scale_post, float offset, float eps,
                                                            float mult, const float* __restrict__ gain_next,
                                                            void* __restrict__ h, int h_dtype, int n_rows, int width) {
  __shared__ float scratch[4];
  const int row = blockIdx.x;
  if (row >= n_rows) return;
  const long base = (long)row * width;
  float* y0 = br.y[0] + base;
  if (n_branches > 1) {
    // the branches' outputs, each normed with its own plain gain, averaged into the first one's buffer
    float r[RMS_MAX_BRANCHES];
    for (int b = 0; b < n_branches; ++b) {
      const float* yb = br.y[b] + base;
      float ss = 0.f;
      if (join_unit)
        for (int c = threadIdx.x; c < width; c += 256) ss = fmaf(yb[c], yb[c], ss);
      r[b] = join_unit ? coef / sqrtf(block_sum_256(ss, scratch) / (float)width + eps) : coef;
    }
    for (int c = threadIdx.x; c < width; c += 256) {
      float v = 0.f;
      for (int b = 0; b < n_branches; ++b) {
        v = fmaf(br.y[b][base + c] * r[b], br.gain[b][c], v);
        if (b) br.y[b][base + c] = 0.f;
      }
      y0[c] = v;      // read again below by the thread that wrote it
    }
  }
  float ss = 0.f;
  for (int c = threadIdx.x; c < width; c += 256) ss = fmaf(y0[c], y0[c], ss);
  const float ry = mult / sqrtf(block_sum_256(ss, scratch) / (float)width + eps);
  float sx = 0.f;
  for (int c = threadIdx.x; c < width; c += 256) {
    const float v = x[base + c] + y0[c] * ry * (offset + gain_post[c]) * (scale_post ? scale_post[c] : 1.0f);
    x[base + c] = v;
    y0[c] = 0.f;
    sx = fmaf(v, v, sx);
  }
  if (!gain_next) {
    if (h)
      for (int c = threadIdx.x; c < width; c += 256) store_f(h, h_dtype, base + c, x[base + c]);
    return;
  }
  const float rx = 1.0f / sqrtf(block_sum_256(sx, scratch) / (float)width + eps);
  for (int c = threadIdx.x; c < width; c += 256)
    store_f(h, h_dtype, base + c, x[base + c] * rx * (offset + gain_next[c]));
}

// The same step for one or two branches and rows of up to 4,096 values, four a lane of W waves: every value is loaded once,
// and all of them (the row, the sublayers' outputs, the gains) are on their way before the first sum.  PIECES: rows that
// 16-byte pieces cover; other rows have a lane's four values 64 W apart, so that a wave's 4-byte loads lie together.  A row's
// sums then run in another order, but always in the same.  Four waves with 4 to 16 values of 4 bytes a thread and a test of the
// output's type for each / here, us a call: 8 rows of 1,024 2.72 / 2.10, of 1,023 3.23 / 2.80, of 2,048 3.6 / 2.4, of 2,047
// 4.2 / 3.1; 3,000 rows of 1,023 10.3 / 9.0, of 2,047 19.4 / 18.5.  The kernel above, which reads a row three to five times,
// took 4.2 and 12.4 for 8 and 3,000 rows of 1,023, 5.7 and 22.9 for rows of 2,047.  (Five and twelve waves: without them
// 1,028 values are a little over half of eight waves' lanes, 1,900 such rows 8.9 us; in five waves 7.9, before 8.4; 1,900 of
// 2,052 15.7 / 13.9 in twelve.)
template <int W, int NB, bool PIECES>
__global__ __launch_bounds__(64 * W) void rms_post_norm_row_kernel(RmsBranches br, float coef, int join_unit,
                                                                   float* __restrict__ x, const float* __restrict__ gain_post,
                                                                   const float* __restrict__ scale_post, float offset,
                                                                   float eps, float mult, const float* __restrict__ gain_next,
                                                                   void* __restrict__ h, int h_dtype, int width) {
  __shared__ float scratch[W];
  const int tid = threadIdx.x;
  const bool in = (PIECES ? 4 * tid : tid) < width;
  const int c = in ? (PIECES ? 4 * tid : tid) : 0;
  const long base = (long)blockIdx.x * width;
  // this thread's values of a row: four neighbouring ones, or those at tid, tid + 64 W, ... (zeros behind the row's end)
  auto load4 = [&](const float* p) {
    if (PIECES) return *reinterpret_cast<const float4*>(p + c);
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (in) v.x = p[c];
    if (c + 64 * W < width) v.y = p[c + 64 * W];
    if (c + 128 * W < width) v.z = p[c + 128 * W];
    if (c + 192 * W < width) v.w = p[c + 192 * W];
    return v;
  };
  auto each = [&](auto store) {   // !PIECES: store(place in the buffer, which value)
    store(base + c, 0);
    if (c + 64 * W < width) store(base + c + 64 * W, 1);
    if (c + 128 * W < width) store(base + c + 128 * W, 2);
    if (c + 192 * W < width) store(base + c + 192 * W, 3);
  };
  // sum over the workgroup, the same value in every thread; waves are added in order
  auto block_sum = [&](float v) {
    v = wave_sum(in ? v : 0.f);
    if (W > 1) __syncthreads();   // the scratch's readers of the call before are done
    if ((tid & 63) == 0) scratch[tid >> 6] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < W; ++i) t += scratch[i];
    return t;
  };
  auto squares = [](float4 v) { return fmaf(v.x, v.x, fmaf(v.y, v.y, fmaf(v.z, v.z, v.w * v.w))); };
  float4 yv[NB], jg[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    yv[b] = load4(br.y[b] + base);
    if (NB > 1) jg[b] = load4(br.gain[b]);
  }
  float4 xv = load4(x + base);
  const float4 gp = load4(gain_post);
  float4 sp = make_float4(1.f, 1.f, 1.f, 1.f), gn = make_float4(0.f, 0.f, 0.f, 0.f);
  if (scale_post) sp = load4(scale_post);
  if (gain_next) gn = load4(gain_next);
  if (NB > 1) {
    // the branches' outputs, each normed with its own plain gain, averaged
    float r[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) r[b] = join_unit ? coef / sqrtf(block_sum(squares(yv[b])) / (float)width + eps) : coef;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      v.x = fmaf(yv[b].x * r[b], jg[b].x, v.x);
      v.y = fmaf(yv[b].y * r[b], jg[b].y, v.y);
      v.z = fmaf(yv[b].z * r[b], jg[b].z, v.z);
      v.w = fmaf(yv[b].w * r[b], jg[b].w, v.w);
    }
    yv[0] = v;
  }
  const float ry = mult / sqrtf(block_sum(squares(yv[0])) / (float)width + eps);
  xv.x += yv[0].x * ry * ((offset + gp.x) * sp.x);
  xv.y += yv[0].y * ry * ((offset + gp.y) * sp.y);
  xv.z += yv[0].z * ry * ((offset + gp.z) * sp.z);
  xv.w += yv[0].w * ry * ((offset + gp.w) * sp.w);
  if (in && PIECES) {
    *reinterpret_cast<float4*>(x + base + c) = xv;
#pragma unroll
    for (int b = 0; b < NB; ++b) *reinterpret_cast<float4*>(br.y[b] + base + c) = make_float4(0.f, 0.f, 0.f, 0.f);
  } else if (in) {
    const float xe[4] = {xv.x, xv.y, xv.z, xv.w};
    each([&](long at, int e) {
      x[at] = xe[e];
#pragma unroll
      for (int b = 0; b < NB; ++b) br.y[b][at] = 0.f;
    });
  }
  if (!gain_next && !h) return;
  float4 v = xv;
  if (gain_next) {
    const float rx = 1.0f / sqrtf(block_sum(squares(xv)) / (float)width + eps);
    v = make_float4(xv.x * rx * (offset + gn.x), xv.y * rx * (offset + gn.y), xv.z * rx * (offset + gn.z),
                    xv.w * rx * (offset + gn.w));
  }
  if (!in) return;
  if (!PIECES) {
    const float ve[4] = {v.x, v.y, v.z, v.w};
    each([&](long at, int e) { store_f(h, h_dtype, at, ve[e]); });
  } else if (h_dtype == MGPT_F32) {
    *reinterpret_cast<float4*>(reinterpret_cast<float*>(h) + base + c) = v;
  } else {
    uint2* dst = reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(h) + base + c);
    *dst = make_uint2(pack_bf16x2(v.x, v.y), pack_bf16x2(v.z, v.w));
  }
}

// y_ptrs / gain_ptrs: n_branches device pointers each (float32 [n_rows, width] buffers; [width] gains, unused
// with one branch).  x, y: contiguous float32 rows.
extern "C" int mgpt_rms_post_norm(float* y0, float* y1, float* y2, float* y3, const float* g0, const float* g1,
                                  const float* g2, const float* g3, int n_branches, float coef, int join_unit, float* x,
                                  const float* gain_post, const float* scale_post, float offset, float eps, float mult,
                                  const float* gain_next,
                                  void* h, int h_dtype, int n_rows, int width, hipStream_t stream) {
  if (n_rows == 0) return MGPT_OK;
  if (!x || !y0 || !gain_post || (gain_next && !h)) return MGPT_ERR_NULL;
  if (n_rows < 0 || width <= 0 || n_branches < 1 || n_branches > RMS_MAX_BRANCHES) return MGPT_ERR_BAD_SHAPE;
  if (h && !dtype_ok(h_dtype)) return MGPT_ERR_BAD_DTYPE;
  RmsBranches br = {{y0, y1, y2, y3}, {g0, g1, g2, g3}};
  for (int b = 0; b < n_branches; ++b)
    if (!br.y[b] || (n_branches > 1 && !br.gain[b])) return MGPT_ERR_NULL;
  uintptr_t together = (uintptr_t)x | (uintptr_t)gain_post | (uintptr_t)scale_post | (uintptr_t)gain_next | (uintptr_t)h;
  for (int b = 0; b < n_branches; ++b) together |= (uintptr_t)br.y[b] | (n_branches > 1 ? (uintptr_t)br.gain[b] : 0);
  const bool row = width <= 4096 && n_branches <= 2, pieces = width % 4 == 0 && (together & 15) == 0;
#define RPN_ROW3(W, NB, PIECES)                                                                                         \
  hipLaunchKernelGGL((rms_post_norm_row_kernel<W, NB, PIECES>), dim3(n_rows), dim3(64 * W), 0, stream, br, coef, join_unit, \
                     x, gain_post, scale_post, offset, eps, mult, gain_next, h, h_dtype, width)
#define RPN_ROW(W)                                          \
  do {                                                      \
    if (n_branches == 1 && pieces) RPN_ROW3(W, 1, true);    \
    else if (n_branches == 1) RPN_ROW3(W, 1, false);        \
    else if (pieces) RPN_ROW3(W, 2, true);                  \
    else RPN_ROW3(W, 2, false);                             \
  } while (0)
  if (row && width <= 256) RPN_ROW(1);
  else if (row && width <= 512) RPN_ROW(2);
  else if (row && width <= 1024) RPN_ROW(4);
  else if (row && width <= 1280) RPN_ROW(5);
  else if (row && width <= 2048) RPN_ROW(8);
  else if (row && width <= 3072) RPN_ROW(12);
  else if (row) RPN_ROW(16);
  else
    hipLaunchKernelGGL(rms_post_norm_kernel, dim3(n_rows), dim3(256), 0, stream, br, n_branches, coef, join_unit, x, gain_post,
                       scale_post, offset, eps, mult, gain_next, h, h_dtype, n_rows, width);
#undef RPN_ROW3
#undef RPN_ROW
  return mgpt_last_error();
}

// float32 rows in another storage type (the residual as the next product's operand, where no norm stands between)
__global__ __launch_bounds__(256) void cast_rows_kernel(const float* __restrict__ x, long ldx, void* __restrict__ out, int out_dtype,
                                                        long ldo, int width) {
  const int row = blockIdx.x;
  for (int c = blockIdx.y * 256 + threadIdx.x; c < width; c += 256 * gridDim.y)
    store_f(out, out_dtype, (long)row * ldo + c, x[(long)row * ldx + c]);
}

extern "C" int mgpt_cast_rows(const float* x, long ldx, void* out, int out_dtype, long ldo, int n_rows, int width,
                              hipStream_t stream) {
  if (n_rows == 0) return MGPT_OK;
  if (!x || !out) return MGPT_ERR_NULL;
  if (n_rows < 0 || width <= 0 || ldx < width || ldo < width) return MGPT_ERR_BAD_SHAPE;
  if (!dtype_ok(out_dtype)) return MGPT_ERR_BAD_DTYPE;
  const int cols = (width + 1023) / 1024;
  hipLaunchKernelGGL(cast_rows_kernel, dim3(n_rows, cols < 64 ? cols : 64), dim3(256), 0, stream, x, ldx, out, out_dtype, ldo, width);
  return mgpt_last_error();
}
