// The statistics of a LayerNorm over a row that one wave holds in vectors of four.
#pragma once
#include "common.h"

// Mean, what is left of it in the distances from it, and 1 / standard deviation of a row of n4 vectors of four, of which
// this lane has those at lane + 64 i; they become the distances from the mean.  One order of sums for every kernel that norms a row.
// Only the last PART of the LN_VEC may lie behind the row's end for some lanes.
template <int LN_VEC, int PART>
__device__ __forceinline__ void layernorm_sums(float4 (&xv)[LN_VEC], int n4, int width, float eps, float& mean, float& corr,
                                               float& rstd) {
  const int lane = threadIdx.x & (MGPT_WAVE - 1);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < LN_VEC; ++i) {
    if (i >= LN_VEC - PART && lane + i * MGPT_WAVE >= n4) xv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    s += (xv[i].x + xv[i].y) + (xv[i].z + xv[i].w);
  }
  mean = wave_sum(s) / (float)width;
  float e = 0.f, v2 = 0.f;
#pragma unroll
  for (int i = 0; i < LN_VEC; ++i) {
    const bool in = i < LN_VEC - PART || lane + i * MGPT_WAVE < n4;
    float* p = reinterpret_cast<float*>(&xv[i]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float d = in ? p[k] - mean : 0.f;
      p[k] = d;
      e += d;
      v2 = fmaf(d, d, v2);
    }
  }
  corr = wave_sum(e) / (float)width;
  const float var = fmaxf(wave_sum(v2) / (float)width - corr * corr, 0.f);
  rstd = 1.0f / sqrtf(var + eps);
}
