// The 32-bit path's matrix product (linear_exact.hip), called by the general product's launcher.
#pragma once
#include <hip/hip_runtime.h>

// Pages that the key and value columns of a product go to as well (see mgpt_linear_exact_qkv).
struct ExactScatter {
  float* kpool; float* vpool;
  const int* slot_mapping;
  int q_width, kv_width, head_dim, page_size;
};

// A [n_rows, k_dim] with row stride lda, W [n_out, k_dim] dense, bias (may be null), out [n_rows, n_out] with row
// stride ldo, all float32; epi: the general product's epilogue codes.  Arguments are checked by the caller.
int mgpt_linear_exact_launch(const float* A, long lda, const float* W, const float* bias, float* out, long ldo, int n_rows,
                             int n_out, int k_dim, int epi, const ExactScatter& sc, hipStream_t stream);
