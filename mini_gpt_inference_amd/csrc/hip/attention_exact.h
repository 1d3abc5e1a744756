// The 32-bit path's attention on the matrix cores (attention_exact.hip), called by the general attention's launcher.
#pragma once
#include <hip/hip_runtime.h>

// As the general attention's arguments, all float32; sinks, gate, dist_bias and slopes may be null.
struct AttentionExactArgs {
  const float* q; long ldq;
  float* out; long ldo;
  const float* kpool; const float* vpool;
  const int* block_tables; int max_blocks;
  const int* cu_q; const int* seq_lens; const int* q_req;
  int n_tokens, n_req, n_head, n_kv_head, page_size;
  float scale; int window;
  const float* sinks; float softcap;
  const float* gate; long ldg;
  int keep_first, chunked;
  const float* dist_bias; int bias_len;
  const float* slopes;
};

// Whether the kernel takes these: nothing in it depends on a step's size (but for a step of no requests, which has nothing to
// do), so a model's calls are all taken or none is.
bool mgpt_attention_exact_takes(const AttentionExactArgs& a, int head_dim);
// single: every request has one token, token n being request n's (q_req[n] < 0: padding).
int mgpt_attention_exact_launch(const AttentionExactArgs& a, int head_dim, int single, hipStream_t stream);
