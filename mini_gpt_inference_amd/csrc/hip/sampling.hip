// Next-token choice from 32-bit logits: one workgroup per row.
//
// Order of operations as the reference (src/minigpt_infer/sampling.py:97-137,
// src/minigpt_infer/engine/engine.py:154-159): ids at or above real_vocab are
// never chosen; temperature <= 0 takes the argmax of the unscaled logits (the
// lowest index among equals); otherwise s = logits / max(T, 1e-6); top-k keeps
// the values >= the k-th largest (ties pass, sampling.py:39-52); top-p keeps a
// token iff the probability mass of the strictly larger ones is <= p, so the
// largest always stays (sampling.py:55-76); then a softmax over what is left.
//
// Where the reference draws with torch.multinomial from one shared generator,
// this draws by inverse CDF in vocabulary order with a uniform number that is a
// pure function of (engine seed, request seed, index of the output token), so a
// request's tokens do not depend on batching or preemption.
#include "common.h"
#include "launchers.h"

#define SAMPLE_THREADS 1024
#define SAMPLE_WAVES (SAMPLE_THREADS / MGPT_WAVE)
#define SAMPLE_SCOUT (SAMPLE_THREADS - MGPT_WAVE)   // the thread that writes the token: the last wave's first
static_assert(SAMPLE_WAVES <= 16, "the greedy path reduces the waves' results within one row of 16 lanes");

__device__ __forceinline__ unsigned int float_key(float f) {
  unsigned int u = __float_as_uint(f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);  // monotone: larger float -> larger key
}

__device__ __forceinline__ uint64_t mix64(uint64_t z) {
  z ^= z >> 30; z *= 0xBF58476D1CE4E5B9ull;
  z ^= z >> 27; z *= 0x94D049BB133111EBull;
  z ^= z >> 31;
  return z;
}

// uniform in [0, 1) with 24 bits
__device__ __forceinline__ float sample_uniform(uint64_t engine_seed, uint64_t request_seed,
                                                uint64_t index) {
  uint64_t z = engine_seed * 0x9E3779B97F4A7C15ull + request_seed * 0xD1B54A32D192ED03ull +
               index * 0x8CB92BA72F3D8DD7ull + 0x2545F4914F6CDD1Dull;
  z = mix64(mix64(z));
  return (float)(z >> 40) * (1.0f / 16777216.0f);
}

__device__ float block_sum(float v, float* red) {
  v = wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < SAMPLE_WAVES; ++i) t += red[i];  // fixed order
  return t;
}

__device__ int block_sum_int(int v, int* red) {
  v = wave_sum_int(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  int t = 0;
  for (int i = 0; i < SAMPLE_WAVES; ++i) t += red[i];
  return t;
}

__device__ float block_max(float v, float* red) {
  v = wave_max(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  float t = -INFINITY;
  for (int i = 0; i < SAMPLE_WAVES; ++i) t = fmaxf(t, red[i]);
  return t;
}

// DPP move within rows of 16 lanes
template <int CTRL>
__device__ __forceinline__ int dpp_i(int v) { return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, false); }

// (value, index) of the largest value, the lowest index among equals, over each row of 16 lanes;
// every lane of the row gets it.  Four DPP exchanges: neighbours, pairs, halves of 8, halves of 16.
__device__ __forceinline__ void argmax_rows16(float& best, int& best_i) {
#define ARGMAX_STEP(CTRL)                                                         \
  {                                                                               \
    const float ov = __int_as_float(dpp_i<CTRL>(__float_as_int(best)));           \
    const int oi = dpp_i<CTRL>(best_i);                                           \
    if (ov > best || (ov == best && oi < best_i)) { best = ov; best_i = oi; }     \
  }
  ARGMAX_STEP(0xB1)   // quad_perm [1,0,3,2]
  ARGMAX_STEP(0x4E)   // quad_perm [2,3,0,1]
  ARGMAX_STEP(0x141)  // row_half_mirror
  ARGMAX_STEP(0x140)  // row_mirror
#undef ARGMAX_STEP
}

// Calls f(index, value) for every logit below nv, each thread taking indices 1024 apart.  When the
// row is 16-byte aligned the loads are four floats wide and eight of them are issued before any
// is used, so one pass over the vocabulary costs a few memory latencies, not one per element.
template <typename F>
__device__ __forceinline__ void scan_row(const float* __restrict__ lg, int nv, F f) {
  const int tid = threadIdx.x;
  if ((reinterpret_cast<uintptr_t>(lg) & 15) == 0) {
    const int n4 = nv >> 2;
    const float4* lg4 = reinterpret_cast<const float4*>(lg);
    constexpr int U = 16;
    for (int base = tid; base < n4; base += SAMPLE_THREADS * U) {
      float4 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i4 = base + u * SAMPLE_THREADS;
        v[u] = lg4[i4 < n4 ? i4 : base];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i4 = base + u * SAMPLE_THREADS;
        if (i4 < n4) {
          f(4 * i4, v[u].x);
          f(4 * i4 + 1, v[u].y);
          f(4 * i4 + 2, v[u].z);
          f(4 * i4 + 3, v[u].w);
        }
      }
    }
    const int i = 4 * n4 + tid;
    if (i < nv) f(i, lg[i]);
  } else {
    for (int i = tid; i < nv; i += SAMPLE_THREADS) f(i, lg[i]);
  }
}

// After a decode-only step (token n is request n's one token and every row is sampled) one thread of the row
// (SAMPLE_SCOUT) can prepare the next step on the device: the sampled token becomes the next input,
// position, length and output index go up by one, the cache slot of the new position is looked up
// in the block tables (which already hold the pages of the steps planned ahead), and the token is
// also appended to the row's column of a history that the host reads once at the end.  Then
// several decode steps run back to back with no copy between them.  token_ids == nullptr: off.
struct AdvanceArgs {
  int* token_ids;
  int* positions;
  int* seq_lens;
  int* out_index;
  const int* q_req;         // -1: a padded row, left alone
  int* slot_mapping;        // [n_groups][n_stride]
  const int* block_tables;  // [n_groups][r_stride][max_blocks]
  const int* page_sizes;    // [n_groups]
  int n_groups, n_stride, r_stride, max_blocks;
  int* history;             // [history_rows][history_stride]
  int* history_pos;         // per row: how many tokens it has appended
  int history_rows, history_stride;
};

// What that thread reads for it, asked for at the kernel's start: none of it depends on the
// token, and two of the loads depend on each other (the position, then the block table's entry), so
// behind the choice they would be two trips to memory more.
#define SAMPLE_ADV_GROUPS 4   // cache groups whose slots are looked up ahead; more are looked up at the end
struct AdvanceAhead {
  bool live;
  int pos, seq_len, out_index, history_pos;
  int slot[SAMPLE_ADV_GROUPS];
};

__device__ __forceinline__ int advance_slot(int row, int pos, int g, const AdvanceArgs& adv) {
  const int ps = adv.page_sizes[g];
  const int idx = pos / ps;
  const int page = idx < adv.max_blocks ? adv.block_tables[((long)g * adv.r_stride + row) * adv.max_blocks + idx] : -1;
  return page >= 0 ? page * ps + pos % ps : -1;
}

__device__ __forceinline__ AdvanceAhead look_ahead(int row, const AdvanceArgs& adv) {
  AdvanceAhead a;
  a.live = adv.token_ids != nullptr && adv.q_req[row] >= 0;
  a.pos = a.seq_len = a.out_index = a.history_pos = 0;
#pragma unroll
  for (int g = 0; g < SAMPLE_ADV_GROUPS; ++g) a.slot[g] = -1;
  if (!a.live) return a;
  a.pos = adv.positions[row] + 1;
  a.seq_len = adv.seq_lens[row] + 1;
  a.out_index = adv.out_index[row] + 1;
  a.history_pos = adv.history_pos[row];
#pragma unroll
  for (int g = 0; g < SAMPLE_ADV_GROUPS; ++g)
    if (g < adv.n_groups) a.slot[g] = advance_slot(row, a.pos, g, adv);
  return a;
}

__device__ __forceinline__ void finish_row(int row, int token, int* out_tokens, const AdvanceArgs& adv,
                                           const AdvanceAhead& ahead) {
  out_tokens[row] = token;
  if (!ahead.live) return;
  adv.token_ids[row] = token;
  adv.positions[row] = ahead.pos;
  adv.seq_lens[row] = ahead.seq_len;
  adv.out_index[row] = ahead.out_index;
#pragma unroll
  for (int g = 0; g < SAMPLE_ADV_GROUPS; ++g)
    if (g < adv.n_groups) adv.slot_mapping[(long)g * adv.n_stride + row] = ahead.slot[g];
  for (int g = SAMPLE_ADV_GROUPS; g < adv.n_groups; ++g)
    adv.slot_mapping[(long)g * adv.n_stride + row] = advance_slot(row, ahead.pos, g, adv);
  const int j = ahead.history_pos;
  if (j < adv.history_rows) adv.history[(long)j * adv.history_stride + row] = token;
  adv.history_pos[row] = j + 1;
}

// The token of a greedy row (temperature <= 0).
__device__ __forceinline__ void greedy_row(const float* __restrict__ lg, int row, int nv,
                                           const float* __restrict__ tile_best,
                                           const int* __restrict__ tile_best_idx, int n_tiles, float* red_f, int* red_i,
                                           int* out_tokens, const AdvanceArgs& adv, const AdvanceAhead& ahead) {
  const int tid = threadIdx.x;
  // argmax, the lowest index among equals.  A thread meets its indices in rising order, so a
  // strictly larger value is all it has to look for; four logits are compared as their maximum.
  float best = -INFINITY;
  int best_i = 0x7fffffff;
  if (tile_best != nullptr) {
    // the kernel that made the logits has left every tile's best (mgpt_linear_head_best, which
    // already kept to the columns below real_vocab): a few kilobytes to read instead of the row
    const float* tb = tile_best + (long)row * n_tiles;
    const int* ti = tile_best_idx + (long)row * n_tiles;
    constexpr int U = 4;
    // The last wave reads none of it: what it looks up for the next step is a chain of four loads, which this way
    // runs beside the other waves' loads and not in front of its own.
    for (int base = tid < SAMPLE_SCOUT ? tid : n_tiles; base < n_tiles; base += SAMPLE_SCOUT * U) {
      float v[U];
      int ix[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = base + u * SAMPLE_SCOUT;
        v[u] = tb[i < n_tiles ? i : base];
        ix[u] = ti[i < n_tiles ? i : base];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (base + u * SAMPLE_SCOUT < n_tiles && v[u] > best) { best = v[u]; best_i = ix[u]; }
    }
  } else if ((reinterpret_cast<uintptr_t>(lg) & 15) == 0) {
    const int n4 = nv >> 2;
    const float4* lg4 = reinterpret_cast<const float4*>(lg);
    constexpr int U = 16;  // loads in flight per thread: one pass covers 64 Ki logits
    for (int base = tid; base < n4; base += SAMPLE_THREADS * U) {
      float4 v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i4 = base + u * SAMPLE_THREADS;
        v[u] = lg4[i4 < n4 ? i4 : base];
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i4 = base + u * SAMPLE_THREADS;
        const float m = fmaxf(fmaxf(v[u].x, v[u].y), fmaxf(v[u].z, v[u].w));
        if (i4 < n4 && m > best) {
          best = m;
          best_i = 4 * i4 + (v[u].x == m ? 0 : (v[u].y == m ? 1 : (v[u].z == m ? 2 : 3)));
        }
      }
    }
    const int i = 4 * n4 + tid;  // the row's last one to three logits
    if (i < nv && lg[i] > best) { best = lg[i]; best_i = i; }
  } else {
    for (int i = tid; i < nv; i += SAMPLE_THREADS)
      if (lg[i] > best) { best = lg[i]; best_i = i; }
  }
  // NaN-free rows always have a candidate; a row of -inf falls back to index 0
  argmax_rows16(best, best_i);
  // lanes 0, 16, 32, 48 hold their rows' best: the wave's best through scalar registers
  {
    float wb = best;
    int wi = best_i;
#pragma unroll
    for (int r = 1; r < 4; ++r) {
      const float ov = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(best), 16 * r));
      const int oi = __builtin_amdgcn_readlane(best_i, 16 * r);
      if (ov > wb || (ov == wb && oi < wi)) { wb = ov; wi = oi; }
    }
    best = wb;  // right in lane 0 (and in every lane of the first row)
    best_i = wi;
  }
  if ((tid & 63) == 0) { red_f[tid >> 6] = best; red_i[tid >> 6] = best_i; }
  __syncthreads();
  if (tid >= SAMPLE_SCOUT) {
    // the sixteen waves' results, one per lane of the wave's first row, reduced the same way
    const int lane = tid - SAMPLE_SCOUT;
    best = lane < SAMPLE_WAVES ? red_f[lane] : -INFINITY;
    best_i = lane < SAMPLE_WAVES ? red_i[lane] : 0x7fffffff;
    argmax_rows16(best, best_i);
  }
  if (tid == SAMPLE_SCOUT) finish_row(row, best_i == 0x7fffffff ? 0 : best_i, out_tokens, adv, ahead);
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_kernel(
    const float* __restrict__ logits, long ld, int vocab, int real_vocab,
    const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, const uint64_t* __restrict__ request_seed,
    const int* out_index, uint64_t engine_seed, int* out_tokens, AdvanceArgs adv,
    const float* __restrict__ tile_best, const int* __restrict__ tile_best_idx, int n_tiles) {
  __shared__ float red_f[SAMPLE_WAVES];
  __shared__ int red_i[SAMPLE_WAVES];
  __shared__ float part[SAMPLE_THREADS];
  __shared__ float wave_off[SAMPLE_WAVES + 1];
  __shared__ int chosen;

  const int row = blockIdx.x, tid = threadIdx.x;
  AdvanceAhead ahead;
  ahead.live = false;
  if (tid == SAMPLE_SCOUT) ahead = look_ahead(row, adv);
  const float* lg = logits + (long)row * ld;
  const int nv = real_vocab < vocab ? real_vocab : vocab;
  const float temp = temperature[row];

  if (temp <= 0.f) {
    greedy_row(lg, row, nv, tile_best, tile_best_idx, n_tiles, red_f, red_i, out_tokens, adv, ahead);
    return;
  }

  const float t_safe = fmaxf(temp, 1e-6f);
  // largest scaled logit
  float mx = -INFINITY;
  scan_row(lg, nv, [&](int, float v) { mx = fmaxf(mx, v / t_safe); });
  mx = block_max(mx, red_f);

  // top-k: key of the k-th largest value, by bisection on the ordered bit pattern
  unsigned int key_floor = 0u;  // keep keys >= key_floor
  const int k = top_k ? top_k[row] : 0;
  if (k > 0 && k < nv) {
    unsigned int lo = 0u, hi = 0xffffffffu;  // invariant: count(key >= lo) >= k
    while (lo < hi) {
      unsigned int mid = lo + (unsigned int)(((uint64_t)hi - lo + 1) >> 1);
      int cnt = 0;
      scan_row(lg, nv, [&](int, float v) { cnt += float_key(v / t_safe) >= mid; });
      cnt = block_sum_int(cnt, red_i);
      if (cnt >= k) lo = mid; else hi = mid - 1;
    }
    key_floor = lo;
  }

  // top-p: smallest key kappa with mass(key > kappa) <= p * Z
  const float p = top_p ? top_p[row] : 1.0f;
  if (p < 1.0f) {
    float z = 0.f;
    scan_row(lg, nv, [&](int, float v) {
      const float s = v / t_safe;
      if (float_key(s) >= key_floor) z += expf(s - mx);
    });
    z = block_sum(z, red_f);
    const float budget = p * z;
    unsigned int lo = key_floor, hi = float_key(mx);  // G(hi) = 0 <= budget always
    while (lo < hi) {
      unsigned int mid = lo + ((hi - lo) >> 1);
      float g = 0.f;
      scan_row(lg, nv, [&](int, float v) {
        const float s = v / t_safe;
        const unsigned int key = float_key(s);
        if (key > mid && key >= key_floor) g += expf(s - mx);
      });
      g = block_sum(g, red_f);
      if (g <= budget) hi = mid; else lo = mid + 1;
    }
    key_floor = lo;
  }

  // inverse CDF in vocabulary order over what is kept
  const int per = (nv + SAMPLE_THREADS - 1) / SAMPLE_THREADS;
  const int i0 = tid * per, i1 = (i0 + per < nv) ? i0 + per : nv;
  float mine = 0.f;
  int last_kept = -1;
  for (int i = i0; i < i1; ++i) {
    float s = lg[i] / t_safe;
    if (float_key(s) >= key_floor) { mine += expf(s - mx); last_kept = i; }
  }
  part[tid] = mine;
  if (tid == 0) chosen = 0x7fffffff;
  __syncthreads();
  // serial scans keep the prefix sums monotone
  if ((tid & 63) == 0) {
    float run = 0.f;
    for (int i = 0; i < MGPT_WAVE; ++i) { run += part[tid + i]; part[tid + i] = run; }
  }
  __syncthreads();
  if (tid == 0) {
    float run = 0.f;
    wave_off[0] = 0.f;
    for (int w = 0; w < SAMPLE_WAVES; ++w) { run += part[w * MGPT_WAVE + MGPT_WAVE - 1]; wave_off[w + 1] = run; }
  }
  __syncthreads();
  const float total = wave_off[SAMPLE_WAVES];
  const float u = sample_uniform(engine_seed, request_seed ? request_seed[row] : 0ull,
                                 (uint64_t)(out_index ? out_index[row] : 0));
  const float target = u * total;
  const int w = tid >> 6;
  const float incl = wave_off[w] + part[tid];
  const float excl = (tid & 63) ? wave_off[w] + part[tid - 1] : wave_off[w];
  if (mine > 0.f && excl <= target && target < incl) {
    float run = excl;
    int pick = last_kept;
    for (int i = i0; i < i1; ++i) {
      float s = lg[i] / t_safe;
      if (float_key(s) >= key_floor) {
        run += expf(s - mx);
        if (run > target) { pick = i; break; }
      }
    }
    atomicMin(&chosen, pick);
  }
  // rounding can leave target >= total: then the last kept id stands
  int lk = last_kept;
  for (int off = 32; off > 0; off >>= 1) lk = max(lk, __shfl_xor(lk, off, MGPT_WAVE));
  __syncthreads();
  if ((tid & 63) == 0) red_i[tid >> 6] = lk;
  __syncthreads();
  if (tid == SAMPLE_SCOUT) {
    int c = chosen;
    if (c == 0x7fffffff) {
      c = 0;
      for (int i = 0; i < SAMPLE_WAVES; ++i) c = max(c, red_i[i]);
    }
    finish_row(row, c, out_tokens, adv, ahead);
  }
}

__device__ __forceinline__ float key_float(unsigned int k) {  // the inverse of float_key
  return __uint_as_float((k & 0x80000000u) ? (k ^ 0x80000000u) : ~k);
}

__device__ __forceinline__ unsigned int wave_min_uint(unsigned int v) {
  for (int off = 32; off > 0; off >>= 1) {
    const unsigned int o = __shfl_xor(v, off, MGPT_WAVE);
    v = o < v ? o : v;
  }
  return v;
}

__device__ unsigned int block_min_uint(unsigned int v, unsigned int* red) {
  v = wave_min_uint(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  unsigned int t = 0xffffffffu;
  for (int i = 0; i < SAMPLE_WAVES; ++i) t = red[i] < t ? red[i] : t;
  return t;
}

// Where a thread's n entries go in a list that holds the entries of all threads in order; total: all of them.
__device__ int block_place(int n, int* red, int& total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = n;
  for (int off = 1; off < MGPT_WAVE; off <<= 1) {
    const int o = __shfl_up(incl, off, MGPT_WAVE);
    if (lane >= off) incl += o;
  }
  __syncthreads();
  if (lane == MGPT_WAVE - 1) red[w] = incl;
  __syncthreads();
  int before = 0, all = 0;
  for (int i = 0; i < SAMPLE_WAVES; ++i) {
    if (i < w) before += red[i];
    all += red[i];
  }
  total = all;
  return before + incl - n;
}

#define SAMPLE_LIST 512                       // candidates that one wave holds, eight a lane
#define SAMPLE_HELD (SAMPLE_LIST / MGPT_WAVE)
#define SAMPLE_KEY_NEG_INF 0x007fffffu        // float_key(-inf)

// Fifty comparisons with x that are made a second time are cheaper than their results kept in scalar registers, which the
// compiler would do and spill them.
#define FORGET_COMPARISONS(x) asm volatile("" : "+v"(x))

// Searches of one wave over 64 N keys x, N a lane (0 stands for none), and their masses e.  A round is a few
// instructions: no barrier, and for counts no sum over lanes.
template <int N>
__device__ __forceinline__ int wave_count(const unsigned int (&x)[N], unsigned int from) {
  int cnt = 0;
#pragma unroll
  for (int q = 0; q < N; ++q) cnt += __popcll(__ballot(x[q] >= from));
  return cnt;
}

// The smallest kappa in [lo, hi] with base + (mass of the keys above kappa) <= budget; hi is known to hold.
template <int N>
__device__ __forceinline__ unsigned int wave_top_p(const unsigned int (&x)[N], const float (&e)[N], unsigned int lo,
                                                   unsigned int hi, float base, float budget) {
  while (lo < hi) {
    const unsigned int mid = lo + ((hi - lo) >> 1);
    float g = 0.f;
#pragma unroll
    for (int q = 0; q < N; ++q) g += x[q] > mid ? e[q] : 0.f;
    g = base + wave_sum(g);
    if (g <= budget) hi = mid; else lo = mid + 1;
  }
  return lo;
}

// Top-k and top-p over a list of n <= SAMPLE_LIST entries in LDS (keys, and masses by key), zeros behind them up to a
// multiple of four: the smallest key that both keep, the same in all threads.  A thread has an entry and goes over the whole list:
// fewer than k keys above its own, and their mass within the budget.  64 rows of 50,304 logits, temperature, top-k 50 and top-p 26.9 us
// with two searches by halving in one wave, some 60 rounds with sums over lanes, 24.4 so.
__device__ __forceinline__ unsigned int list_floor(const unsigned int* key, const float* mass, int n, int k, float p, float* red_f,
                                                   int* red_i) {
  const int t = threadIdx.x;
  const unsigned int mine = t < n ? key[t] : 0xffffffffu;
  int above = 0;
  double before = 0.;                              // (a chain of 128 additions in 32 bits is off by up to 1.5e-6)
  if (t < n) {
    for (int q = 0; q < n; q += 4) {
      const uint4 x = *reinterpret_cast<const uint4*>(key + q);
      const float4 e = *reinterpret_cast<const float4*>(mass + q);
      above += (x.x > mine) + (x.y > mine) + (x.z > mine) + (x.w > mine);
      const float four = ((x.x > mine ? e.x : 0.f) + (x.y > mine ? e.y : 0.f)) + ((x.z > mine ? e.z : 0.f) + (x.w > mine ? e.w : 0.f));
      before += (double)four;
    }
  }
  bool keep = t < n && above < k;
  if (p < 1.0f) {
    const float z = block_sum(keep ? mass[t] : 0.f, red_f);
    keep = keep && (before <= (double)p * z || above == 0);   // (the largest logit stays whatever p is)
  }
  return block_min_uint(keep ? mine : 0xffffffffu, reinterpret_cast<unsigned int*>(red_i));
}

// The same choice for rows of at most 1024 x K logits, each thread keeping its stretch of `per` consecutive logits in
// registers (K of them at most), so that the row is read from memory once.  The kernel above reads it again for each of
// the 30 to 65 counts and sums of its two searches, about 6 us a time.  Rows of 50,304 logits, 64 of them, us a call,
// above / here: temperature, top-k 50 and top-p 447 / 24; top-p alone 414 / 118 (flat), 373 / 81 (sharp); temperature
// alone 47 / 35; greedy rows 6.3 / 6.3.  What is left is one workgroup's load of 200 KB (4 us) and the instructions of
// its 16 waves over 50 logits a thread; a row cut over workgroups would need them to meet.
//
// A thread's stretch comes through LDS: a wave loads its 64 stretches, which lie one behind the other, 64 logits at a
// time, half of the lanes' stretches after the other.  Stretches and the order of the inverse CDF's sums are those of the
// kernel above: from the same kept logits the token is the same.  What top-k keeps is the same; top-p's masses are summed
// in another order here, so a logit whose mass ends within float32 rounding of p may be kept by one and not by the other.
//
// Top-k: the k-th largest of the threads' own largest logits bounds the k-th largest logit from below; the few logits
// above that bound go to a list, which every thread then counts over for one entry.  The bound is on the unscaled logits, eight representable numbers lower, because logits that differ by
// less may be equal after the division by a temperature of at most 4.  Rows with infinities or NaN, higher temperatures,
// k over 512 and rows whose list would be too long search over all registers instead; so does top-p alone, until at
// most SAMPLE_LIST logits are left undecided.
template <int K>
__global__ __launch_bounds__(SAMPLE_THREADS) void sample_held_kernel(
    const float* __restrict__ logits, long ld, int vocab, int real_vocab,
    const float* __restrict__ temperature, const int* __restrict__ top_k,
    const float* __restrict__ top_p, const uint64_t* __restrict__ request_seed,
    const int* out_index, uint64_t engine_seed, int* out_tokens, AdvanceArgs adv,
    const float* __restrict__ tile_best, const int* __restrict__ tile_best_idx, int n_tiles) {
  extern __shared__ __attribute__((aligned(16))) float sh_lds[];   // 32 stretches of each wave; then lists
  __shared__ float red_f[SAMPLE_WAVES];
  __shared__ int red_i[SAMPLE_WAVES];
  __shared__ unsigned int shared_key;
  __shared__ int chosen;

  const int row = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  __shared__ AdvanceAhead kept_ahead;              // the scout's, for the end; in LDS, where they take no registers
  __shared__ AdvanceArgs kept_adv;
  __shared__ int* kept_out;
  AdvanceAhead ahead;
  ahead.live = false;
  if (tid == SAMPLE_SCOUT) ahead = look_ahead(row, adv);
  const float* lg = logits + (long)row * ld;
  const int nv = real_vocab < vocab ? real_vocab : vocab;
  const float temp = temperature[row];
  if (temp <= 0.f) {
    greedy_row(lg, row, nv, tile_best, tile_best_idx, n_tiles, red_f, red_i, out_tokens, adv, ahead);
    return;
  }
  if (tid == SAMPLE_SCOUT) {
    kept_ahead = ahead;
    kept_adv = adv;
    kept_out = out_tokens;
  }
  const float u = sample_uniform(engine_seed, request_seed ? request_seed[row] : 0ull,
                                 (uint64_t)(out_index ? out_index[row] : 0));
  const int k = top_k ? top_k[row] : 0;
  const float p = top_p ? top_p[row] : 1.0f;
  const float t_safe = fmaxf(temp, 1e-6f);
  const bool cut_k = k > 0 && k < nv;

  const int per = (nv + SAMPLE_THREADS - 1) / SAMPLE_THREADS;   // <= K
  const int i0 = tid * per;
  const int n_mine = nv - i0 < 0 ? 0 : (nv - i0 < per ? nv - i0 : per);
  float v[K];                                                   // logits i0 .. i0 + n_mine - 1, then NaN
  float m = -INFINITY;
  bool odd = false;                                             // an infinity or NaN among them
  {
    // Stretches lie one behind the other; 32 lanes that each read their own stretch's j-th logit meet in few banks when
    // its length is a multiple of 8, so a word is then left out behind every 64.
    const int pad = (per & 7) == 0;
    float* mine = sh_lds + w * (32 * per + (per >> 1) + 1);
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      const int first = h * 32 * per, r0 = first >> 6;
      float raw[K / 2 + 1];
#pragma unroll
      for (int r = 0; r <= K / 2; ++r) {
        const int i = (w * per + r0 + r) * MGPT_WAVE + lane;
        raw[r] = lg[i < nv ? i : nv - 1];
      }
      if (h) __syncthreads();
#pragma unroll
      for (int r = 0; r <= K / 2; ++r) {
        odd |= !(fabsf(raw[r]) <= 3.402823466e38f);
        const int e = (r0 + r) * MGPT_WAVE + lane - first;
        if (e >= 0 && e < 32 * per) mine[e + (pad ? e >> 6 : 0)] = raw[r];
      }
      __syncthreads();
      if ((lane >> 5) == h) {
        const float* own = mine + (lane & 31) * per;                   // past the stretch: dropped below
        if (pad) {
#pragma unroll
          for (int j = 0; j < K; ++j) v[j] = own[j + (((lane & 31) * per + (j & ~7)) >> 6)];   // eights do not straddle
        } else {
#pragma unroll
          for (int j = 0; j < K; ++j) v[j] = own[j];
        }
      }
    }
#pragma unroll
    for (int j = 0; j < K; ++j) {
      v[j] = j < n_mine ? v[j] : __uint_as_float(0x7fc00000u);
      m = fmaxf(m, v[j]);
    }
  }
  const float mx = block_max(m, red_f) / t_safe;   // the largest scaled logit: division keeps the order
  const bool any_odd = __syncthreads_or(odd);      // also: every lane has its stretch, the LDS is free

  unsigned int key_floor = 1u;                     // keep keys >= key_floor; 0 stands for no logit
  float mine = 0.f;
  int last_kept = -1, mine_from = 0, mine_to = 0;  // the thread's entries of the list
  unsigned int* list_key = reinterpret_cast<unsigned int*>(sh_lds);
  float* list_e = sh_lds + SAMPLE_LIST;
  int* list_i = reinterpret_cast<int*>(sh_lds + 2 * SAMPLE_LIST);
  bool listed = cut_k && k <= SAMPLE_LIST && t_safe <= 4.f && !any_odd;
  if (listed) {
    sh_lds[tid] = m;
    __syncthreads();
    if (w == 0) {
      unsigned int x[SAMPLE_WAVES];
#pragma unroll
      for (int q = 0; q < SAMPLE_WAVES; ++q) x[q] = float_key(sh_lds[q * MGPT_WAVE + lane]);
      // count(key >= lo) >= k: from the smallest maximum on, if enough threads have one, to the largest (half as many rounds as over
      // all floats: 22.9 us for 23.9)
      unsigned int least = 0xffffffffu, hi = 0u;
#pragma unroll
      for (int q = 0; q < SAMPLE_WAVES; ++q) {
        least = x[q] > SAMPLE_KEY_NEG_INF && x[q] < least ? x[q] : least;
        hi = x[q] > hi ? x[q] : hi;
      }
      least = wave_min_uint(least);
      hi = ~wave_min_uint(~hi);
      unsigned int lo = wave_count(x, SAMPLE_KEY_NEG_INF + 1u) >= k ? least : SAMPLE_KEY_NEG_INF;
      while (lo < hi) {
        const unsigned int mid = lo + ((hi - lo + 1) >> 1);
        const int cnt = wave_count(x, mid);
        if (cnt >= k) {
          lo = mid;
          if (cnt <= k + (k >> 1) + 16) break;    // any bound below the k-th largest will do
        } else {
          hi = mid - 1;
        }
      }
      if (lane == 0) shared_key = lo > SAMPLE_KEY_NEG_INF + 8u ? lo - 8u : SAMPLE_KEY_NEG_INF;
    }
    __syncthreads();
    float bound = key_float(shared_key);
    int n_c = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) n_c += v[j] >= bound;            // false for NaN
    int total;
    mine_from = block_place(n_c, red_i, total);
    mine_to = mine_from + n_c;
    listed = total <= SAMPLE_LIST;
    if (listed) {
      FORGET_COMPARISONS(bound);
      int at = mine_from;
#pragma unroll
      for (int j = 0; j < K; ++j)
        if (v[j] >= bound) { list_e[at] = v[j]; list_i[at++] = i0 + j; }
      __syncthreads();
      if (tid < total) {
        const float s = list_e[tid] / t_safe;
        list_key[tid] = float_key(s);
        list_e[tid] = expf(s - mx);
      } else if (tid < ((total + 3) & ~3)) {
        list_key[tid] = 0u;
        list_e[tid] = 0.f;
      }
      __syncthreads();
      key_floor = list_floor(list_key, list_e, total, k, p, red_f, red_i);
      for (int q = mine_from; q < mine_to; ++q)
        if (list_key[q] >= key_floor) { mine += list_e[q]; last_kept = list_i[q]; }
    }
  }
  if (!listed) {
    // all keys in registers, 0 behind the stretch
#pragma unroll
    for (int j = 0; j < K; ++j) v[j] = __uint_as_float(j < n_mine ? float_key(v[j] / t_safe) : 0u);
#define HELD_KEY(j) __float_as_uint(v[j])
    if (cut_k) {
      unsigned int lo = 0u, hi = 0xffffffffu;     // count(key >= lo) >= k
      while (lo < hi) {
        const unsigned int mid = lo + (unsigned int)(((uint64_t)hi - lo + 1) >> 1);
        int cnt = 0;
#pragma unroll
        for (int j = 0; j < K; ++j) cnt += HELD_KEY(j) >= mid;
        cnt = block_sum_int(cnt, red_i);
        if (cnt >= k) lo = mid; else hi = mid - 1;
      }
      key_floor = lo > 1u ? lo : 1u;
    }
    if (p < 1.0f) {
      float z = 0.f;
      unsigned int least = 0xffffffffu;
#pragma unroll
      for (int j = 0; j < K; ++j)
        if (HELD_KEY(j) >= key_floor) {
          z += expf(key_float(HELD_KEY(j)) - mx);
          least = HELD_KEY(j) < least ? HELD_KEY(j) : least;
        }
      z = block_sum(z, red_f);
      FORGET_COMPARISONS(key_floor);
      least = block_min_uint(least, (unsigned int*)red_i);
      const float budget = p * z;
      // invariant: mass(key > hi) = base <= budget; the answer lies in [lo, hi].  Halved by value, so that the
      // undecided logits become few soon; by key after forty rounds, which ends whatever the values are.
      unsigned int lo = least != 0xffffffffu && least > key_floor ? least : key_floor, hi = float_key(mx);
      float base = 0.f;
      int left = nv;
      for (int round = 0; lo < hi && left > SAMPLE_LIST; ++round) {
        unsigned int mid = float_key(0.5f * key_float(lo) + 0.5f * key_float(hi));
        if (round >= 40 || mid < lo || mid >= hi) mid = lo + ((hi - lo) >> 1);
        float g = 0.f;
        int above = 0, below = 0;
#pragma unroll
        for (int j = 0; j < K; ++j) {
          FORGET_COMPARISONS(v[j]);               // nor are the fifty masses carried through the loop
          const unsigned int key = HELD_KEY(j);
          if (key > mid && key <= hi) { g += expf(key_float(key) - mx); ++above; }
          below += key > lo && key <= mid;
        }
        g = base + block_sum(g, red_f);
        const int counts = block_sum_int(above, red_i);
        below = block_sum_int(below, red_i);
        if (g <= budget) { hi = mid; base = g; left = below; } else { lo = mid + 1; left = counts; }
      }
      if (lo < hi) {
        int n_c = 0, total;
#pragma unroll
        for (int j = 0; j < K; ++j) n_c += HELD_KEY(j) > lo && HELD_KEY(j) <= hi;
        int at = block_place(n_c, red_i, total);   // total <= left <= SAMPLE_LIST
        FORGET_COMPARISONS(lo);
        FORGET_COMPARISONS(hi);
#pragma unroll
        for (int j = 0; j < K; ++j)
          if (HELD_KEY(j) > lo && HELD_KEY(j) <= hi && at < SAMPLE_LIST) list_key[at++] = HELD_KEY(j);
        __syncthreads();
        if (w == 0) {
          unsigned int x[SAMPLE_HELD];
          float e[SAMPLE_HELD];
#pragma unroll
          for (int q = 0; q < SAMPLE_HELD; ++q) {
            x[q] = 0u;
            e[q] = 0.f;
            if (q * MGPT_WAVE + lane < total) {
              x[q] = list_key[q * MGPT_WAVE + lane];
              e[q] = expf(key_float(x[q]) - mx);
            }
          }
          lo = wave_top_p(x, e, lo, hi, base, budget);
          if (lane == 0) shared_key = lo;
        }
        __syncthreads();
        lo = shared_key;
      }
      key_floor = lo;
    }
    FORGET_COMPARISONS(key_floor);
#pragma unroll
    for (int j = 0; j < K; ++j) {
      FORGET_COMPARISONS(v[j]);
      if (HELD_KEY(j) >= key_floor) { mine += expf(key_float(HELD_KEY(j)) - mx); last_kept = i0 + j; }
    }
  }

  // inverse CDF in vocabulary order over what is kept, the sums in the order of the kernel above: within a stretch,
  // over a wave's stretches one after the other (which keeps the prefix sums monotone), over the waves
  float run = 0.f, before = 0.f;                   // before: the wave's stretches below this one
  if (__ballot(mine != 0.f)) {
#pragma unroll
    for (int i = 0; i < MGPT_WAVE; ++i) {
      before = lane == i ? run : before;
      run += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(mine), i));
    }
  }
  int lk = last_kept;
  for (int off = 32; off > 0; off >>= 1) lk = max(lk, __shfl_xor(lk, off, MGPT_WAVE));
  __syncthreads();
  if (lane == 0) { red_f[w] = run; red_i[w] = lk; }
  if (tid == 0) chosen = 0x7fffffff;
  __syncthreads();
  float off_w = 0.f, total = 0.f;
#pragma unroll
  for (int i = 0; i < SAMPLE_WAVES; ++i) {
    if (i == w) off_w = total;
    total += red_f[i];
  }
  const float target = u * total;
  const float excl = lane ? off_w + before : off_w, incl = off_w + (before + mine);
  if (mine > 0.f && excl <= target && target < incl) {
    FORGET_COMPARISONS(key_floor);
    float sum = excl;
    int pick = 0x7fffffff;
    if (listed) {
      for (int q = mine_from; q < mine_to && pick == 0x7fffffff; ++q)
        if (list_key[q] >= key_floor) {
          sum += list_e[q];
          if (sum > target) pick = list_i[q];
        }
    } else {
#pragma unroll
      for (int j = 0; j < K; ++j) {
        FORGET_COMPARISONS(v[j]);
        if (HELD_KEY(j) >= key_floor) {
          sum += expf(key_float(HELD_KEY(j)) - mx);
          if (pick == 0x7fffffff && sum > target) pick = i0 + j;
        }
      }
    }
    atomicMin(&chosen, pick == 0x7fffffff ? last_kept : pick);
  }
#undef HELD_KEY
  __syncthreads();
  if (tid == SAMPLE_SCOUT) {
    int c = chosen;
    if (c == 0x7fffffff) {                         // rounding can leave target >= total: then the last kept id stands
      c = 0;
      for (int i = 0; i < SAMPLE_WAVES; ++i) c = max(c, red_i[i]);
    }
    finish_row(row, c, kept_out, kept_adv, kept_ahead);
  }
}

// logits: [n_rows, vocab] floats with row stride ld.  top_k (0 = off), top_p (1 = off),
// request_seed and out_index may be null.  tile_best, tile_best_idx [n_rows][n_tiles] (optional): what
// mgpt_linear_head_best left beside these logits with best_limit = real_vocab; greedy rows then read
// those instead of the logits.
static int launch_sample(const float* logits, long ld, int n_rows, int vocab, int real_vocab,
                         const float* temperature, const int* top_k, const float* top_p,
                         const uint64_t* request_seed, const int* out_index, uint64_t engine_seed,
                         int* out_tokens, const AdvanceArgs& adv, const float* tile_best,
                         const int* tile_best_idx, int n_tiles, hipStream_t stream) {
  if (n_rows == 0) return MGPT_OK;
  if (!logits || !temperature || !out_tokens) return MGPT_ERR_NULL;
  if (n_rows < 0 || vocab <= 0 || real_vocab <= 0 || ld < vocab) return MGPT_ERR_BAD_SHAPE;
  if (tile_best && (!tile_best_idx || n_tiles <= 0)) return MGPT_ERR_BAD_SHAPE;
  const int per = ((real_vocab < vocab ? real_vocab : vocab) + SAMPLE_THREADS - 1) / SAMPLE_THREADS;
#define SAMPLE_LAUNCH(KERNEL, BYTES)                                                                                   \
  hipLaunchKernelGGL(KERNEL, dim3(n_rows), dim3(SAMPLE_THREADS), BYTES, stream, logits, ld, vocab, real_vocab,         \
                     temperature, top_k, top_p, request_seed, out_index, engine_seed, out_tokens, adv, tile_best,      \
                     tile_best_idx, n_tiles)
#define SAMPLE_LAUNCH_HELD(K)                                                                                          \
  {                                                                                                                    \
    constexpr int words = SAMPLE_WAVES * (32 * K + K / 2 + 1) + 2 * MGPT_WAVE;                                         \
    constexpr int bytes = (words > 3 * SAMPLE_LIST ? words : 3 * SAMPLE_LIST) * (int)sizeof(float);                    \
    static_assert(bytes <= 160 * 1024 && bytes >= 3 * SAMPLE_LIST * 4, "a workgroup's LDS");                           \
    static bool allowed = false; /* more LDS than a kernel gets without asking */                                      \
    if (!allowed) {                                                                                                    \
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(sample_held_kernel<K>),                   \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, bytes);                     \
      if (e != hipSuccess) return (int)e;                                                                              \
      allowed = true;                                                                                                  \
    }                                                                                                                  \
    SAMPLE_LAUNCH(sample_held_kernel<K>, bytes);                                                                       \
  }
  // a thread's stretch fits its registers up to 64 logits (a vocabulary of 65,536); longer rows are read again and again
  if (per <= 4) SAMPLE_LAUNCH_HELD(4)
  else if (per <= 16) SAMPLE_LAUNCH_HELD(16)
  else if (per <= 32) SAMPLE_LAUNCH_HELD(32)
  else if (per <= 52) SAMPLE_LAUNCH_HELD(52)
  else if (per <= 64) SAMPLE_LAUNCH_HELD(64)
  else SAMPLE_LAUNCH(sample_kernel, 0);
#undef SAMPLE_LAUNCH_HELD
#undef SAMPLE_LAUNCH
  return mgpt_last_error();
}

extern "C" int mgpt_sample(const float* logits, long ld, int n_rows, int vocab, int real_vocab,
                           const float* temperature, const int* top_k, const float* top_p,
                           const uint64_t* request_seed, const int* out_index, uint64_t engine_seed,
                           int* out_tokens, const float* tile_best, const int* tile_best_idx, int n_tiles,
                           hipStream_t stream) {
  AdvanceArgs adv = {};
  return launch_sample(logits, ld, n_rows, vocab, real_vocab, temperature, top_k, top_p, request_seed,
                       out_index, engine_seed, out_tokens, adv, tile_best, tile_best_idx, n_tiles, stream);
}

// mgpt_sample, then each row prepares the next decode step on the device (AdvanceArgs above).
// Rows are requests: n_rows <= n_stride, r_stride.
extern "C" int mgpt_sample_advance(const float* logits, long ld, int n_rows, int vocab, int real_vocab,
                                   const float* temperature, const int* top_k, const float* top_p,
                                   const uint64_t* request_seed, int* out_index, uint64_t engine_seed,
                                   int* out_tokens, int* token_ids, int* positions, int* seq_lens,
                                   const int* q_req, int* slot_mapping, const int* block_tables,
                                   const int* page_sizes, int n_groups, int n_stride, int r_stride,
                                   int max_blocks, int* history, int* history_pos, int history_rows,
                                   int history_stride, const float* tile_best, const int* tile_best_idx,
                                   int n_tiles, hipStream_t stream) {
  if (!token_ids || !positions || !seq_lens || !out_index || !q_req || !slot_mapping || !block_tables ||
      !page_sizes || !history || !history_pos)
    return MGPT_ERR_NULL;
  if (n_groups <= 0 || n_rows > n_stride || n_rows > r_stride || max_blocks <= 0 || history_rows <= 0 ||
      history_stride < n_rows)
    return MGPT_ERR_BAD_SHAPE;
  AdvanceArgs adv = {token_ids, positions, seq_lens, out_index, q_req, slot_mapping, block_tables, page_sizes,
                     n_groups, n_stride, r_stride, max_blocks, history, history_pos, history_rows, history_stride};
  return launch_sample(logits, ld, n_rows, vocab, real_vocab, temperature, top_k, top_p, request_seed,
                       out_index, engine_seed, out_tokens, adv, tile_best, tile_best_idx, n_tiles, stream);
}
