// Linear attention with a fixed decay per head: a mixer whose memory is one float32 matrix per
// request and head instead of a cache of keys and values.
//
//   S_t = decay_h S_(t-1) + k_t v_t^T      (S: [D, E], zero before a request's first token)
//   o_t = S_t^T q_t
//
// q, k [H, D] and v [H, E] of a token lie in one row of `z` (the output of the stacked projection),
// in the compute dtype.  On their way in they may pass an activation (silu), q and k a rotation by
// position (pairs (i, i + rot_dims/2), angle position * freq[i], all float32), and k a constant
// scale.  Everything from there on is float32: the state, its decay, the products that enter it and
// the output.  On the way out a head's output may be divided by its root mean square (eps inside
// the root) and multiplied by silu(gate); the result is stored as float32 or in the compute dtype.
//
// One workgroup per (request, head) walks the request's tokens of this step in order, whatever
// their number (a prompt, a portion of one, one decoded token), from the state that the step
// before left in the request's slot, and leaves the new state there.  The state lives in
// registers: thread (dg, e) owns S[d][e] for d = dg, dg + NG, ... (256 threads a workgroup, or 1,024 for a
// large state, so that a thread's share stays small); the tokens' q, k, v are staged
// through LDS eight at a time, and the partial sums over dg meet there once per eight tokens.
#include "common.h"
#include "dtype_io.h"
#include "launchers.h"

#define DS_MAX 256  // largest D and E
#define DS_TC 8     // tokens staged at once

__device__ __forceinline__ float ds_act(float v, int act) { return act == 1 ? v / (1.0f + expf(-v)) : v; }

// The end of a phase: what the workgroup wrote to LDS is there; loads from memory stay on their way, which __syncthreads() would wait for.
__device__ __forceinline__ void ds_meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// R: state values a thread; NT: threads a workgroup; T: the storage type of z (with a type chosen at run time every load is waited for by
// itself).
//
// A request's single token (every request of a decode step) takes three phases between two barriers, with everything that it reads on its
// way at once: the state, the gate, and for each work item of the inputs (a rotated pair of channels of q and k, a channel that is not
// rotated, a value) what that needs.  What bounds it is that chain of latencies: the walk below reads queries, keys, values,
// angles and the gate one behind the other.  8 requests x 8 heads of 128 x 128 with norm and gate: 11.1 us by that walk, so 7.7.
template <int R, int NT, typename T>
__global__ __launch_bounds__(NT) void decay_state_kernel(
    const T* __restrict__ z, long ldz, int q_off, int k_off, int v_off, int g_off, int n_head, int D, int E,
    int act, const int* __restrict__ positions, const float* __restrict__ freq, int rot_dims, float k_scale,
    const float* __restrict__ decay, float* __restrict__ state, const int* __restrict__ state_slots,
    const int* __restrict__ cu_q, float norm_eps, void* __restrict__ out, int out_dtype, long ldo) {
  __shared__ float q_s[DS_TC][DS_MAX], k_s[DS_TC][DS_MAX], v_s[DS_TC][DS_MAX], red[DS_TC][NT];
  const int r = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int slot = state_slots[r];
  const int t_begin = cu_q[r], t_end = cu_q[r + 1];
  if (slot < 0 || t_end <= t_begin) return;     // a request of the padding
  const int NG = NT / E < D ? NT / E : D;       // groups of threads over d (at least 1: E <= 256)
  const bool owner = tid < NG * E;
  const int e = tid % E, dg = tid / E;
  const int count = owner ? (D - dg + NG - 1) / NG : 0;
  const float lambda = decay[h];
  float S[R];
  float* st = state + ((long)slot * n_head + h) * (long)D * E;
  const int first_pos = positions[t_begin];
  const bool fresh = first_pos == 0;            // the request's first token: its state starts at zero
  const int half = rot_dims / 2;
  const int wave = tid >> 6, lane = tid & 63;

  // All of a few values are on their way at once, and chosen from later; many one behind the other (4 heads of 256 x 256, 64 values a
  // thread: 29 us a token, chosen from later 64).
  // Of large states with more than a workgroup a compute unit bytes count for more than the wait for the position, and a new request's are
  // left alone.  us, always loaded / so: 128 new requests x 8 heads of 128 x 128 36.2 / 21.9, x 16 59.6 / 37.1, 32 x 16 17.2 / 13.8; 128 that
  // are not new x 8 36.2 / 32.6, 8 requests x 8 8.1 / 7.1 (the same loads, in a branch); 32 requests of 3 tokens x 16 22.4 / 22.8.
  if constexpr (R == 16) {
    bool leave = false;
    if (gridDim.x * gridDim.y > 256) {
      int first = first_pos;
      asm volatile("" : "+s"(first));             // (waited for here only)
      leave = first == 0;
    }
    if (leave) {
#pragma unroll
      for (int j = 0; j < R; ++j) S[j] = 0.f;
    } else {
#pragma unroll
      for (int j = 0; j < R; ++j) S[j] = j < count ? st[(long)(dg + j * NG) * E + e] : 0.f;
    }
  } else if constexpr (R < 16) {
#pragma unroll
    for (int j = 0; j < R; ++j) S[j] = j < count ? st[(long)(dg + j * NG) * E + e] : 0.f;
  } else {
#pragma unroll
    for (int j = 0; j < R; ++j) S[j] = (j < count && !fresh) ? st[(long)(dg + j * NG) * E + e] : 0.f;
  }
  if (R <= 16 && t_end - t_begin == 1) {       // (more values a thread leave no registers for it)
    const T* row = z + (long)t_begin * ldz;
    constexpr int GATES = DS_MAX / 64;
    T gate[GATES];
    if (wave == 0 && g_off >= 0) {
#pragma unroll
      for (int m = 0; m < GATES; ++m) gate[m] = row[g_off + (long)h * E + (lane + 64 * m < E ? lane + 64 * m : 0)];
    }
    const int plain = half + (D - rot_dims);    // rotated pairs, then single channels of q and k, then values
    for (int i = tid; i < plain + E; i += NT) {
      if (i < plain) {
        const int d = i < half ? i : i + half;
        const T* q = row + q_off + (long)h * D + d;
        const T* k = row + k_off + (long)h * D + d;
        const int other = i < half ? half : 0;
        const T q0 = q[0], k0 = k[0], q1 = q[other], k1 = k[other];
        const float f = i < half ? freq[i] : 0.f;
        const float qu = ds_act(to_float<T>(q0), act), ku = ds_act(to_float<T>(k0), act);
        if (i < half) {
          const float qw = ds_act(to_float<T>(q1), act), kw = ds_act(to_float<T>(k1), act);
          const float a = (float)first_pos * f;
          const float co = cosf(a), si = sinf(a);
          q_s[0][d] = qu * co - qw * si;
          q_s[0][d + half] = qw * co + qu * si;
          k_s[0][d] = (ku * co - kw * si) * k_scale;
          k_s[0][d + half] = (kw * co + ku * si) * k_scale;
        } else {
          q_s[0][d] = qu;
          k_s[0][d] = ku * k_scale;
        }
      } else {
        v_s[0][i - plain] = ds_act(to_float<T>(row[v_off + (long)h * E + (i - plain)]), act);
      }
    }
    ds_meet();
    if (owner) {
      const float ve = v_s[0][e];
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < R; ++j) {
        if (j < count) {
          const int d = dg + j * NG;
          const float was = fresh ? 0.f : S[j];
          S[j] = fmaf(lambda, was, k_s[0][d] * ve);
          acc = fmaf(S[j], q_s[0][d], acc);
        }
      }
      red[0][tid] = acc;
    }
    ds_meet();
    if (wave == 0) {                            // the sums over dg in order, the head's norm, the gate, the store
      float o[GATES], ss = 0.f;
#pragma unroll
      for (int m = 0; m < GATES; ++m) {
        const int c = lane + 64 * m;
        o[m] = 0.f;
        if (c < E) {
          for (int g = 0; g < NG; ++g) o[m] += red[0][g * E + c];
          ss = fmaf(o[m], o[m], ss);
        }
      }
      float scale = 1.0f;
      if (norm_eps >= 0.f) scale = 1.0f / sqrtf(wave_sum(ss) / (float)E + norm_eps);
#pragma unroll
      for (int m = 0; m < GATES; ++m) {
        const int c = lane + 64 * m;
        float v = o[m] * scale;
        if (g_off >= 0) {
          const float g = to_float<T>(gate[m]);
          v *= g / (1.0f + expf(-g));
        }
        if (c < E) store_f(out, out_dtype, (long)t_begin * ldo + (long)h * E + c, v);
      }
    }
#pragma unroll
    for (int j = 0; j < R; ++j)
      if (j < count) st[(long)(dg + j * NG) * E + e] = S[j];
    return;
  }
  if constexpr (R <= 16) {
#pragma unroll
    for (int j = 0; j < R; ++j) S[j] = fresh ? 0.f : S[j];
  }

  for (int t0 = t_begin; t0 < t_end; t0 += DS_TC) {
    const int nt = t_end - t0 < DS_TC ? t_end - t0 : DS_TC;
    __syncthreads();     // the chunk before is read
    for (int i = tid; i < nt * D; i += NT) {
      const int tt = i / D, d = i - tt * D;
      const long row = (long)(t0 + tt) * ldz + (long)h * D + d;
      q_s[tt][d] = ds_act(to_float<T>(z[row + q_off]), act);
      k_s[tt][d] = ds_act(to_float<T>(z[row + k_off]), act);
    }
    for (int i = tid; i < nt * E; i += NT) {
      const int tt = i / E, c = i - tt * E;
      v_s[tt][c] = ds_act(to_float<T>(z[(long)(t0 + tt) * ldz + v_off + (long)h * E + c]), act);
    }
    __syncthreads();
    if (freq) {
      for (int i = tid; i < nt * half; i += NT) {
        const int tt = i / half, c = i - tt * half;
        const float a = (float)positions[t0 + tt] * freq[c];
        const float co = cosf(a), si = sinf(a);
        const float qu = q_s[tt][c], qw = q_s[tt][c + half], ku = k_s[tt][c], kw = k_s[tt][c + half];
        q_s[tt][c] = qu * co - qw * si;
        q_s[tt][c + half] = qw * co + qu * si;
        k_s[tt][c] = (ku * co - kw * si) * k_scale;
        k_s[tt][c + half] = (kw * co + ku * si) * k_scale;
      }
      if (k_scale != 1.0f)
        for (int i = tid; i < nt * (D - rot_dims); i += NT) {
          const int tt = i / (D - rot_dims), c = rot_dims + i - tt * (D - rot_dims);
          k_s[tt][c] *= k_scale;
        }
    } else if (k_scale != 1.0f) {
      for (int i = tid; i < nt * D; i += NT) k_s[i / D][i % D] *= k_scale;
    }
    __syncthreads();
    if (owner) {
      for (int tt = 0; tt < nt; ++tt) {
        const float ve = v_s[tt][e];
        float acc = 0.f;
#pragma unroll
        for (int j = 0; j < R; ++j) {
          if (j < count) {
            const int d = dg + j * NG;
            S[j] = fmaf(lambda, S[j], k_s[tt][d] * ve);
            acc = fmaf(S[j], q_s[tt][d], acc);
          }
        }
        red[tt][tid] = acc;
      }
    }
    __syncthreads();
    // a wave a token: the sums over dg in order, the head's norm, the gate, the store
    for (int tt = wave; tt < nt; tt += NT / 64) {
      float ss = 0.f;
      for (int c = lane; c < E; c += 64) {
        float o = 0.f;
        for (int g = 0; g < NG; ++g) o += red[tt][g * E + c];
        red[tt][c] = o;
        ss = fmaf(o, o, ss);
      }
      float scale = 1.0f;
      if (norm_eps >= 0.f) scale = 1.0f / sqrtf(wave_sum(ss) / (float)E + norm_eps);
      const long n = t0 + tt;
      for (int c = lane; c < E; c += 64) {
        float o = red[tt][c] * scale;
        if (g_off >= 0) {
          const float g = to_float<T>(z[n * ldz + g_off + (long)h * E + c]);
          o *= g / (1.0f + expf(-g));
        }
        store_f(out, out_dtype, n * ldo + (long)h * E + c, o);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < R; ++j)
    if (j < count) st[(long)(dg + j * NG) * E + e] = S[j];
}

// z: [n_tokens, ldz] rows in `dtype`; q at q_off, k at k_off, v at v_off, the gate at g_off (-1: none), head by head.
// state: [slots, n_head * D * E] float32; state_slots[r] the slot of request r (-1: none), cu_q its tokens.
extern "C" int mgpt_decay_state(const void* z, int dtype, long ldz, int q_off, int k_off, int v_off, int g_off, int n_head,
                                int head_dim, int value_dim, int act, const int* positions, const float* freq,
                                int rot_dims, float k_scale, const float* decay, float* state, const int* state_slots,
                                const int* cu_q, int n_req, float norm_eps, void* out, int out_dtype, long ldo,
                                hipStream_t stream) {
  if (n_req == 0) return MGPT_OK;
  if (!z || !positions || !decay || !state || !state_slots || !cu_q || !out) return MGPT_ERR_NULL;
  if (!dtype_ok(dtype) || !dtype_ok(out_dtype)) return MGPT_ERR_BAD_DTYPE;
  const int D = head_dim, E = value_dim;
  if (n_req < 0 || n_head <= 0 || D <= 0 || E <= 0 || D > DS_MAX || E > DS_MAX || rot_dims < 0 || (rot_dims & 1) ||
      rot_dims > D || (act != 0 && act != 1))
    return MGPT_ERR_BAD_SHAPE;
  if (n_head > 65535) return MGPT_ERR_TOO_LARGE;
  // a workgroup of 256 threads while a thread then owns at most 16 values of the state, else one of 1,024
  auto per_thread = [&](int threads) {
    const int ng = threads / E < D ? threads / E : D;
    return (D + ng - 1) / ng;
  };
  dim3 grid(n_req, n_head);
  if (!freq) rot_dims = 0;
#define DS_LAUNCH_AS(R, NT, T)                                                                                             \
  hipLaunchKernelGGL((decay_state_kernel<R, NT, T>), grid, dim3(NT), 0, stream, (const T*)z, ldz, q_off, k_off, v_off, g_off,   \
                     n_head, D, E, act, positions, rot_dims ? freq : nullptr, rot_dims, k_scale, decay, state, state_slots, \
                     cu_q, norm_eps, out, out_dtype, ldo)
#define DS_LAUNCH(R, NT)                                                                                                   \
  do {                                                                                                                     \
    if (dtype == MGPT_F32) DS_LAUNCH_AS(R, NT, float);                                                                     \
    else DS_LAUNCH_AS(R, NT, bf16_t);                                                                                      \
  } while (0)
  if (per_thread(256) <= 8) DS_LAUNCH(8, 256);
  else if (per_thread(256) <= 16) DS_LAUNCH(16, 256);
  else if (per_thread(1024) <= 16) DS_LAUNCH(16, 1024);
  else if (per_thread(1024) <= 32) DS_LAUNCH(32, 1024);
  else if (per_thread(1024) <= 64) DS_LAUNCH(64, 1024);
  else return MGPT_ERR_BAD_SHAPE;
#undef DS_LAUNCH
#undef DS_LAUNCH_AS
  return mgpt_last_error();
}

// ---------------------------------------------------------------------------------------------
// Prompt portions: the same recurrence a chunk of 32 tokens at a time, as matrix products on the
// float32 matrix cores (v_mfma_f32_16x16x4_f32: true 32-bit products and sums).  For a chunk whose
// tokens have in-chunk indices i = 0 .. n-1, with L = decay:
//   P[i][j] = (q_i . k_j) L^(i-j) for j <= i, else 0
//   o_i     = sum_j P[i][j] v_j + L^(i+1) S^T q_i
//   S      <- L^n S + sum_j L^(n-1-j) k_j v_j^T
// A workgroup owns (request, head, 32 or 16 value channels): the columns of S are independent of each
// other, so a head's value channels are dealt out over workgroups, each of which makes P for itself.
// Queries and keys come ready (activation, rotation, scale) as float32 from state_inputs_kernel.

#define DC_C 32        // tokens a chunk
#define DC_DMAX 128    // largest head size of this path
#define DC_LDP (DC_C + 4)

typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T>
__global__ __launch_bounds__(256) void state_inputs_kernel(const T* __restrict__ z, long ldz, int q_off,
                                                           int k_off, int n_head, int D, int act,
                                                           const int* __restrict__ positions, const float* __restrict__ freq,
                                                           int rot_dims, float k_scale, float* __restrict__ qk, int n_tokens) {
  __shared__ float cos_s[DS_MAX / 2], sin_s[DS_MAX / 2];
  const int n = blockIdx.x, half = rot_dims / 2;
  if (freq) {
    const float p = (float)positions[n];
    for (int i = threadIdx.x; i < half; i += 256) {
      const float a = p * freq[i];
      cos_s[i] = cosf(a);
      sin_s[i] = sinf(a);
    }
  }
  __syncthreads();
  const int HD = n_head * D;
  float* dst = qk + (long)n * 2 * HD;
  // thread: one channel of one head; a rotated pair is made by the thread of its first channel
  for (int i = threadIdx.x; i < HD; i += 256) {
    const int d = i % D;
    if (d >= half && d < rot_dims) continue;
    const long at = (long)n * ldz + i;
    const int other = d < half ? half : 0;
    const T q0 = z[at + q_off], k0 = z[at + k_off], q1 = z[at + other + q_off], k1 = z[at + other + k_off];
    float q = ds_act(to_float<T>(q0), act), k = ds_act(to_float<T>(k0), act);
    if (d < half) {
      const float q2 = ds_act(to_float<T>(q1), act), k2 = ds_act(to_float<T>(k1), act);
      const float co = cos_s[d], si = sin_s[d];
      dst[i + half] = q2 * co + q * si;
      dst[HD + i + half] = (k2 * co + k * si) * k_scale;
      const float qr = q * co - q2 * si, kr = k * co - k2 * si;
      q = qr;
      k = kr;
    }
    dst[i] = q;
    dst[HD + i] = k * k_scale;
  }
}

// A request's chunks are a chain, 3 to 4 us each, and a step of few long prompts has few chains: 8 requests x 8 heads with the
// longest of 1,024 tokens take 129 us, 32 chunks one behind the other.  With scratch for them the requests are cut into segments
// of 256 tokens instead (numbered over the requests one behind the other): a first launch makes, for all segments but a request's
// last, what the segment adds to the state (sum_t L^(n-1-t) k_t v_t^T, a third of a chunk's work; the first segment starts from
// the request's state and so leaves the state behind it, and copies that state to the last segment's place, where nobody adds);
// a second launch puts a segment's starting state together from those before it, S <- L^256 S + added, and runs its chunks.
// 103 us there.  The caller decides where that is less (a chunk's work is then done 1.4 times, so not where the chains fill the
// chip).  Error against 64 bits over 1,024 tokens: 2.1e-7 either way.
//
// What bounds a chunk: 104 matrix instructions a wave (1.5 us), four barriers, and three workgroups a compute unit to cover each
// other's waits.  With the state in LDS (two workgroups a unit), the pieces' places divided out anew for every chunk, and barriers
// that waited for the next chunk's loads (which came one by one, their type being chosen at run time) these took 239 us whole and
// 202 cut, error 2.5e-7; 2 x 1,024 tokens x 8 heads 180 / 129, now 102 / 81; one of 2,048 x 16 heads 342 / 159, now 195 / 91.
#define DC_SEGMENT 256
#define DC_WHOLE 0      // a request's chunks one behind the other
#define DC_ADDED 1      // what the segments add
#define DC_OUTPUTS 2    // the segments' outputs, and the last one's state

// EB: value channels a workgroup: 32, or 16 where that is what fills the machine.  DL: the head's channels as they are staged and
// multiplied, those beyond D as zeros (64 or 128: a bound known when compiling, so that the products are straight-line code and a
// piece's place costs no division).  V: queries and keys in pieces of V channels (4: head sizes that are multiples of four).  T: the
// storage type of z.  added: [segments][n_head][E][Dp].
template <int EB, int MODE, int DL, int V, typename T>
__global__ __launch_bounds__(256, V == 1 && DL == 128 ? 1 : MODE == DC_ADDED ? 4 : 3) void decay_state_chunk_kernel(
    const float* __restrict__ qk, const T* __restrict__ z, long ldz, int v_off, int n_head, int D, int E,
    int act, const int* __restrict__ positions, const float* __restrict__ decay, float* __restrict__ state,
    const int* __restrict__ state_slots, const int* __restrict__ cu_q, float* __restrict__ out, long ldo, int n_req,
    float* __restrict__ added) {
  constexpr int NJ = EB / 16;                   // column tiles of the workgroup's value channels
  constexpr int PARTS = 4 / NJ, TILES = DL / 16 / PARTS;
  // Queries and keys [token][d]; the values transposed, [value channel][token]; P [token][token].  Every product's index of
  // summation runs along a row, so that a lane's operands of four matrix instructions are one 16-byte read: instruction s of
  // such a group takes k = k0 + 4 g + s from lane (r16, g) (any dealing of a stretch's 16 values of k over four instructions
  // gives the same sum, if both operands agree).  The state stays in registers: what a lane holds of a sum's 16 x 16 tile,
  // rows 4 g .. 4 g + 3 of column r16, is what it must bring of the state as the second operand of Q S.  Wave (part, sj) has
  // column tile sj and the rows' tiles part, part + PARTS, ...; Q S is the sum of the PARTS waves' shares, which meet in LDS.
  // (With the state in LDS a workgroup took 60 KB, two a compute unit, here 51.)
  __shared__ __attribute__((aligned(16))) float Qs[DC_C][DL + 4], Ks[DC_C][DL + 4], Vt[EB][DC_LDP], Ps[DC_C][DC_LDP],
      share[PARTS][2][NJ][256];
  __shared__ float pw[DC_C + 1];
  const int h = blockIdx.y, e0 = blockIdx.z * EB, tid = threadIdx.x;
  const int wave = tid >> 6, lane = tid & 63, r16 = lane & 15, g = lane >> 4;
  int r = blockIdx.x, seg = 0, first = 0;       // the request, its segment, the number of its first segment
  if (MODE != DC_WHOLE) {
    seg = blockIdx.x;
    r = piece_owner(n_req, seg, [&](int i) { return (cu_q[i + 1] - cu_q[i] + DC_SEGMENT - 1) / DC_SEGMENT; });
    if (r < 0) return;                          // beyond the step's segments: the whole workgroup
    first = (int)blockIdx.x - seg;
  }
  const int slot = state_slots[r];
  int t_begin = cu_q[r], t_end = cu_q[r + 1];
  if (slot < 0 || t_end <= t_begin) return;     // a request of the padding
  const int n_seg = (t_end - t_begin + DC_SEGMENT - 1) / DC_SEGMENT;
  if (MODE == DC_ADDED && seg == n_seg - 1) return;
  const bool fresh = positions[t_begin] == 0;
  if (MODE != DC_WHOLE) {
    t_begin += seg * DC_SEGMENT;
    if (seg != n_seg - 1) t_end = t_begin + DC_SEGMENT;
  }
  const int Dp = (D + 15) & ~15;                // rows of S and steps along d, padded with zeros
  const int HD = n_head * D;
  const float lambda = decay[h];
  const float log_l = logf(lambda);
  if (tid <= DC_C) pw[tid] = tid == 0 ? 1.0f : expf((float)tid * log_l);
  float* st = state + ((long)slot * n_head + h) * (long)D * E;
  // a segment's place in `added`, and its row of value channel e0 + c
  auto place = [&](int number, int c) { return added + (((long)number * n_head + h) * E + e0 + c) * Dp; };
  const int sj = wave % NJ, part = wave / NJ, d_tiles = Dp >> 4;
  const int mine = sj * 16 + r16;               // this lane's value channel
  f32x4_t S[TILES];
  // the state is read with its last row or column in place of those that are not there
  const int there = e0 + mine < E ? mine : 0;
  const float across = expf((float)DC_SEGMENT * log_l);
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int d0 = (part + PARTS * i) * 16 + 4 * g;
    S[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (part + PARTS * i >= d_tiles) continue;  // the same in all lanes
    if (MODE == DC_OUTPUTS && n_seg > 1) {
      const float* p = place(seg == 0 ? first + n_seg - 1 : first, there) + d0;
#pragma unroll
      for (int v = 0; v < 4; ++v) S[i][v] = p[v];
      for (int j = 1; j < seg; ++j) {
        const float* add = place(first + j, there) + d0;
#pragma unroll
        for (int v = 0; v < 4; ++v) S[i][v] = fmaf(across, S[i][v], add[v]);
      }
    } else if (!(fresh || (MODE == DC_ADDED && seg > 0))) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float was = st[(long)(d0 + v < D ? d0 + v : D - 1) * E + e0 + there];
        S[i][v] = d0 + v < D ? was : 0.f;
      }
    }
    if (e0 + mine >= E) S[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    if (MODE == DC_ADDED && seg == 0 && e0 + mine < E) {
      float* p = place(first + n_seg - 1, mine) + d0;
#pragma unroll
      for (int v = 0; v < 4; ++v) p[v] = S[i][v];
    }
  }
  const int ti = wave >> 1, tj = wave & 1;      // this wave's 16 x 16 tile of P and of the chunk's outputs

  // A chunk's rows travel from memory into registers while the chunk before is multiplied: thread tid holds
  // pieces tid, tid + 256, ... of the chunk's [32, Dp] queries and keys and elements of its [32, EB] values.
  typedef float piece_t __attribute__((ext_vector_type(V)));
  constexpr int PER_ROW = DL / V, QK_PT = DC_C * PER_ROW / 256, V_PT = DC_C * EB / 256;
  piece_t q_r[QK_PT], k_r[QK_PT];
  T v_r[V_PT];
  // (what lies beyond the tokens or the head's channels is read from the last ones and put away as zero: no branch between the loads)
  auto fetch = [&](int t0) {
#pragma unroll
    for (int u = 0; u < QK_PT; ++u) {
      const int tt = (tid + u * 256) / PER_ROW, d = (tid + u * 256) % PER_ROW * V;
      const float* at = qk + (long)(t0 + tt < t_end ? t0 + tt : t_end - 1) * 2 * HD + (long)h * D + (d < D ? d : 0);
      if (MODE != DC_ADDED) q_r[u] = *reinterpret_cast<const piece_t*>(at);
      k_r[u] = *reinterpret_cast<const piece_t*>(at + HD);
    }
#pragma unroll
    for (int u = 0; u < V_PT; ++u) {
      const int i = tid + u * 256, tt = i / EB, c = i - tt * EB;
      v_r[u] = z[(long)(t0 + tt < t_end ? t0 + tt : t_end - 1) * ldz + v_off + (long)h * E + (e0 + c < E ? e0 + c : 0)];
    }
  };
  fetch(t_begin);

  for (int t0 = t_begin; t0 < t_end; t0 += DC_C) {
    const int nt = t_end - t0 < DC_C ? t_end - t0 : DC_C;
    ds_meet();           // the chunk before is done with the staged rows; S is whole
#pragma unroll
    for (int u = 0; u < QK_PT; ++u) {
      const int tt = (tid + u * 256) / PER_ROW, d = (tid + u * 256) % PER_ROW * V;
      const piece_t none = {};
      const bool held = tt < nt && d < D;
      if (MODE != DC_ADDED) *reinterpret_cast<piece_t*>(&Qs[tt][d]) = held ? q_r[u] : none;
      *reinterpret_cast<piece_t*>(&Ks[tt][d]) = held ? k_r[u] : none;
    }
#pragma unroll
    for (int u = 0; u < V_PT; ++u) {
      const int i = tid + u * 256, tt = i / EB, c = i - tt * EB;
      Vt[c][tt] = tt < nt && e0 + c < E ? ds_act(to_float<T>(v_r[u]), act) : 0.f;
    }
    ds_meet();
    fetch(t0 + DC_C);
    if (MODE != DC_ADDED) {
      // ---- P = Q K^T with the decay of the distance, lower triangle
      {
        f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
        if (tj <= ti) {
#pragma unroll 2
          for (int k0 = 0; k0 < DL; k0 += 16) {
            const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&Qs[ti * 16 + r16][k0 + 4 * g]);
            const f32x4_t b = *reinterpret_cast<const f32x4_t*>(&Ks[tj * 16 + r16][k0 + 4 * g]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], acc, 0, 0, 0);
          }
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = ti * 16 + 4 * g + v, j = tj * 16 + r16;
          Ps[i][j] = j <= i ? acc[v] * pw[i - j] : 0.f;
        }
      }
      ds_meet();
      // ---- o = P V + L^(i+1) Q S: wave t puts tile (oi, oj) = (t / NJ, t % NJ) of the chunk's [32, EB] outputs together
      const int oi = wave / NJ;
      f32x4_t pv = {0.f, 0.f, 0.f, 0.f}, qs[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
      if (oi < 2) {
        for (int k0 = 0; k0 < (oi + 1) * 16; k0 += 16) {
          const f32x4_t a = *reinterpret_cast<const f32x4_t*>(&Ps[oi * 16 + r16][k0 + 4 * g]);
          const f32x4_t b = *reinterpret_cast<const f32x4_t*>(&Vt[mine][k0 + 4 * g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) pv = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], b[e], pv, 0, 0, 0);
        }
      }
#pragma unroll
      for (int i = 0; i < TILES; ++i) {
        const f32x4_t a0 = *reinterpret_cast<const f32x4_t*>(&Qs[r16][(part + PARTS * i) * 16 + 4 * g]);
        const f32x4_t a1 = *reinterpret_cast<const f32x4_t*>(&Qs[16 + r16][(part + PARTS * i) * 16 + 4 * g]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          qs[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a0[e], S[i][e], qs[0], 0, 0, 0);
          qs[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a1[e], S[i][e], qs[1], 0, 0, 0);
        }
      }
#pragma unroll
      for (int o = 0; o < 2; ++o) *reinterpret_cast<f32x4_t*>(&share[part][o][sj][lane * 4]) = qs[o];
      ds_meet();
      if (oi < 2) {
        f32x4_t sum = *reinterpret_cast<const f32x4_t*>(&share[0][oi][sj][lane * 4]);
#pragma unroll
        for (int q = 1; q < PARTS; ++q) {
          const f32x4_t more = *reinterpret_cast<const f32x4_t*>(&share[q][oi][sj][lane * 4]);
#pragma unroll
          for (int v = 0; v < 4; ++v) sum[v] += more[v];
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int i = oi * 16 + 4 * g + v, c = e0 + mine;
          if (i < nt && c < E) out[(long)(t0 + i) * ldo + (long)h * E + c] = pv[v] + pw[i + 1] * sum[v];
        }
      }
    }
    // ---- S <- L^n S + sum_t k_t (L^(n-1-t) v_t)^T: the wave's tiles of the state
    f32x4_t b[DC_C / 16];
#pragma unroll
    for (int k0 = 0; k0 < DC_C; k0 += 16) {
      b[k0 / 16] = *reinterpret_cast<const f32x4_t*>(&Vt[mine][k0 + 4 * g]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int tk = k0 + 4 * g + e;
        b[k0 / 16][e] *= pw[tk < nt ? nt - 1 - tk : 0];          // (tokens that are not there: zeros already)
      }
    }
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
#pragma unroll
      for (int v = 0; v < 4; ++v) S[i][v] *= pw[nt];
    }
#pragma unroll
    for (int k0 = 0; k0 < DC_C; k0 += 16)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < TILES; ++i)
          S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ks[k0 + 4 * g + e][(part + PARTS * i) * 16 + r16], b[k0 / 16][e], S[i], 0, 0, 0);
    // (a zero key times an infinite value is a NaN, also where there is no channel; Q S adds these up as well)
#pragma unroll
    for (int i = 0; i < TILES; ++i)
      if (part + PARTS * i >= d_tiles) S[i] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  }
  if (MODE == DC_OUTPUTS && seg != n_seg - 1) return;
#pragma unroll
  for (int i = 0; i < TILES; ++i) {
    const int d0 = (part + PARTS * i) * 16 + 4 * g;
    if (part + PARTS * i >= d_tiles || e0 + mine >= E) continue;
    if (MODE == DC_ADDED) {
      float* p = place(first + seg, mine) + d0;
#pragma unroll
      for (int v = 0; v < 4; ++v) p[v] = S[i][v];
    } else {
#pragma unroll
      for (int v = 0; v < 4; ++v)
        if (d0 + v < D) st[(long)(d0 + v) * E + e0 + mine] = S[i][v];
    }
  }
}

// The chunked form for steps with prompt portions: qk is scratch, float32 [n_tokens, 2 * n_head * head_dim]; out is
// float32 [n_tokens, >= n_head * value_dim]: the heads' raw outputs (norm and gate are the caller's next kernel).
// Head sizes up to 128 (value sizes up to 256); others are refused with MGPT_ERR_BAD_SHAPE and nothing launched.  added
// (optional): scratch of added_floats floats; with it the requests are cut into segments, for which it must hold
// n_head * value_dim * (head_dim rounded up to 16) floats each, (n_tokens + 255 * min(n_req, n_tokens)) / 256 of them.
extern "C" int mgpt_decay_state_chunked(const void* z, int dtype, long ldz, int q_off, int k_off, int v_off, int n_head,
                                        int head_dim, int value_dim, int act, const int* positions, const float* freq,
                                        int rot_dims, float k_scale, const float* decay, float* state,
                                        const int* state_slots, const int* cu_q, int n_req, int n_tokens, float* qk,
                                        float* out, long ldo, float* added, long added_floats,
                                        hipStream_t stream) {
  if (n_req == 0 || n_tokens == 0) return MGPT_OK;
  if (!z || !positions || !decay || !state || !state_slots || !cu_q || !out || !qk) return MGPT_ERR_NULL;
  if (!dtype_ok(dtype)) return MGPT_ERR_BAD_DTYPE;
  const int D = head_dim, E = value_dim;
  if (n_req < 0 || n_tokens < 0 || n_head <= 0 || D <= 0 || E <= 0 || D > DC_DMAX || E > DS_MAX || rot_dims < 0 ||
      (rot_dims & 1) || rot_dims > D || (act != 0 && act != 1))
    return MGPT_ERR_BAD_SHAPE;
  if (n_head > 65535) return MGPT_ERR_TOO_LARGE;
  const long segments = ((long)n_tokens + (DC_SEGMENT - 1L) * (n_req < n_tokens ? n_req : n_tokens)) / DC_SEGMENT;
  if (added && (segments > 0x7fffffffL || added_floats < segments * n_head * E * ((D + 15) & ~15))) return MGPT_ERR_BAD_SHAPE;
  const bool vec = D % 4 == 0 && (((size_t)qk) & 15) == 0;   // (an odd number of heads of 4 x odd channels: still whole pieces)
#define DC_INPUTS(T)                                                                                                       \
  hipLaunchKernelGGL(state_inputs_kernel<T>, dim3(n_tokens), dim3(256), 0, stream, (const T*)z, ldz, q_off, k_off, n_head, D, act, \
                     positions, rot_dims ? freq : nullptr, rot_dims, k_scale, qk, n_tokens)
  if (dtype == MGPT_F32) DC_INPUTS(float);
  else DC_INPUTS(bf16_t);
#undef DC_INPUTS
  // 32 value channels a workgroup; 16 where that many workgroups would leave compute units idle
#define DC_LAUNCH_AS(EB, MODE, X, DL, V, T)                                                                                \
  hipLaunchKernelGGL((decay_state_chunk_kernel<EB, MODE, DL, V, T>), dim3((unsigned int)(X), n_head, (E + EB - 1) / EB), dim3(256), \
                     0, stream, qk, (const T*)z, ldz, v_off, n_head, D, E, act, positions, decay, state, state_slots, cu_q, out, \
                     ldo, n_req, added)
#define DC_LAUNCH(EB, MODE, X)                                                                                             \
  do {                                                                                                                     \
    if (dtype == MGPT_F32) {                                                                                               \
      if (vec && D <= 64) DC_LAUNCH_AS(EB, MODE, X, 64, 4, float);                                                              \
      else if (vec) DC_LAUNCH_AS(EB, MODE, X, 128, 4, float);                                                                        \
      else if (D <= 64) DC_LAUNCH_AS(EB, MODE, X, 64, 1, float);                                                                \
      else DC_LAUNCH_AS(EB, MODE, X, 128, 1, float);                                                                            \
    } else {                                                                                                               \
      if (vec && D <= 64) DC_LAUNCH_AS(EB, MODE, X, 64, 4, bf16_t);                                                             \
      else if (vec) DC_LAUNCH_AS(EB, MODE, X, 128, 4, bf16_t);                                                                       \
      else if (D <= 64) DC_LAUNCH_AS(EB, MODE, X, 64, 1, bf16_t);                                                               \
      else DC_LAUNCH_AS(EB, MODE, X, 128, 1, bf16_t);                                                                           \
    }                                                                                                                      \
  } while (0)
  if (added) {
    if (segments * n_head * ((E + 31) / 32) >= 256) {
      DC_LAUNCH(32, DC_ADDED, segments);
      DC_LAUNCH(32, DC_OUTPUTS, segments);
    } else {
      DC_LAUNCH(16, DC_ADDED, segments);
      DC_LAUNCH(16, DC_OUTPUTS, segments);
    }
  } else if ((long)n_req * n_head * ((E + 31) / 32) >= 256) {
    DC_LAUNCH(32, DC_WHOLE, n_req);
  } else {
    DC_LAUNCH(16, DC_WHOLE, n_req);
  }
#undef DC_LAUNCH
#undef DC_LAUNCH_AS
  return mgpt_last_error();
}
