// Draft-side tree expansion (gfx950): log-softmax + top-k of the draft logits and the
// per-level bookkeeping of generate_draft_tree (mlx_eagle.py:97-213, 410-412), kept on the
// device so that the expansion loop needs no device-to-host round trip.
//
// Scores are carried in fp16, as the reference carries them in the model dtype; every
// ordering is "larger score first, equal scores lowest index first".
#include "common.h"

#include <math.h>

namespace {

constexpr int TOPK_MAX = 8;          // k of the expansion (candidates per node)
constexpr int CHUNK = 4096;          // logits per workgroup
constexpr int THREADS = 256;

__device__ inline uint32_t wave_max(uint32_t v) {
  return wave_reduce(v, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// A candidate as one integer: its value (fp16, exactly) as an ordered integer, then its place from the back, so that
// the larger integer is the better candidate ("larger score first, equal scores lowest index first").  0: none
// (also a NaN, which is never picked).
__device__ inline uint32_t key_of(float v, int place) {
  uint32_t h = __builtin_bit_cast(unsigned short, (half_t)v);
  if (h == 0x8000u) h = 0u;
  const uint32_t key = (h & 0x8000u ? ~h & 0xffffu : h | 0x8000u) << 16 | (0xffffu - (uint32_t)place);
  return v != v ? 0u : key;
}
__device__ inline float key_value(uint32_t key) {
  const uint32_t o = key >> 16;
  return (float)__builtin_bit_cast(half_t, (unsigned short)(o & 0x8000u ? o & 0x7fffu : ~o & 0xffffu));
}
__device__ inline int key_place(uint32_t key) { return (int)(0xffffu - (key & 0xffffu)); }

// The k best of the keys that the lanes of a wave hold (N each, distinct apart from 0); lane n gets the n-th.
template <int N>
__device__ inline uint32_t wave_topk(uint32_t (&key)[N], int k) {
  const int lane = threadIdx.x & 63;
  uint32_t mine = 0;
  for (int n = 0; n < k; ++n) {
    uint32_t best = key[0];
#pragma unroll
    for (int j = 1; j < N; ++j) best = key[j] > best ? key[j] : best;
    best = wave_max(best);
#pragma unroll
    for (int j = 0; j < N; ++j) key[j] = key[j] == best ? 0u : key[j];
    if (lane == n) mine = best;
  }
  return mine;
}

__device__ inline const half_t* row_ptr(const half_t* logits, const int32_t* row_index, int row,
                                        long V) {
  const long r = row_index ? (long)row_index[row] : (long)row;
  return logits + r * V;
}

// Pass 1: per chunk, the maximum and sum of exp(x - max).  Grid (chunks, rows).
__global__ __launch_bounds__(THREADS) void lse_partial_kernel(
    const half_t* __restrict__ logits, const int32_t* __restrict__ row_index, long V,
    float* __restrict__ pm, float* __restrict__ ps) {
  __shared__ float red[THREADS / 64];
  const int row = blockIdx.y, ch = blockIdx.x, nch = gridDim.x;
  const half_t* r = row_ptr(logits, row_index, row, V);
  const long beg = (long)ch * CHUNK;
  float x[CHUNK / THREADS];
  float m = -INFINITY;
#pragma unroll
  for (int j = 0; j < CHUNK / THREADS; ++j) {
    const long i = beg + threadIdx.x + (long)j * THREADS;
    x[j] = i < V ? (float)r[i] : -INFINITY;
    m = fmaxf(m, x[j]);
  }
  m = wave_max(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float s = 0.f;
#pragma unroll
  for (int j = 0; j < CHUNK / THREADS; ++j) s += x[j] == -INFINITY ? 0.f : expf(x[j] - m);
  s = wave_sum(s);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    pm[row * nch + ch] = m;
    ps[row * nch + ch] = (red[0] + red[1]) + (red[2] + red[3]);
  }
}

// Row statistics from the partials, the same arithmetic in every workgroup that needs them: the terms of the sum in
// parallel, the sum itself over the chunks in order.  shared: STATS floats.
constexpr int STATS = 256;
__device__ inline void row_stats(const float* pm, const float* ps, int row, int nch, float* shared, float* M, float* S) {
  const float *rm = pm + row * nch, *rs = ps + row * nch;
  float m = -INFINITY, s = 0.f;
  if (nch > STATS) {
    for (int c = 0; c < nch; ++c) m = fmaxf(m, rm[c]);
    for (int c = 0; c < nch; ++c)
      if (rm[c] != -INFINITY) s += rs[c] * expf(rm[c] - m);
  } else {
    const int lane = threadIdx.x & 63;
    float v[STATS / 64], t[STATS / 64];
#pragma unroll
    for (int j = 0; j < STATS / 64; ++j) {
      const int c = lane + 64 * j;
      v[j] = c < nch ? rm[c] : -INFINITY;
      t[j] = c < nch ? rs[c] : 0.f;
      m = fmaxf(m, v[j]);
    }
    m = wave_max(m);
#pragma unroll
    for (int j = 0; j < STATS / 64; ++j)             // (every wave writes the same values)
      shared[lane + 64 * j] = v[j] == -INFINITY ? 0.f : t[j] * expf(v[j] - m);
    __syncthreads();
    for (int c = 0; c < nch; c += 4) {
      const float4_t t4 = *reinterpret_cast<const float4_t*>(shared + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) s += t4[e];        // (zeros past the last chunk)
    }
  }
  *M = m;
  *S = s;
}

// The fp16 log-probability the reference would hold for logit x.
//   MODE 0 (mlx_eagle.py:410-412): topk over the logits, then fp16(x) - fp16(logsumexp)
//   MODE 1 (mlx_eagle.py:103):     log(softmax(x)) with both tensors materialised in fp16
template <int MODE>
__device__ inline float score_of(float x, float M, float S, float lse16) {
  if (MODE == 0) return (float)(half_t)(x - lse16);
  const float p16 = (float)(half_t)(expf(x - M) / S);
  return (float)(half_t)logf(p16);
}

// Pass 2: per chunk the k best entries by the ordering key (MODE 0: the logit; MODE 1: the
// fp16 log-probability, in which distinct logits can tie).  Grid (chunks, rows).  Bound by the chain of its
// phases; each wave picks the k best of its entries with integer maxima over registers and lanes, one wave the k best
// of those (with shuffles through LDS and a barrier per pick the three passes took 40 us for 8 rows of 152064; now 16.5).
template <int MODE>
__global__ __launch_bounds__(THREADS) void topk_partial_kernel(
    const half_t* __restrict__ logits, const int32_t* __restrict__ row_index, long V, int k,
    const float* __restrict__ pm, const float* __restrict__ ps, float* __restrict__ pv,
    int32_t* __restrict__ pi) {
  static_assert(CHUNK <= 0x10000, "the place of a candidate takes sixteen bits");
  __shared__ __attribute__((aligned(16))) float stats[STATS];
  __shared__ uint32_t best[THREADS / 64 * TOPK_MAX];
  const int row = blockIdx.y, ch = blockIdx.x, nch = gridDim.x;
  const half_t* r = row_ptr(logits, row_index, row, V);
  const long beg = (long)ch * CHUNK;
  float x[CHUNK / THREADS];
#pragma unroll
  for (int j = 0; j < CHUNK / THREADS; ++j) {
    const long i = beg + threadIdx.x + (long)j * THREADS;
    x[j] = (float)r[i < V ? i : V - 1];
  }
  float M = 0.f, S = 1.f;
  if (MODE == 1) row_stats(pm, ps, row, nch, stats, &M, &S);
  uint32_t key[CHUNK / THREADS];
#pragma unroll
  for (int j = 0; j < CHUNK / THREADS; ++j) {
    const int place = threadIdx.x + j * THREADS;
    key[j] = beg + place < V ? key_of(MODE == 0 ? x[j] : score_of<1>(x[j], M, S, 0.f), place) : 0u;
  }
  const uint32_t mine = wave_topk(key, k);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane < TOPK_MAX) best[wave * TOPK_MAX + lane] = mine;
  __syncthreads();
  if (wave) return;
  uint32_t last[1] = {lane < THREADS / 64 * TOPK_MAX ? best[lane] : 0u};
  const uint32_t pick = wave_topk(last, k);
  if (lane < k) {
    const long at = ((long)row * nch + ch) * TOPK_MAX + lane;
    pv[at] = pick ? key_value(pick) : -INFINITY;
    pi[at] = pick ? (int)beg + key_place(pick) : 0x7fffffff;     // 0x7fffffff: chunk exhausted
  }
}

// Pass 3: one wave per row merges the chunk candidates and writes indices and fp16 scores.  The candidates stand in the
// order of their indexes wherever scores are equal (chunks in order, picks of a chunk in order), so a candidate's
// place breaks ties as its index would.
constexpr int MERGE = 8;               // candidates per lane at a time
template <int MODE>
__global__ __launch_bounds__(64) void topk_merge_kernel(
    const half_t* __restrict__ logits, const int32_t* __restrict__ row_index, long V, int k,
    int nch, const float* __restrict__ pm, const float* __restrict__ ps,
    const float* __restrict__ pv, const int32_t* __restrict__ pi, int32_t* __restrict__ out_index,
    half_t* __restrict__ out_score) {
  __shared__ __attribute__((aligned(16))) float stats[STATS];
  const int row = blockIdx.x, lane = threadIdx.x;
  const int ncand = nch * TOPK_MAX;
  uint32_t mine = 0;
  for (int from = 0; from < ncand; from += 64 * MERGE) {
    uint32_t key[MERGE + 1];
    float v[MERGE];
    int32_t ix[MERGE];
#pragma unroll
    for (int j = 0; j < MERGE; ++j) {
      const int c = from + j * 64 + lane;
      const long at = (long)row * ncand + (c < ncand ? c : ncand - 1);
      v[j] = pv[at];
      ix[j] = pi[at];
    }
#pragma unroll
    for (int j = 0; j < MERGE; ++j) {
      const int c = from + j * 64 + lane;
      key[j] = c < ncand && c % TOPK_MAX < k && ix[j] != 0x7fffffff ? key_of(v[j], c) : 0u;
    }
    key[MERGE] = mine;
    mine = wave_topk(key, k);
  }
  float M = 0.f, S = 1.f, lse16 = 0.f;
  if (MODE == 0) {
    row_stats(pm, ps, row, nch, stats, &M, &S);
    lse16 = (float)(half_t)(M + logf(S));
  }
  const half_t* r = row_ptr(logits, row_index, row, V);
  if (lane < k) {
    const int idx = mine ? pi[(long)row * ncand + key_place(mine)] : 0;
    out_index[row * k + lane] = idx;
    out_score[row * k + lane] = MODE == 0 ? (half_t)score_of<0>((float)r[idx], M, S, lse16) : (half_t)(mine ? key_value(mine) : -INFINITY);
  }
}

// mlx_eagle.py:130-141: state before the first expansion level.
//   saved_scores / saved_tokens [k + k*k*depth], parents [1 + k*depth], mask_words [k][2],
//   cur_scores [k] fp16, cur_ids [k].
__global__ void draft_tree_init_kernel(const int32_t* __restrict__ topk_index,
                                       const half_t* __restrict__ topk_score, int k,
                                       half_t* __restrict__ saved_scores,
                                       int32_t* __restrict__ saved_tokens,
                                       uint32_t* __restrict__ parents, half_t* __restrict__ cur_scores,
                                       int32_t* __restrict__ cur_ids, uint32_t* __restrict__ mask_words) {
  const int r = threadIdx.x;
  if (r == 0) parents[0] = 0u;
  if (r < k) {
    saved_scores[r] = topk_score[r];
    saved_tokens[r] = topk_index[r];
    parents[1 + r] = (uint32_t)r + 1u;      // level 0: arange(k) + 1 (mlx_eagle.py:155-162)
    cur_scores[r] = topk_score[r];
    cur_ids[r] = topk_index[r];
    mask_words[2 * r] = 1u << r;            // the identity block of level 0 (mlx_eagle.py:171)
    mask_words[2 * r + 1] = 0u;
  }
}

// process_generate_tree_iteration (mlx_eagle.py:97-115) after the per-row top-k, plus what
// generate_draft_tree does with its results (mlx_eagle.py:157-162, 171, 194-207).  One wave;
// lane c is candidate c = k * row + column of the level's k x k table.
__global__ __launch_bounds__(64) void draft_tree_level_kernel(
    const int32_t* __restrict__ topk_index, const half_t* __restrict__ topk_score, int level, int k,
    int depth, half_t* __restrict__ saved_scores, int32_t* __restrict__ saved_tokens,
    uint32_t* __restrict__ parents, half_t* __restrict__ cur_scores, int32_t* __restrict__ cur_ids,
    uint32_t* __restrict__ mask_words, int32_t* __restrict__ out_ids,
    int32_t* __restrict__ topk_cs_index) {
  __shared__ float cu[64];
  __shared__ uint32_t old_mask[2 * TOPK_MAX];
  const int c = threadIdx.x;
  const int kk = k * k;
  float mine = -INFINITY;
  int tok = 0;
  if (c < kk) {
    // cumulative score in fp16 (mlx_eagle.py:106)
    mine = (float)(half_t)((float)topk_score[c] + (float)cur_scores[c / k]);
    tok = topk_index[c];
    saved_scores[k + kk * level + c] = (half_t)mine;
    saved_tokens[k + kk * level + c] = tok;
  }
  cu[c] = mine;
  if (c < 2 * k) old_mask[c] = mask_words[c];
  __syncthreads();
  int rank = 0;
  for (int j = 0; j < kk; ++j) rank += (cu[j] > mine) || (cu[j] == mine && j < c);
  if (c < kk && rank < k) {
    const int parent_row = c / k;
    topk_cs_index[rank] = c;
    out_ids[rank] = parent_row;
    cur_scores[rank] = (half_t)mine;
    cur_ids[rank] = tok;
    if (level + 1 < depth) {
      // rows of the next level's block of the parents table: selected flat id + 1
      const uint32_t bias = 1u + (uint32_t)kk * (uint32_t)level + (uint32_t)k;
      parents[1 + k * (level + 1) + rank] = (uint32_t)c + bias;
    }
    // children inherit the parent's row (mlx_eagle.py:207) and see themselves in the next
    // identity block (mlx_eagle.py:171)
    const int col = k * (level + 1) + rank;
    uint32_t lo = old_mask[2 * parent_row], hi = old_mask[2 * parent_row + 1];
    if (col < 32) lo |= 1u << col; else if (col < 64) hi |= 1u << (col - 32);
    mask_words[2 * rank] = lo;
    mask_words[2 * rank + 1] = hi;
  }
}

// Loop state of the speculative step kept on the device (mlx_eagle.py:393-394, 591-599).
__global__ void spec_begin_kernel(const int32_t* __restrict__ draft_len,
                                  const int32_t* __restrict__ accept, int32_t* __restrict__ expand_len,
                                  int32_t* __restrict__ write_len) {
  if (threadIdx.x == 0) {
    const int32_t v = *draft_len + 1 + accept[1];     // draft_offset (mlx_eagle.py:394)
    *expand_len = v;
    *write_len = v;
  }
}

__global__ void spec_update_kernel(const int32_t* __restrict__ accept,
                                   const int32_t* __restrict__ accepted_tokens, int32_t* __restrict__ y,
                                   int y_len, int32_t* __restrict__ draft_len,
                                   const int32_t* __restrict__ expand_len, int32_t* __restrict__ root_token,
                                   int32_t* __restrict__ out_tokens, int32_t* __restrict__ out_count,
                                   int max_out) {
  const int j = threadIdx.x;
  const int a = accept[1];
  const int32_t next = accept[3];
  const int base = *out_count;
  int32_t v = 0;
  if (j < a) v = accepted_tokens[j]; else if (j == a) v = next;
  if (j < y_len) y[j] = v;                            // accepted tokens, bonus token, zero padding
  if (j <= a && base + j < max_out) out_tokens[base + j] = v;
  __syncthreads();
  if (j == 0) {
    *draft_len = *expand_len;                         // the expansion rows are dropped (:593-594)
    *root_token = next;
    *out_count = base + a + 1;
  }
}

inline int chunks_for(long V) { return (int)((V + CHUNK - 1) / CHUNK); }

}  // namespace

EAGLE_EXPORT size_t eagle_logsoftmax_topk_workspace_bytes(int R, long V) {
  if (R < 1 || V < 1) return 0;
  const size_t nch = (size_t)chunks_for(V);
  return (size_t)R * nch * (2 + 2 * TOPK_MAX) * sizeof(float);
}

EAGLE_EXPORT int eagle_logsoftmax_topk_f16(const void* logits, const int32_t* row_index, int R, long V,
                                           int k, int mode, int32_t* out_index, void* out_score,
                                           void* workspace, size_t workspace_bytes,
                                           eagle_stream_t stream) {
  if (!logits || !out_index || !out_score) return EAGLE_ERR_NULL;
  if (R < 1 || R > EAGLE_MAX_TREE || V < 1 || k < 1 || k > TOPK_MAX || k > V) return EAGLE_ERR_SHAPE;
  if (chunks_for(V) * TOPK_MAX > 0x10000) return EAGLE_ERR_SHAPE;
  if (mode != 0 && mode != 1) return EAGLE_ERR_UNSUPPORTED;
  if (!workspace || !eagle_aligned16(workspace) ||
      workspace_bytes < eagle_logsoftmax_topk_workspace_bytes(R, V))
    return EAGLE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int nch = chunks_for(V);
  float* pm = static_cast<float*>(workspace);
  float* ps = pm + (size_t)R * nch;
  float* pv = ps + (size_t)R * nch;
  int32_t* pi = reinterpret_cast<int32_t*>(pv + (size_t)R * nch * TOPK_MAX);
  const half_t* lg = static_cast<const half_t*>(logits);
  half_t* os = static_cast<half_t*>(out_score);
  hipLaunchKernelGGL(lse_partial_kernel, dim3(nch, R), dim3(THREADS), 0, st, lg, row_index, V, pm, ps);
  if (mode == 0) {
    hipLaunchKernelGGL(topk_partial_kernel<0>, dim3(nch, R), dim3(THREADS), 0, st, lg, row_index, V, k,
                       pm, ps, pv, pi);
    hipLaunchKernelGGL(topk_merge_kernel<0>, dim3(R), dim3(64), 0, st, lg, row_index, V, k, nch, pm,
                       ps, pv, pi, out_index, os);
  } else {
    hipLaunchKernelGGL(topk_partial_kernel<1>, dim3(nch, R), dim3(THREADS), 0, st, lg, row_index, V, k,
                       pm, ps, pv, pi);
    hipLaunchKernelGGL(topk_merge_kernel<1>, dim3(R), dim3(64), 0, st, lg, row_index, V, k, nch, pm,
                       ps, pv, pi, out_index, os);
  }
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_draft_tree_init(const int32_t* topk_index, const void* topk_score, int k,
                                       void* saved_scores, int32_t* saved_tokens, uint32_t* parents,
                                       void* cur_scores, int32_t* cur_ids, uint32_t* mask_words,
                                       eagle_stream_t stream) {
  if (!topk_index || !topk_score || !saved_scores || !saved_tokens || !parents || !cur_scores ||
      !cur_ids || !mask_words)
    return EAGLE_ERR_NULL;
  if (k < 1 || k > TOPK_MAX) return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(draft_tree_init_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                     topk_index, static_cast<const half_t*>(topk_score), k,
                     static_cast<half_t*>(saved_scores), saved_tokens, parents,
                     static_cast<half_t*>(cur_scores), cur_ids, mask_words);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_draft_tree_level(const int32_t* topk_index, const void* topk_score, int level,
                                        int k, int depth, void* saved_scores, int32_t* saved_tokens,
                                        uint32_t* parents, void* cur_scores, int32_t* cur_ids,
                                        uint32_t* mask_words, int32_t* out_ids,
                                        int32_t* topk_cs_index, eagle_stream_t stream) {
  if (!topk_index || !topk_score || !saved_scores || !saved_tokens || !parents || !cur_scores ||
      !cur_ids || !mask_words || !out_ids || !topk_cs_index)
    return EAGLE_ERR_NULL;
  if (k < 1 || k > TOPK_MAX || depth < 1 || level < 0 || level >= depth || k * depth > 64)
    return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(draft_tree_level_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                     topk_index, static_cast<const half_t*>(topk_score), level, k, depth,
                     static_cast<half_t*>(saved_scores), saved_tokens, parents,
                     static_cast<half_t*>(cur_scores), cur_ids, mask_words, out_ids, topk_cs_index);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_spec_begin(const int32_t* draft_len_dev, const int32_t* accept,
                                  int32_t* expand_len_dev, int32_t* write_len_dev,
                                  eagle_stream_t stream) {
  if (!draft_len_dev || !accept || !expand_len_dev || !write_len_dev) return EAGLE_ERR_NULL;
  hipLaunchKernelGGL(spec_begin_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                     draft_len_dev, accept, expand_len_dev, write_len_dev);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_spec_update(const int32_t* accept, const int32_t* accepted_tokens, int32_t* y,
                                   int y_len, int32_t* draft_len_dev, const int32_t* expand_len_dev,
                                   int32_t* root_token_dev, int32_t* out_tokens, int32_t* out_count_dev,
                                   int max_out, eagle_stream_t stream) {
  if (!accept || !accepted_tokens || !y || !draft_len_dev || !expand_len_dev || !root_token_dev ||
      !out_tokens || !out_count_dev)
    return EAGLE_ERR_NULL;
  if (y_len < 1 || y_len > 64 || max_out < 1) return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(spec_update_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), accept,
                     accepted_tokens, y, y_len, draft_len_dev, expand_len_dev, root_token_dev, out_tokens,
                     out_count_dev, max_out);
  return eagle_launch_status();
}
