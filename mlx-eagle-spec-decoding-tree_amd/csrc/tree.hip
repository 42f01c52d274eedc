// Integer side of the tree step (gfx950): draft-tree layout, root-to-leaf paths, greedy
// longest-accepted-path selection, KV compaction.  Every kernel here is tiny exact
// integer work; they exist so that a verify step needs no device-to-host round trip.
#include "common.h"

#include <math.h>

namespace {

constexpr int MAXT = EAGLE_MAX_TREE_SLOTS;   // 64: tree tokens the kernels of this file lay out
constexpr int MAXC = 1024;             // draft candidates (k + k*k*depth)

// The candidates as they come from the expansion: a list of per-level pieces for each of scores,
// tokens and parents (or one piece each), read where they are instead of concatenated first.
struct TreeLists {
  const half_t* scores[EAGLE_MAX_SEGMENTS];
  const int32_t* tokens[EAGLE_MAX_SEGMENTS];
  const uint32_t* parents[EAGLE_MAX_SEGMENTS];
  int end[EAGLE_MAX_SEGMENTS];        // candidates up to and including piece i
  int pend[EAGLE_MAX_SEGMENTS];       // parents up to and including piece i
  const void* root;                   // the root token, int32 or int64
  int n, pn, root64;
};

// Element i of a list.  The pieces are compared in turn with constant indexes: their ends and addresses are scalar
// loads at the kernel's start, where a search per lane would wait for memory at every piece.
template <typename T>
__device__ inline T list_at(const T* const (&ptr)[EAGLE_MAX_SEGMENTS], const int (&end)[EAGLE_MAX_SEGMENTS], int n, int i) {
  const T* p = ptr[0];
  int base = 0;
#pragma unroll
  for (int s = 1; s < EAGLE_MAX_SEGMENTS; ++s)
    if (s < n && i >= end[s - 1]) {
      p = ptr[s];
      base = end[s - 1];
    }
  return p[i - base];
}

constexpr int TREE_THREADS = 1024;
constexpr int RANK_PARTS = 8;                              // threads that share the ranking of a candidate
constexpr int RANK_BASE = TREE_THREADS / RANK_PARTS;       // candidates c, c + RANK_BASE, ... to a thread

// Adds to the ranks of candidates c0 + r RANK_BASE (r < N) how many of keys[from .. to) are ahead of each
template <int N>
__device__ inline void count_ahead(const uint32_t* keys, int* ranks, int c0, int C, int from, int to) {
  uint32_t key[N];
  int ahead[N];
#pragma unroll
  for (int r = 0; r < N; ++r) {
    const int i = c0 + r * RANK_BASE;
    key[r] = keys[i < C ? i : 0];
    ahead[r] = 0;
  }
#pragma unroll 2
  for (int j = from; j < to; j += 4) {
    const uint4_t k4 = *reinterpret_cast<const uint4_t*>(keys + j);
#pragma unroll
    for (int r = 0; r < N; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) ahead[r] += k4[e] > key[r];
  }
#pragma unroll
  for (int r = 0; r < N; ++r)
    if (c0 + r * RANK_BASE < C) atomicAdd(ranks + c0 + r * RANK_BASE, ahead[r]);
}

// mlx_eagle.py:217-250 (with topk :24-58 and search_sorted :61-93).  One workgroup; bound by the chain of its
// phases (two dependent loads, the ranks, the walk), so none of them is a loop of one thread: a candidate is ranked by eight
// threads, on one integer comparison per pair, and a thread ranks several, so that a read of four keys from LDS serves
// several comparisons; the picked ones are counted with ballots; every token walks up to the root by itself.  39 of 328 candidates,
// us in a graph: 7.0 (7.7 with a candidate to two threads and a read for every four comparisons), of 200 5.4 (6.4), 7 of 72 4.4 (4.9);
// the comparisons themselves are what is left above that.
__global__ __launch_bounds__(TREE_THREADS) void process_draft_tree_kernel(
    TreeLists in, int C, int k, int total, int32_t* __restrict__ pos_ids, int32_t* __restrict__ mask_index,
    int32_t* __restrict__ draft_tokens, uint32_t* __restrict__ bits_out, uint16_t* __restrict__ mask_out) {
  __shared__ __attribute__((aligned(16))) uint32_t keys[MAXC];
  __shared__ int ranks[MAXC];
  __shared__ int wave_picked[MAXC / 64];
  __shared__ int sel[MAXT];
  __shared__ int midx[MAXT];
  __shared__ unsigned long long bits[MAXT];
  const int tid = threadIdx.x;
  // Key of a candidate: its fp16 score as an ordered integer, then its index from the back, so that a larger key is
  // ahead in the stable descending order.  A NaN score ranks as -inf and -0 as 0: the order is total and exactly
  // `total` candidates are picked whatever the scores hold.
  static_assert(TREE_THREADS == MAXC, "a thread per candidate");
  constexpr int ROUND = 4 * RANK_PARTS;
  const int CR = (C + ROUND - 1) / ROUND * ROUND;        // every part whole reads of four keys (keys of 0 are never ahead)
  ranks[tid] = 0;
  if (tid < CR) {
    uint32_t key = 0;
    if (tid < C) {
      uint32_t h = __builtin_bit_cast(unsigned short, list_at(in.scores, in.end, in.n, tid));
      if ((h & 0x7fffu) > 0x7c00u) h = 0xfc00u;
      if (h == 0x8000u) h = 0u;
      key = (h & 0x8000u ? ~h & 0xffffu : h | 0x8000u) << 16 | (0xffffu - (uint32_t)tid);
    }
    keys[tid] = key;
  }
  __syncthreads();
  {
    const int c0 = tid % RANK_BASE, from = tid / RANK_BASE * (CR / RANK_PARTS), to = from + CR / RANK_PARTS;
    if (C <= RANK_BASE) count_ahead<1>(keys, ranks, c0, C, from, to);
    else if (C <= 2 * RANK_BASE) count_ahead<2>(keys, ranks, c0, C, from, to);
    else if (C <= 3 * RANK_BASE) count_ahead<3>(keys, ranks, c0, C, from, to);
    else if (C <= 4 * RANK_BASE) count_ahead<4>(keys, ranks, c0, C, from, to);
    else count_ahead<MAXC / RANK_BASE>(keys, ranks, c0, C, from, to);
  }
  __syncthreads();
  // the picked candidates in ascending flat index
  const bool picked = tid < C && ranks[tid] < total;
  const unsigned long long m = __ballot(picked);
  if ((tid & 63) == 0) wave_picked[tid >> 6] = __popcll(m);
  __syncthreads();
  if (picked) {
    int before = __popcll(m & ((1ull << (tid & 63)) - 1ull));
    for (int w = 0; w < (tid >> 6); ++w) before += wave_picked[w];
    if (before < total) sel[before] = tid;
  }
  __syncthreads();
  if (tid < total) {
    const int c = sel[tid];
    draft_tokens[tid + 1] = list_at(in.tokens, in.end, in.n, c);
    const uint32_t dp = list_at(in.parents, in.pend, in.pn, c / k);
    // fixed-step left binary search for the flat id dp - 1 (uint32 arithmetic, wraps for dp == 0)
    const uint32_t target = dp - 1u;
    uint32_t low = 0, high = (uint32_t)total;
    int steps = 0;
    while ((1 << steps) < total) ++steps;   // ceil(log2(total))
    for (int s = 0; s < steps; ++s) {
      const uint32_t mid = (low + high) >> 1;
      if (mid < (uint32_t)total) {
        const uint32_t val = (uint32_t)sel[mid];
        if (val < target) low = mid + 1; else high = mid;
      }
    }
    const int mi = (dp == 0u) ? 0 : (int)low + 1;
    midx[tid] = mi;
    mask_index[tid] = mi;
  }
  if (tid == 0)
    draft_tokens[0] = in.root64 ? (int32_t)*static_cast<const int64_t*>(in.root) : *static_cast<const int32_t*>(in.root);
  __syncthreads();
  if (tid <= total) {
    // identity rows ORed in ascending order (mlx_eagle.py:239-243): a row inherits its parent's
    // finished row where the parent comes earlier, and the bare identity row of a parent slot at or
    // after its child (which only poisoned scores can produce), where the walk therefore ends
    unsigned long long row = 1ull << tid;
    int cur = tid;
    while (cur > 0) {
      const int m = midx[cur - 1];
      const int par = m < 0 ? 0 : (m > total ? total : m);
      row |= 1ull << par;
      if (par >= cur) break;
      cur = par;
    }
    bits[tid] = row;
    // one mask word per row for trees of at most 32 tokens, two (low, high) above that
    if (bits_out) {
      if (total + 1 <= 32) {
        bits_out[tid] = (uint32_t)row;
      } else {
        bits_out[2 * tid] = (uint32_t)row;
        bits_out[2 * tid + 1] = (uint32_t)(row >> 32);
      }
    }
    pos_ids[tid] = __popcll(row) - 1;
  }
  if (!mask_out) return;
  // the additive mask of the module path, bf16: 0 where visible, -inf elsewhere
  __syncthreads();
  const int T = total + 1;
  for (int i = tid; i < T * T; i += TREE_THREADS)
    mask_out[i] = (bits[i / T] >> (i % T)) & 1ull ? 0u : 0xff80u;
}

// mlx_eagle.py:254-295 in one wave (a lane per token, T <= 64).  retrieve [64][64], shape {leaf_num,
// max_depth + 1}; PACKED: rows of max_depth + 1 entries, leaf_num of them, without padding, and the shape last, as one 8-byte
// store to memory that the host may be watching: who sees it may use the rows, on any stream, as after a wait for this one.  (A shape
// that is not aligned for that store is written as two words, for a caller that waits for the stream.)
template <bool PACKED>
__global__ __launch_bounds__(64) void post_process_kernel(const int32_t* __restrict__ pos_ids,
                                                         const int32_t* __restrict__ mask_index,
                                                         int total, int32_t* __restrict__ retrieve,
                                                         int32_t* __restrict__ shape) {
  __shared__ int inner[MAXT + 1];
  __shared__ int par[MAXT];
  const int tid = threadIdx.x;
  const int T = total + 1;
  inner[tid] = 0;
  if (tid == 0) inner[MAXT] = 0;
  const int depth = tid < T ? pos_ids[tid] : 0;
  if (tid < total) par[tid] = mask_index[tid];
  __syncthreads();
  if (tid < total) {
    const int p = par[tid];
    if (p >= 0 && p <= MAXT) inner[p] = 1;   // benign race: all writers store 1
  }
  __syncthreads();
  const unsigned long long inner_mask = __ballot(inner[tid] != 0);
  const int n_inner = __popcll(inner_mask) + inner[MAXT];
  int md = depth;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const int other = __shfl_xor(md, o, 64);
    md = other > md ? other : md;
  }
  const int leaves = total - (n_inner - 1), cols = md + 1;
  if (!PACKED && tid == 0) {
    shape[0] = leaves;
    shape[1] = cols;
  }
  const int ld = PACKED ? (cols < 1 ? 1 : (cols > MAXT ? MAXT : cols)) : MAXT;
  const int rows = PACKED ? (leaves < 1 ? 1 : (leaves > MAXT ? MAXT : leaves)) : MAXT;
  for (int i = tid; i < rows * ld; i += 64) retrieve[i] = -1;
  __syncthreads();
  if (tid < T && !inner[tid]) {
    const int r = __popcll(~inner_mask & ((1ull << tid) - 1ull));
    int cur = tid;
    for (int col = depth; col >= 0; --col) {
      if (col < ld && r < rows) retrieve[r * ld + col] = cur;
      cur = (cur == 0) ? par[total - 1] : par[cur - 1];
      cur = cur < 0 ? 0 : (cur > total ? total : cur);
    }
  }
  if (PACKED) {
    __syncthreads();
    if (tid != 0) return;
    if (reinterpret_cast<uintptr_t>(shape) & 7u) {
      shape[0] = leaves;
      shape[1] = cols;
    } else {
      __hip_atomic_store(reinterpret_cast<unsigned long long*>(shape),
                         (unsigned long long)(uint32_t)cols << 32 | (uint32_t)leaves, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// mlx_eagle.py:311-326 on per-node argmax tokens, with the gathers of :582-589.
__global__ __launch_bounds__(128) void greedy_accept_kernel(
    const int32_t* __restrict__ node_argmax, const int32_t* __restrict__ draft_tokens,
    const int32_t* __restrict__ retrieve, const int32_t* __restrict__ shape, int T,
    int32_t* __restrict__ result, int32_t* __restrict__ accepted_tokens) {
  __shared__ int len[MAXT];
  const int tid = threadIdx.x;
  int leaves = shape[0], cols = shape[1];
  leaves = leaves < 1 ? 1 : (leaves > MAXT ? MAXT : leaves);
  cols = cols < 1 ? 1 : (cols > MAXT ? MAXT : cols);
  if (tid < MAXT) len[tid] = -1;
  __syncthreads();
  if (tid < leaves) {
    int n = 0;
    for (int j = 0; j + 1 < cols; ++j) {
      int a = retrieve[tid * MAXT + j];
      int b = retrieve[tid * MAXT + j + 1];
      a = a < 0 ? a + T : a;   // a negative gather index counts from the end
      b = b < 0 ? b + T : b;
      if (draft_tokens[b] == node_argmax[a]) ++n; else break;
    }
    len[tid] = n;
  }
  __syncthreads();
  if (tid == 0) {
    int best = 0, al = len[0];
    for (int r = 1; r < leaves; ++r)
      if (len[r] > al) { al = len[r]; best = r; }
    if (al == 0) best = 0;
    int bonus = retrieve[best * MAXT + al];
    bonus = bonus < 0 ? bonus + T : bonus;
    result[0] = best;
    result[1] = al;
    result[2] = bonus;
    result[3] = node_argmax[bonus];
    for (int j = 0; j < MAXT; ++j) {
      int idx = 0, tok = 0;
      if (j < al) {
        idx = retrieve[best * MAXT + 1 + j];
        const int w = idx < 0 ? idx + T : idx;
        tok = draft_tokens[w];
      }
      result[4 + j] = idx;
      accepted_tokens[j] = tok;
    }
  }
}

// mlx_eagle.py:366-374: rows P + idx[j] -> P + 1 + j, gather first, then scatter.
// grid (G, n_caches); the accepted rows of one head are staged in LDS.
__global__ __launch_bounds__(256) void kv_compact_kernel(half_t* const* __restrict__ caches,
                                                         const int32_t* __restrict__ accept,
                                                         const int32_t* __restrict__ len_dev,
                                                         int hd, long cap) {
  extern __shared__ __attribute__((aligned(16))) unsigned char stage[];
  const int al = accept[1];
  if (al <= 0) return;
  const int n = al > MAXT ? MAXT : al;
  const long P = *len_dev;
  half_t* base = caches[blockIdx.y] + (long)blockIdx.x * cap * hd;
  const int vec_row = hd / 8;
  for (int v = threadIdx.x; v < n * vec_row; v += blockDim.x) {
    const int j = v / vec_row;
    const int c = v % vec_row;
    long src = P + accept[4 + j];
    src = src < 0 ? 0 : (src >= cap ? cap - 1 : src);
    reinterpret_cast<half8_t*>(stage)[v] = *reinterpret_cast<const half8_t*>(base + src * hd + c * 8);
  }
  __syncthreads();
  for (int v = threadIdx.x; v < n * vec_row; v += blockDim.x) {
    const int j = v / vec_row;
    const int c = v % vec_row;
    const long dst = P + 1 + j;
    if (dst < cap)
      *reinterpret_cast<half8_t*>(base + dst * hd + c * 8) = reinterpret_cast<const half8_t*>(stage)[v];
  }
}

// the length saturates at the capacity: a caller that replays steps beyond it gets a full
// cache (the append kernels skip rows at or beyond the capacity), never a length that points
// outside the buffers
__global__ void set_len_after_accept(const int32_t* __restrict__ accept, int32_t* len_dev, long cap) {
  if (threadIdx.x == 0 && blockIdx.x == 0) {
    const int al = accept[1] < 0 ? 0 : accept[1];
    const long n = (long)*len_dev + al + 1;
    *len_dev = (int32_t)(n < cap ? n : cap);
  }
}

__global__ void fill_i32_kernel(int32_t* dst, int32_t value, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) dst[i] = value;
}

__global__ void tree_positions_kernel(const int32_t* __restrict__ pos_ids,
                                      const int32_t* __restrict__ len_dev,
                                      int32_t* __restrict__ positions, int T) {
  const int i = threadIdx.x;
  if (i < T) positions[i] = *len_dev + pos_ids[i];
}

// rows *len .. *len + R - 1 of a prompt chunk and the first row of each of its pieces of 32
__global__ void chunk_positions_kernel(const int32_t* __restrict__ len_dev, int32_t* __restrict__ positions,
                                       int32_t* __restrict__ piece_len, int R) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= R) return;
  const int at = *len_dev + i;
  positions[i] = at;
  if ((i & 31) == 0) piece_len[i >> 5] = at;
}

__global__ void advance_len_kernel(int32_t* len_dev, int delta) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *len_dev += delta;
}

}  // namespace

static int process_tree(const TreeLists& in, int C, int k, int total, int32_t* tree_position_ids, int32_t* mask_index,
                        int32_t* draft_tokens, uint32_t* bits, void* mask, eagle_stream_t stream) {
  if (k < 1 || C < 1 || C > MAXC || (C % k) != 0 || total < 1 || total >= MAXT || total > C)
    return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(process_draft_tree_kernel, dim3(1), dim3(TREE_THREADS), 0, static_cast<hipStream_t>(stream),
                     in, C, k, total, tree_position_ids, mask_index, draft_tokens, bits,
                     static_cast<uint16_t*>(mask));
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_process_draft_tree(const void* scores, const int32_t* tokens,
                                          const uint32_t* parents_list,
                                          const int32_t* sampled_token_dev, int C, int k,
                                          int total, int32_t* tree_position_ids,
                                          int32_t* mask_index, int32_t* draft_tokens,
                                          uint32_t* tree_mask_bits, eagle_stream_t stream) {
  if (!scores || !tokens || !parents_list || !sampled_token_dev || !tree_position_ids ||
      !mask_index || !draft_tokens || !tree_mask_bits)
    return EAGLE_ERR_NULL;
  TreeLists in = {};
  in.scores[0] = static_cast<const half_t*>(scores);
  in.tokens[0] = tokens;
  in.parents[0] = parents_list;
  in.end[0] = in.pend[0] = MAXC;
  in.n = in.pn = 1;
  in.root = sampled_token_dev;
  return process_tree(in, C, k, total, tree_position_ids, mask_index, draft_tokens, tree_mask_bits, nullptr, stream);
}

EAGLE_EXPORT int eagle_process_draft_tree_lists(const void* const* scores, const int32_t* const* tokens,
                                                const int* counts, int n, const uint32_t* const* parents,
                                                const int* parent_counts, int parents_n,
                                                const void* sampled_token_dev, int sampled_is_64bit, int k,
                                                int total, int32_t* tree_position_ids, int32_t* mask_index,
                                                int32_t* draft_tokens, void* tree_mask_bf16,
                                                eagle_stream_t stream) {
  if (!scores || !tokens || !counts || !parents || !parent_counts || !sampled_token_dev || !tree_position_ids ||
      !mask_index || !draft_tokens || !tree_mask_bf16)
    return EAGLE_ERR_NULL;
  if (n < 1 || n > EAGLE_MAX_SEGMENTS || parents_n < 1 || parents_n > EAGLE_MAX_SEGMENTS) return EAGLE_ERR_SHAPE;
  TreeLists in = {};
  int C = 0, P = 0;
  for (int i = 0; i < n; ++i) {
    if (!scores[i] || !tokens[i]) return EAGLE_ERR_NULL;
    if (counts[i] < 1 || counts[i] > MAXC) return EAGLE_ERR_SHAPE;
    in.scores[i] = static_cast<const half_t*>(scores[i]);
    in.tokens[i] = tokens[i];
    in.end[i] = C += counts[i];
  }
  for (int i = 0; i < parents_n; ++i) {
    if (!parents[i]) return EAGLE_ERR_NULL;
    if (parent_counts[i] < 1 || parent_counts[i] > MAXC) return EAGLE_ERR_SHAPE;
    in.parents[i] = parents[i];
    in.pend[i] = P += parent_counts[i];
  }
  if (k < 1 || P < C / k) return EAGLE_ERR_SHAPE;
  in.n = n;
  in.pn = parents_n;
  in.root = sampled_token_dev;
  in.root64 = sampled_is_64bit;
  return process_tree(in, C, k, total, tree_position_ids, mask_index, draft_tokens, nullptr, tree_mask_bf16, stream);
}

static int post_process(const int32_t* tree_position_ids, const int32_t* mask_index, int total,
                        int32_t* retrieve_indices, int32_t* shape_out, bool packed, eagle_stream_t stream) {
  if (!tree_position_ids || !mask_index || !retrieve_indices || !shape_out) return EAGLE_ERR_NULL;
  if (total < 1 || total >= MAXT) return EAGLE_ERR_SHAPE;
  if (packed)
    hipLaunchKernelGGL(post_process_kernel<true>, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                       tree_position_ids, mask_index, total, retrieve_indices, shape_out);
  else
    hipLaunchKernelGGL(post_process_kernel<false>, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                       tree_position_ids, mask_index, total, retrieve_indices, shape_out);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_post_process_draft_tree(const int32_t* tree_position_ids,
                                               const int32_t* mask_index, int total,
                                               int32_t* retrieve_indices, int32_t* shape_out,
                                               eagle_stream_t stream) {
  return post_process(tree_position_ids, mask_index, total, retrieve_indices, shape_out, false, stream);
}

EAGLE_EXPORT int eagle_post_process_draft_tree_packed(const int32_t* tree_position_ids,
                                                      const int32_t* mask_index, int total,
                                                      int32_t* retrieve_indices, int32_t* shape_out,
                                                      eagle_stream_t stream) {
  return post_process(tree_position_ids, mask_index, total, retrieve_indices, shape_out, true, stream);
}

EAGLE_EXPORT int eagle_greedy_accept(const int32_t* node_argmax, const int32_t* draft_tokens,
                                     const int32_t* retrieve_indices, const int32_t* shape, int T,
                                     int32_t* result, int32_t* accepted_tokens,
                                     eagle_stream_t stream) {
  if (!node_argmax || !draft_tokens || !retrieve_indices || !shape || !result || !accepted_tokens)
    return EAGLE_ERR_NULL;
  if (T < 1 || T > MAXT) return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(greedy_accept_kernel, dim3(1), dim3(128), 0, static_cast<hipStream_t>(stream),
                     node_argmax, draft_tokens, retrieve_indices, shape, T, result,
                     accepted_tokens);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_kv_compact_f16(void* const* caches_dev, int n_caches, const int32_t* accept,
                                      int32_t* cache_len_dev, int G, int hd, long capacity,
                                      eagle_stream_t stream) {
  if (!caches_dev || !accept || !cache_len_dev) return EAGLE_ERR_NULL;
  if (n_caches < 1 || n_caches > 65535 || G < 1 || hd < 8 || (hd % 8) != 0 || capacity < 2)
    return EAGLE_ERR_SHAPE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const size_t lds = (size_t)MAXT * hd * 2;
  hipLaunchKernelGGL(kv_compact_kernel, dim3(G, n_caches), dim3(256), lds, st,
                     reinterpret_cast<half_t* const*>(caches_dev), accept, cache_len_dev, hd,
                     capacity);
  hipLaunchKernelGGL(set_len_after_accept, dim3(1), dim3(64), 0, st, accept, cache_len_dev, capacity);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_fill_i32(int32_t* dst, int32_t value, long n, eagle_stream_t stream) {
  if (!dst) return EAGLE_ERR_NULL;
  if (n < 1) return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(fill_i32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), dst, value, n);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_tree_positions(const int32_t* tree_position_ids,
                                      const int32_t* cache_len_dev, int32_t* positions, int T,
                                      eagle_stream_t stream) {
  if (!tree_position_ids || !cache_len_dev || !positions) return EAGLE_ERR_NULL;
  if (T < 1 || T > MAXT) return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(tree_positions_kernel, dim3(1), dim3(64), 0,
                     static_cast<hipStream_t>(stream), tree_position_ids, cache_len_dev, positions,
                     T);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_chunk_positions(const int32_t* cache_len_dev, int32_t* positions, int32_t* piece_len, int R,
                                       eagle_stream_t stream) {
  if (!cache_len_dev || !positions || !piece_len) return EAGLE_ERR_NULL;
  if (R < 32 || (R % 32) != 0 || R > EAGLE_MAX_CHUNK) return EAGLE_ERR_SHAPE;
  hipLaunchKernelGGL(chunk_positions_kernel, dim3((R + 255) / 256), dim3(256), 0, static_cast<hipStream_t>(stream), cache_len_dev,
                     positions, piece_len, R);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_advance_len(int32_t* cache_len_dev, int delta, eagle_stream_t stream) {
  if (!cache_len_dev) return EAGLE_ERR_NULL;
  hipLaunchKernelGGL(advance_len_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream),
                     cache_len_dev, delta);
  return eagle_launch_status();
}

EAGLE_EXPORT const char* eagle_status_string(int status) {
  switch (status) {
    case EAGLE_OK: return "ok";
    case EAGLE_ERR_NULL: return "required pointer is NULL";
    case EAGLE_ERR_SHAPE: return "dimension outside the supported range";
    case EAGLE_ERR_ALIGN: return "pointer is not sufficiently aligned";
    case EAGLE_ERR_UNSUPPORTED: return "only group_size=64, bits=4 is supported";
    case EAGLE_ERR_WORKSPACE: return "workspace missing, misaligned or too small";
    case EAGLE_ERR_HIP: return "HIP runtime error at launch";
    case EAGLE_ERR_ARCH: return "device is not gfx950";
    default: return "unknown status";
  }
}

EAGLE_EXPORT int eagle_abi_version(void) { return 1; }

EAGLE_EXPORT int eagle_check_device(void) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return EAGLE_ERR_HIP;
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return EAGLE_ERR_HIP;
  const char* a = prop.gcnArchName;
  return (a[0] == 'g' && a[1] == 'f' && a[2] == 'x' && a[3] == '9' && a[4] == '5' && a[5] == '0')
             ? EAGLE_OK
             : EAGLE_ERR_ARCH;
}
