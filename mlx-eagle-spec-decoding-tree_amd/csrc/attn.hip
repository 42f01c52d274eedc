// Grouped-query attention of tree, draft and prompt rows against a KV cache (gfx950).
//
//   out[t, h*hd + d] = sum_j softmax_j( scale * q[h,t,:] . k[g,j,:] + mask[t,j] ) v[g,j,d]
//
// The first P = *cache_len_dev cache rows are the prefix, visible to every row; of the masked rows
// P .. P+Tk-1, row j is visible to token i iff bit j of its mask words is set (the ancestor-or-self mask of
// mlx_eagle.py:239-248,337-338; Tk = T in a tree pass; on the draft side (mlx_eagle.py:143-178,207) T queries see the
// Tk <= 64 rows of the earlier expansion levels and this one).  Call site replaced: mlx_llama.py:185-195.
//
// tree_attn_kernel: 1..64 query rows, one launch, or two where the keys are split over workgroups.
// causal_attn_kernel: a prompt chunk (mlx_llama.py:275-276) in pieces of 32 rows, each with its own cache length, the mask
// generated in the kernel, one launch for all pieces (two where the keys are split).
#include "common.h"

#include <math.h>

namespace {

constexpr float M_FLOOR = -3.0e38f;   // running maximum of a row that has seen no key yet

// ds_read_b64_tr_b16: 16 lanes x 4 halves, transposed (lane i of a group of 16 receives element
// i % 4 of the lanes 4 j + i / 4, j = 0..3 of the group); the address is 8-byte aligned
typedef __fp16 fp16x4_t __attribute__((__vector_size__(4 * sizeof(__fp16))));
__device__ inline half4_t lds_read_tr16(const unsigned char* p) {
  const fp16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4f16(
      (__attribute__((address_space(3))) fp16x4_t*)(p));
  return __builtin_bit_cast(half4_t, v);
}

// over the lane 32 away, and over the four lanes sixteen apart: without a trip through LDS
__device__ inline float max32(float v) { return wave_f32(wave_reduce32(wave_u32(v), WaveMax())); }
__device__ inline float sum32(float v) { return wave_f32(wave_reduce32(wave_u32(v), WaveAdd())); }
__device__ inline float max16_32(float v) { return max32(wave_f32(wave_reduce16(wave_u32(v), WaveMax()))); }
__device__ inline float sum16_32(float v) { return sum32(wave_f32(wave_reduce16(wave_u32(v), WaveAdd()))); }

// ---- 1..64 query rows (a tree, a draft pass): queries packed over heads and tokens ----
//
// A workgroup owns 16 NC columns of S^T = K Q^T, (query head, token) pairs of one KV group, and a range of the keys.  Its
// eight waves deal the 32-key blocks among themselves, each with an online softmax of its own, and share nothing until
// their (m, l, O) meet in LDS in fp32: no barrier in the loop.  A block comes in by whole rows and goes through the wave's slice of
// LDS (K for the operand layout, V for the transposing read); the first is requested before the length is known.
//
// What bounds it: the launch, the round trip of the length and of the first block (3.0 us on a short cache), then 0.10
// (head dimension 64) or 0.18 us per block and compute unit, about half of that the block's way through LDS and back, the rest its
// instructions (a scalar wave index, 32-bit lane offsets and lane swaps instead of shuffles took 5 % off).
// (K straight from memory into the operand layout, 16 bytes of 64 lines per load, 0.14 / 0.28; ten, twelve or sixteen waves, two blocks
// ahead or 32 columns per workgroup: slower; K and V one after the other in one buffer: no gain at 64, spills at 128.)
// Against one wave per query head with up to 33 key splits, partial results in fp16 and a merge of them, us per
// call in a graph (before / now): 14 heads of 64 in 2 groups, 8 rows behind 560 keys 10.1 / 4.9, behind 2048 11.5 / 9.0 (one split),
// 32 rows behind 4000 15.8 / 7.7; 28 heads of 128 in 4 groups, 32 rows behind 1024 14.6 / 9.1, 2048 17.0 / 10.8, 40 rows behind 1000 15.9 / 11.3.
// Those are of K and V of 28 layers in turn; from HBM (2 GiB of them in turn) 8 rows behind 2048 11.6 / 11.0, 32 behind 1024 14.7 / 9.3, 2048 17.3 / 11.3.
constexpr int NW = 8;                   // waves per workgroup

// Key splits of a launch: `most` in the grid; `least` always in use, behind a prefix of P rows no more than one per 512 keys and, up to `half`
// rows, than `few`, so that a short prefix in a large cache pays for few partial results.
struct TreeSplits {
  int least, few, most, half;
};
__device__ inline int tree_splits_in_use(int P, const TreeSplits& s) {
  int n = P >> 9;
  const int top = P > s.half ? s.most : s.few;
  n = n < top ? n : top;
  return n > s.least ? n : s.least;
}
// cached rows before the masked ones: never past the cache, whatever the counter says
__device__ inline int tree_prefix(const int32_t* len_dev, long cap, int Tk) {
  int P = len_dev[0];
  if (P > cap - Tk) P = (int)(cap - Tk);
  return P < 0 ? 0 : P;
}

template <int HD, int NC, bool WIDE>
__global__ __launch_bounds__(NW * 64) void tree_attn_kernel(
    const half_t* __restrict__ q, const half_t* __restrict__ kc, const half_t* __restrict__ vc,
    const uint32_t* __restrict__ mask_bits, const int32_t* __restrict__ len_dev, half_t* __restrict__ out, float* __restrict__ part,
    int T, int H, int G, long cap, float scale_log2e, int Tk, uint32_t inv_T, TreeSplits splits, uint32_t inv_G) {
  constexpr int KSTEPS = HD / 32;       // MFMA steps over the head dimension for S
  constexpr int DB = HD / 16;           // 16-wide blocks of the head dimension for O
  constexpr int STR = HD * 2 + 16;      // LDS row stride in bytes of a wave's V block
  constexpr int VR = HD / 8;            // 16-byte vectors per V row
  constexpr int NV = 32 * VR / 64;      // vectors of a V block per lane
  constexpr int SLICE = 64 * STR;       // a wave's K block, then its V block
  constexpr int OSTR = HD + 4;          // floats per column of a wave's O tile, over its blocks
  static_assert(NC * 16 * OSTR * 4 <= SLICE, "a wave's O tile does not fit over its blocks");
  __shared__ __attribute__((aligned(16))) unsigned char slices[NW][SLICE];
  __shared__ float2_t ml[NW][16 * NC];
  const int nsplit = splits.most;
  // this workgroup's KV group and key split; with inv_G the grid is 8 x columns x eighths of the (split, group) pairs, which puts
  // the columns that read the same keys on one XCD
  int g = blockIdx.x, split = blockIdx.z;
  if (inv_G) {
    const int pair = blockIdx.z * 8 + blockIdx.x;
    split = (int)((uint32_t)pair * inv_G >> 16);
    g = pair - split * G;
  }
  if (split >= nsplit) return;
  const int rep = H / G;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, kq = lane >> 4;
  const int cols = rep * T;
  const int first = split * NW + wave;          // this wave's first block
  const int col0 = blockIdx.y * 16 * NC;
  const char* kb_ptr = reinterpret_cast<const char*>(kc + (long)g * cap * HD);
  const char* vb_ptr = reinterpret_cast<const char*>(vc + (long)g * cap * HD);

  half8_t kreg[NV], vreg[NV];
  const int vrow = lane / VR, vcol = lane % VR;
  auto fetch = [&](int blk, int last) {              // rows past `last` read row `last`
    const int kb = blk * 32 < last ? blk * 32 : last, most = last - kb;
    const char* kp = kb_ptr + (long)kb * (HD * 2);   // uniform, with 32 bits of a lane's own
    const char* vp = vb_ptr + (long)kb * (HD * 2);
    uint32_t at[NV];
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      const int row = it * (64 / VR) + vrow;
      at[it] = (uint32_t)(row < most ? row : most) * (HD * 2) + vcol * 16;
    }
#pragma unroll
    for (int it = 0; it < NV; ++it) kreg[it] = *reinterpret_cast<const half8_t*>(kp + at[it]);
#pragma unroll
    for (int it = 0; it < NV; ++it) vreg[it] = *reinterpret_cast<const half8_t*>(vp + at[it]);
  };
  // A wave's first block is requested before the length is known: rows of the buffer, whatever they hold
  // (scores of rows past the end are masked, their V rows replaced by zeros).
  const int cap_last = (int)cap - 1;
  fetch(first, cap_last);
  half8_t qreg[NC][KSTEPS];
  uint32_t lo_bits[NC], hi_bits[NC];
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    int col = col0 + 16 * n + c;
    if (col > cols - 1) col = cols - 1;              // columns past the end repeat the last one and are not stored
    const int t = col - (int)((uint32_t)col * inv_T >> 16) * T;
    const half_t* qp = q + (long)g * cols * HD + col * HD + kq * 8;       // [group][head, token]
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk) qreg[n][kk] = *reinterpret_cast<const half8_t*>(qp + kk * 32);
    lo_bits[n] = mask_bits[WIDE ? 2 * t : t];
    hi_bits[n] = WIDE ? mask_bits[2 * t + 1] : 0u;
  }
  __builtin_amdgcn_sched_barrier(0);
  const int P = tree_prefix(len_dev, cap, Tk);
  const int Ltot = P + Tk;
  const int nblk = (Ltot + 31) >> 5;
  const int in_use = tree_splits_in_use(P, splits), stride = in_use * NW;
  if (split >= in_use) return;

  float m_run[NC], l_run[NC];
  float4_t o_acc[NC][DB];
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    m_run[n] = M_FLOOR;
    l_run[n] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) o_acc[n][db] = float4_t{0.f, 0.f, 0.f, 0.f};
  }
  unsigned char* ldsK = slices[wave];
  unsigned char* ldsV = ldsK + 32 * STR;
  // transposing loads: lane s of 16 asks for key row 4 kq + s / 4 at the four d columns 4 (s % 4) .. + 3
  const unsigned char* vt_base = ldsV + (4 * kq + (c >> 2)) * STR + (4 * (c & 3)) * 2;

  for (int blk = first; blk < nblk; blk += stride) {
    const int kb = blk * 32;
    if (kb + 32 > Ltot) {
#pragma unroll
      for (int it = 0; it < NV; ++it)
        if (kb + it * (64 / VR) + vrow >= Ltot) vreg[it] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int it = 0; it < NV; ++it) {
      *reinterpret_cast<half8_t*>(ldsK + (it * (64 / VR) + vrow) * STR + vcol * 16) = kreg[it];
      *reinterpret_cast<half8_t*>(ldsV + (it * (64 / VR) + vrow) * STR + vcol * 16) = vreg[it];
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_sched_barrier(0);
    fetch(blk + stride, Ltot - 1);                   // unconditional, so that what is in flight is known at every wait
    __builtin_amdgcn_sched_barrier(0);
    float4_t sacc[NC][2];
#pragma unroll
    for (int n = 0; n < NC; ++n) sacc[n][0] = sacc[n][1] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int kk = 0; kk < KSTEPS; ++kk) {
        const half8_t a = *reinterpret_cast<const half8_t*>(ldsK + (16 * h + c) * STR + kk * 64 + kq * 16);
#pragma unroll
        for (int n = 0; n < NC; ++n) sacc[n][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, qreg[n][kk], sacc[n][h], 0, 0, 0);
      }
    // Register i of block half h is key kb + 16 h + 4 kq + i.  The scores stay unscaled: the scale (> 0) goes into
    // the exponent's fused multiply-add, and the running maximum starts at a finite floor instead of -inf, so that
    // no case needs a select.
    const bool prefix = kb + 32 <= P;
    half8_t bp[NC];       // exp(S^T) as the B operand: slot (kq, 4 h + i) of the contraction is key 16 h + 4 kq + i
#pragma unroll
    for (int n = 0; n < NC; ++n) {
      float bm = M_FLOOR;
      if (!prefix) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int key = kb + 16 * h + 4 * kq + i;
            const int rel = key - P;
            const uint32_t word = (WIDE && rel >= 32) ? hi_bits[n] : lo_bits[n];
            const bool vis = (rel < 0) | ((key < Ltot) & (((word >> (rel & 31)) & 1u) != 0u));
            sacc[n][h][i] = vis ? sacc[n][h][i] : -INFINITY;
          }
      }
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) bm = fmaxf(bm, sacc[n][h][i]);
      bm = max16_32(bm);
      const float m_new = fmaxf(m_run[n], bm * scale_log2e);
      const float alpha = __builtin_amdgcn_exp2f(m_run[n] - m_new);
      float psum = 0.f;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float pv = __builtin_amdgcn_exp2f(fmaf(sacc[n][h][i], scale_log2e, -m_new));
          psum += pv;
          bp[n][4 * h + i] = (half_t)pv;
        }
      l_run[n] = l_run[n] * alpha + psum;            // this lane's keys; the four lanes of a column add theirs at the end
      m_run[n] = m_new;
#pragma unroll
      for (int db = 0; db < DB; ++db) o_acc[n][db] *= alpha;
    }
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      const half4_t lo = lds_read_tr16(vt_base + db * 32);
      const half4_t hi = lds_read_tr16(vt_base + 16 * STR + db * 32);
      const half8_t a = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
      for (int n = 0; n < NC; ++n) o_acc[n][db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, bp[n], o_acc[n][db], 0, 0, 0);
    }
  }

  // (m, l, O) of the waves with blocks through LDS
#pragma unroll
  for (int n = 0; n < NC; ++n) {
    l_run[n] = sum16_32(l_run[n]);
    if (kq == 0) ml[wave][16 * n + c] = float2_t{m_run[n], l_run[n]};
  }
  __builtin_amdgcn_wave_barrier();
  float* o_tile = reinterpret_cast<float*>(ldsK);
#pragma unroll
  for (int n = 0; n < NC; ++n)
#pragma unroll
    for (int db = 0; db < DB; ++db)
      *reinterpret_cast<float4_t*>(o_tile + (16 * n + c) * OSTR + 16 * db + 4 * kq) = o_acc[n][db];
  __syncthreads();
  constexpr int QW = HD / 4;                         // threads per column
  for (int id = threadIdx.x; id < NC * 16 * QW; id += NW * 64) {
    const int oc = id / QW, dq = id % QW;
    const int col = col0 + oc;
    if (col >= cols) break;
    float mx = M_FLOOR;
    float2_t w[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      w[i] = ml[i][oc];
      mx = fmaxf(mx, w[i][0]);
    }
    float den = 0.f;
    float4_t acc = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NW; ++i) {
      const float f = __builtin_amdgcn_exp2f(w[i][0] - mx);
      den += f * w[i][1];
      const float4_t o = *reinterpret_cast<const float4_t*>(reinterpret_cast<const float*>(slices[i]) + oc * OSTR + dq * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(f, o[e], acc[e]);
    }
    if (nsplit > 1) {
      // partials: O [H * T][nsplit][HD], then (m, l) [H * T][nsplit][2] (behind O, so that O is 16-byte aligned whatever their number)
      const long slot = ((long)g * cols + col) * nsplit + split;
      if (dq == 0) *reinterpret_cast<float2_t*>(part + (long)H * T * nsplit * HD + slot * 2) = float2_t{mx, den};
      *reinterpret_cast<float4_t*>(part + slot * HD + dq * 4) = acc;
    } else {
      const float inv = den > 0.f ? 1.f / den : 0.f;
      const int hr = (uint32_t)col * inv_T >> 16, t = col - hr * T;
      *reinterpret_cast<half4_t*>(out + ((long)t * H + g * rep + hr) * HD + dq * 4) =
          half4_t{(half_t)(acc[0] * inv), (half_t)(acc[1] * inv), (half_t)(acc[2] * inv), (half_t)(acc[3] * inv)};
    }
  }
}

// Adds the key splits: one thread per four output elements, the NS splits that are always in use requested at once; those that a long
// prefix adds (LONG: a grid of most > NS splits) eight at a time behind them.
template <int HD, int NS, bool LONG>
__global__ __launch_bounds__(256) void tree_attn_add_kernel(const float* __restrict__ part, half_t* __restrict__ out, int T, int H, TreeSplits splits,
                                                            const int32_t* __restrict__ len_dev, long cap, int Tk) {
  constexpr int QW = HD / 4, MORE = 8;
  const int id = blockIdx.x * 256 + threadIdx.x;
  const int row = id / QW, dq = id % QW;             // row = head * T + token
  if (row >= H * T) return;
  const int most = LONG ? splits.most : NS;
  const float* ml = part + (long)H * T * most * HD + (long)row * most * 2;
  const float* po = part + (long)row * most * HD + dq * 4;
  float2_t w[NS];
  float4_t o[NS];
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    w[i] = *reinterpret_cast<const float2_t*>(ml + 2 * i);
    o[i] = *reinterpret_cast<const float4_t*>(po + i * HD);
  }
  const int in_use = LONG ? tree_splits_in_use(tree_prefix(len_dev, cap, Tk), splits) : NS;
  float mx = M_FLOOR;
#pragma unroll
  for (int i = 0; i < NS; ++i) mx = fmaxf(mx, w[i][0]);
  float den = 0.f;
  float4_t acc = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NS; ++i) {
    const float f = __builtin_amdgcn_exp2f(w[i][0] - mx);
    den += f * w[i][1];
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] = fmaf(f, o[i][e], acc[e]);
  }
  for (int s0 = NS; s0 < in_use; s0 += MORE) {
    float2_t wm[MORE];
    float4_t om[MORE];
#pragma unroll
    for (int i = 0; i < MORE; ++i) {                 // (past the end the last one again, with a weight of zero)
      const int at = s0 + i < in_use ? s0 + i : in_use - 1;
      wm[i] = *reinterpret_cast<const float2_t*>(ml + 2 * at);
      om[i] = *reinterpret_cast<const float4_t*>(po + (long)at * HD);
    }
    float m_new = mx;
#pragma unroll
    for (int i = 0; i < MORE; ++i) m_new = fmaxf(m_new, wm[i][0]);
    const float alpha = __builtin_amdgcn_exp2f(mx - m_new);
    mx = m_new;
    den *= alpha;
    acc *= alpha;
#pragma unroll
    for (int i = 0; i < MORE; ++i) {
      const float f = s0 + i < in_use ? __builtin_amdgcn_exp2f(wm[i][0] - mx) : 0.f;
      den += f * wm[i][1];
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] = fmaf(f, om[i][e], acc[e]);
    }
  }
  const float inv = den > 0.f ? 1.f / den : 0.f;
  const int head = row / T, t = row - head * T;
  *reinterpret_cast<half4_t*>(out + ((long)t * H + head) * HD + dq * 4) =
      half4_t{(half_t)(acc[0] * inv), (half_t)(acc[1] * inv), (half_t)(acc[2] * inv), (half_t)(acc[3] * inv)};
}

// Key splits of a launch.  One where the keys are few: a second launch that adds the splits costs 2.0 us, a compute unit takes
// 3.2 us per 1000 keys of head dimension 64 and 5.7 of 128, and the live length is usually well below the capacity that
// the rule sees (14 heads of 64: one split 4.9 / 9.1 us at 560 / 2040 keys, eight 6.2 / 6.6; 28 heads
// of 128: one 8.2 / 11.1 / 16.9, four 8.9 / 9.2 / 10.8).  Otherwise as many as give every compute unit a workgroup at 32 query rows
// and a wave a block.  It does not look at the rows, so a query's result is the same bits whatever else is in the launch (but for long
// caches, launch_tree): above 32 rows of head dimension 128, where LDS holds one workgroup per compute unit, a workgroup takes 32 columns
// instead (40 rows behind 2048 keys, four splits: 13.4 us against 16.7 for 288 workgroups of 16).
int key_splits(int max_len, int H, int hd) {
  if (max_len <= (hd > 64 ? 768 : 2048)) return 1;
  const int fit = 256 / (2 * H), len = (max_len + 32 * NW - 1) / (32 * NW);
  static const int counts[] = {16, 12, 8, 6, 4, 3, 2};
  for (int n : counts)
    if (n <= fit && n <= len) return n;
  return 1;
}

template <int HD, bool WIDE>
int launch_tree(const void* q, const void* kc, const void* vc, const uint32_t* bits, const int32_t* len, void* out, int T,
                int Tk, int H, int G, long cap, int max_len, float scale, void* workspace, hipStream_t st) {
  constexpr int LONG_CACHE = 6144, MAX_LONG_SPLITS = 32;
  const int least = key_splits(max_len, H, HD), rep_T = H / G * T;
  int nc = HD > 64 && T > 32 ? 2 : 1;
  TreeSplits splits = {least, least, least, 0};
  uint32_t inv_G = 0;
  // Long caches: key_splits gives a few rows a handful of workgroups, each with thousands of keys (32 heads of 128 in 8 groups, one row
  // behind 8192 keys 27 us, 32768 84; 64 heads 45 and 152).  The rows then say how many splits fill the compute units and how many columns
  // a workgroup takes, the prefix how many of those splits are used.  The workgroups of a group and split read the same keys and go to
  // one XCD (35 heads in 5 groups, 27 rows behind 31451: 42 us, 75 spread over all of them).  By the least predicted time (us), fitted to 549
  // shapes in all their divisions (1 .. 64 rows behind 6 .. 32 thousand keys): rounds of the workgroups of an XCD, each the blocks of a wave,
  // the bytes that all of them read, a second launch and its partial results.  A cache is seldom full: the splits of three quarters of it are
  // used from half of it up, those of a quarter below, and the columns are those with the smaller loss in both.
  if (max_len > LONG_CACHE) {
    struct Cost {
      double start, block[2], add, parts, read;
    };
    constexpr Cost cost = HD > 64 ? Cost{1.63, {1.53, 1.79}, 6.9, 2.1e-6, 2.1e-9} : Cost{0., {0.66, 0.95}, 2.8, 4.9e-6, 0.55e-9};
    double us[2][2];
    int best[2][2];
    for (int c = 0; c < 2; ++c) {
      const int ny = (rep_T + 16 * c + 15) / (16 * c + 16);
      for (int l = 0; l < 2; ++l) {
        const int blocks = max_len / 128 * (l ? 3 : 1);
        us[c][l] = 1e30;
        for (int n = least; n <= MAX_LONG_SPLITS && (n == least || n * 16 <= blocks); ++n) {
          const int rounds = ((G * n + 7) / 8 * ny + 31) / 32, each = (blocks + n * NW - 1) / (n * NW);
          const double t = rounds * (cost.start + cost.block[c] * each) + (n > 1 ? cost.add + cost.parts * T * H * HD * n : 0.) +
                           cost.read * ny * G * blocks * (32. * HD * 4);
          if (t < us[c][l]) {
            us[c][l] = t;
            best[c][l] = n;
          }
        }
      }
    }
    const int c = us[1][0] / us[0][0] + us[1][1] / us[0][1] < 2. ? 1 : 0;
    nc = c + 1;
    splits.few = best[c][0];
    splits.most = best[c][1] > best[c][0] ? best[c][1] : best[c][0];
    splits.half = max_len / 2;
    if (G <= 48) inv_G = (65536 + G - 1) / G;          // (pair / G = pair inv_G >> 16 for up to 32 G + 7 pairs of up to 50 groups)
  }
  const int ny = (rep_T + 16 * nc - 1) / (16 * nc);
  const dim3 grid = inv_G ? dim3(8, ny, (G * splits.most + 7) / 8) : dim3(G, ny, splits.most);
  const float sl2 = scale * 1.4426950408889634f;
  const uint32_t inv_T = (65536 + T - 1) / T;          // col / T = col inv_T >> 16 for the at most 512 columns of a group
  float* part = static_cast<float*>(workspace);
  half_t* o = static_cast<half_t*>(out);
#define EAGLE_ATTN(NC)                                                                                              \
  hipLaunchKernelGGL((tree_attn_kernel<HD, NC, WIDE>), grid, dim3(NW * 64), 0, st, static_cast<const half_t*>(q),   \
                     static_cast<const half_t*>(kc), static_cast<const half_t*>(vc), bits, len, o, part, T, H, G, cap, sl2, Tk, inv_T, \
                     splits, inv_G)
  if (nc == 2) EAGLE_ATTN(2);
  else EAGLE_ATTN(1);
#undef EAGLE_ATTN
  const dim3 add((H * T * (HD / 4) + 255) / 256);
#define EAGLE_ATTN_ADD(NS)                                                                                                              \
  case NS:                                                                                                                              \
    if (splits.most > NS) hipLaunchKernelGGL((tree_attn_add_kernel<HD, NS, true>), add, dim3(256), 0, st, part, o, T, H, splits, len, cap, Tk); \
    else hipLaunchKernelGGL((tree_attn_add_kernel<HD, NS, false>), add, dim3(256), 0, st, part, o, T, H, splits, len, cap, Tk);            \
    break
  if (splits.most > 1) switch (least) {
    EAGLE_ATTN_ADD(1);
    EAGLE_ATTN_ADD(2);
    EAGLE_ATTN_ADD(3);
    EAGLE_ATTN_ADD(4);
    EAGLE_ATTN_ADD(6);
    EAGLE_ATTN_ADD(8);
    EAGLE_ATTN_ADD(12);
    EAGLE_ATTN_ADD(16);
    default: break;
  }
#undef EAGLE_ATTN_ADD
  return eagle_launch_status();
}

// ---- a prompt chunk in pieces of 32 rows ----
//
// A workgroup of eight waves owns up to four (query head, piece) pairs of a KV group: four heads of one piece, or with fewer
// heads per group several pieces.  K and V go through LDS in tiles of 128 keys; four waves take the first 64 keys of a tile, the other
// four the second, so that two waves of a SIMD work on the same rows, and the halves' (m, l, O) meet in LDS at the end.
// Per block of 32 keys a wave computes S^T = K Q^T with v_mfma_f32_32x32x16_f16 (rows = keys, columns = the 32 rows of its piece),
// runs the online softmax on its accumulator (a lane owns one row, its partner lane + 32 the other half of the keys) and feeds
// exp(S^T) straight back as the B operand of O^T += V^T P^T; only V needs a transposed read from LDS (ds_read_b64_tr_b16).
//
// A chunk has hundreds of pairs, so the keys are split over workgroups only where a few pairs would leave most of the GPU idle (O / l of
// a split in fp16, added by a second kernel: in fp32 128 rows behind 1536 keys, seven splits, take 20.6 us, so 17.3).  What bounds it: 2.5 us per tile of a workgroup, of which the matrix instructions are 0.9,
// and the last workgroups of a causal triangle.  Before, a workgroup held all heads of a group (seven waves) on tiles of 64 keys, one
// per compute unit, the longest twice the average, and every result went through partials and a merge; us per chunk
// (28 heads of 128 in 4 groups, K and V of 28 layers in turn in a graph; before / now): 2048 rows 98 / 52, 512 rows 24.8 / 14.8, 128 rows
// 13.9 / 7.6, 512 rows behind 1536 40 / 31; 14 heads of 64 in 2 groups, 2048 rows 37 / 26.  With K and V from HBM 2048 rows take 98 / 51, 512
// 24.7 / 15.4.
constexpr int CAUSAL_TILE = 128;

// cached rows before piece p (never past the cache, whatever the counter says: a graph replayed beyond the capacity
// would otherwise read beyond the last head's buffer), and rows that pieces p .. p + n - 1 see
__device__ inline int causal_length(const int32_t* len_dev, int p, long cap) {
  int P = len_dev[p];
  if (P > cap - 32) P = (int)(cap - 32);
  return P < 0 ? 0 : P;
}
__device__ inline int causal_rows(const int32_t* len_dev, int p, int n, int pieces, long cap) {
  int most = 0;
  for (int i = p; i < p + n && i < pieces; ++i) {
    const int rows = causal_length(len_dev, i, cap) + 32;
    most = rows > most ? rows : most;
  }
  return most;
}

// Key splits in use for `ntiles` tiles in a grid of `nsplit`, of `least` tiles or more: a cache much shorter than the launch was sized for,
// and the shorter pieces of a chunk, pay for few partial results.
__device__ inline int causal_splits(int ntiles, int nsplit, int least) {
  int tpw = (ntiles + nsplit - 1) / nsplit;
  tpw = tpw > least ? tpw : least;
  return (ntiles + tpw - 1) / tpw;
}

constexpr int MAX_CAUSAL_SPLITS = 64;     // what the workspace holds

template <int V>
struct Stage { static constexpr int value = V; };

// SEVERAL: more than one piece in a workgroup (pp > 1).  The tiles then hold rows past the end of a wave's own piece.  Their probabilities
// are zero, but zero times an infinity is not: the lanes that fetch such a row for the transposing read of V fetch zeros instead.
template <int HD, int DEPTH, bool SEVERAL>
__global__ __launch_bounds__(512, 2) void causal_attn_kernel(
    const half_t* __restrict__ q, const half_t* __restrict__ kc, const half_t* __restrict__ vc,
    const int32_t* __restrict__ len_dev, half_t* __restrict__ out, half_t* __restrict__ part_o, float* __restrict__ part_ml, int H,
    int G, long cap, float scale_log2e, int pieces, int hp, int pp, int least) {
  constexpr int KSTEPS = HD / 16;       // MFMA steps over the head dimension for S
  constexpr int DB = HD / 32;           // 32-wide blocks of the head dimension for O
  constexpr int STR = HD * 2 + 16;      // LDS row stride in bytes (pad: conflict-free reads)
  constexpr int VEC_ROW = HD / 8;       // 16-byte vectors per K/V row
  constexpr int KTT = CAUSAL_TILE;
  constexpr int NVU = KTT * VEC_ROW / 512;        // vectors of K (or V) per thread
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * KTT * STR + (SEVERAL ? HD * 2 : 0)];
  __shared__ float2_t ml_half[4][32];
  const unsigned char* zeros = lds + 2 * KTT * STR;
  if (SEVERAL && threadIdx.x < HD / 2) reinterpret_cast<uint32_t*>(lds + 2 * KTT * STR)[threadIdx.x] = 0u;   // (read behind the barriers of a tile)
  unsigned char* ldsK = lds;
  unsigned char* ldsV = lds + KTT * STR;
  const int rep = H / G, quads = (rep + hp - 1) / hp;
  const int g = blockIdx.x / quads, hq = blockIdx.x % quads;
  const int split = blockIdx.z, nsplit = gridDim.z;      // (the slowest: splits that are not in use leave no gaps between the others)
  const int group = gridDim.y - 1 - blockIdx.y;   // (the last pieces see the most keys: dispatched first)
  const int tid = threadIdx.x;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wave = wid & 3, khalf = wid >> 2;
  const int ql = lane & 31, hb = lane >> 5;
  // this wave's head of the group and piece; a wave that has none carries keys and values like the others
  int hin = hq * hp + wave % hp, piece = group * pp + wave / hp;
  const bool live = hin < rep && piece < pieces && wave < hp * pp;
  if (!live) {
    hin = 0;
    piece = group * pp;
  }
  const int head = g * rep + hin;
  const int P = causal_length(len_dev, piece, cap);
  const int Ltot = causal_rows(len_dev, group * pp, pp, pieces, cap);
  const int ntiles = (Ltot + KTT - 1) / KTT;
  const int own = live ? P + 32 : 0;       // keys up to here concern this wave's rows
  const int nactive = causal_splits(ntiles, nsplit, least);
  if (split >= nactive) return;
  half8_t qreg[KSTEPS];
  const half_t* qp = q + ((long)head * pieces * 32 + piece * 32 + ql) * HD;
#pragma unroll
  for (int kk = 0; kk < KSTEPS; ++kk) qreg[kk] = *reinterpret_cast<const half8_t*>(qp + kk * 16 + hb * 8);

  float m_run = M_FLOOR, l_run = 0.f;
  // this lane's address for the transposing loads of V: within 16 lanes, lane s asks for key row s / 4 at the four d
  // columns 4 (s % 4) .. + 3 of the group's 16 and gets four keys of its own d
  const int vt_row = 4 * hb + ((lane & 15) >> 2);
  const unsigned char* vt_base = ldsV + (64 * khalf + vt_row) * STR + (16 * ((lane >> 4) & 1) + 4 * (lane & 3)) * 2;
  float16_t o_acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; ++i) o_acc[db][i] = 0.f;
  const half_t* kbase_ptr = kc + (long)g * cap * HD;
  const half_t* vbase_ptr = vc + (long)g * cap * HD;
  half8_t kreg[DEPTH][NVU], vreg[DEPTH][NVU];
  auto fetch = [&](auto S, int tile) {
    constexpr int st = decltype(S)::value;
    const int kb = tile * KTT;
#pragma unroll
    for (int it = 0; it < NVU; ++it) {
      const int v = tid + it * 512;
      int kidx = kb + v / VEC_ROW;
      if (kidx > Ltot - 1) kidx = Ltot - 1;
      kreg[st][it] = *reinterpret_cast<const half8_t*>(kbase_ptr + (long)kidx * HD + v % VEC_ROW * 8);
      vreg[st][it] = *reinterpret_cast<const half8_t*>(vbase_ptr + (long)kidx * HD + v % VEC_ROW * 8);
    }
  };
  auto stash = [&](auto S) {
    constexpr int st = decltype(S)::value;
#pragma unroll
    for (int it = 0; it < NVU; ++it) {
      const int v = tid + it * 512;
      *reinterpret_cast<half8_t*>(ldsK + v / VEC_ROW * STR + v % VEC_ROW * 16) = kreg[st][it];
      *reinterpret_cast<half8_t*>(ldsV + v / VEC_ROW * STR + v % VEC_ROW * 16) = vreg[st][it];
    }
  };
  // every fetch is issued whether or not its tile exists (the last one again), so that what is in flight is known at every wait
  auto tile_at = [&](int t) { return t < ntiles ? t : ntiles - 1; };
  __builtin_amdgcn_sched_barrier(0);
  fetch(Stage<0>{}, split);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (DEPTH > 1) fetch(Stage<1>{}, tile_at(split + nactive));
  __builtin_amdgcn_sched_barrier(0);
  auto do_tile = [&](auto S, int tile) {
    const int kb = tile * KTT + 64 * khalf;
    __syncthreads();
    stash(S);
    fetch(S, tile_at(tile + DEPTH * nactive));
    __syncthreads();
    if (kb >= own) return;                        // (a wave)
    float16_t sacc[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 16; ++i) sacc[h][i] = 0.f;
#pragma unroll
    for (int kk = 0; kk < KSTEPS; ++kk)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const half8_t a = *reinterpret_cast<const half8_t*>(ldsK + (64 * khalf + 32 * h + ql) * STR + kk * 32 + hb * 16);
        sacc[h] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qreg[kk], sacc[h], 0, 0, 0);
      }
    // accumulator register i of this lane is key 8*(i/4) + 4*hb + i%4 of its block of 32; unscaled, as in the kernel above
    float bm = M_FLOOR;
    if (kb + 64 > P) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = kb + 32 * h + 8 * (i >> 2) + 4 * hb + (i & 3);
          sacc[h][i] = key - P <= ql ? sacc[h][i] : -INFINITY;
        }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 16; ++i) bm = fmaxf(bm, sacc[h][i]);
    bm = max32(bm);
    const float m_new = fmaxf(m_run, bm * scale_log2e);
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    float psum = 0.f;
    half8_t bp[2][2];       // exp(S^T) as the B operand of the O products: step u = registers 8u..8u+7
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float pv = __builtin_amdgcn_exp2f(fmaf(sacc[h][i], scale_log2e, -m_new));
        psum += pv;
        bp[h][i >> 3][i & 7] = (half_t)pv;
      }
    l_run = l_run * alpha + psum;                 // this lane's keys; its partner's are added at the end
    m_run = m_new;
    if (alpha != 1.f) {
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o_acc[db][i] *= alpha;
    }
    const int left = own - kb;                    // rows of this half tile before the wave's end
    auto v_rows = [&](int c) { return !SEVERAL || vt_row < left - c ? vt_base + c * STR : zeros; };
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int db = 0; db < DB; ++db) {
          const half4_t lo = lds_read_tr16(v_rows(32 * h + 16 * u) + db * 64);
          const half4_t hi = lds_read_tr16(v_rows(32 * h + 16 * u + 8) + db * 64);
          const half8_t a = half8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
          o_acc[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, bp[h][u], o_acc[db], 0, 0, 0);
        }
  };
  int t0 = split;
  for (; t0 + (DEPTH - 1) * nactive < ntiles; t0 += DEPTH * nactive) {
    do_tile(Stage<0>{}, t0);
    if constexpr (DEPTH > 1) do_tile(Stage<1>{}, t0 + nactive);
  }
  if constexpr (DEPTH > 1)
    if (t0 < ntiles) do_tile(Stage<0>{}, t0);
  l_run = sum32(l_run);
  // the second half of the waves hands its (m, l, O) to the first through LDS
  __syncthreads();
  constexpr int OS = HD + 4;
  static_assert(4 * 32 * OS * 4 <= 2 * KTT * STR, "the halves' tiles do not fit over K and V");
  float* half_o = reinterpret_cast<float*>(lds) + wave * (32 * OS) + ql * OS + 4 * hb;
  if (khalf) {
    if (hb == 0) ml_half[wave][ql] = float2_t{m_run, l_run};
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        *reinterpret_cast<float4_t*>(half_o + db * 32 + 8 * i4) =
            float4_t{o_acc[db][4 * i4], o_acc[db][4 * i4 + 1], o_acc[db][4 * i4 + 2], o_acc[db][4 * i4 + 3]};
  }
  __syncthreads();
  if (khalf) return;
  {
    const float2_t other = ml_half[wave][ql];
    const float m_new = fmaxf(m_run, other[0]);
    const float fa = __builtin_amdgcn_exp2f(m_run - m_new), fb = __builtin_amdgcn_exp2f(other[0] - m_new);
    l_run = l_run * fa + other[1] * fb;
    m_run = m_new;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4) {
        const float4_t o = *reinterpret_cast<const float4_t*>(half_o + db * 32 + 8 * i4);
#pragma unroll
        for (int e = 0; e < 4; ++e) o_acc[db][4 * i4 + e] = o_acc[db][4 * i4 + e] * fa + o[e] * fb;
      }
  }
  if (nactive > 1) {
    if (!live) return;
    const long slot = (((long)piece * H + head) * nsplit + split) * 32 + ql;
    if (hb == 0) {
      part_ml[slot * 2 + 0] = m_run;
      part_ml[slot * 2 + 1] = l_run;
    }
    // O / l, a weighted mean of values: O itself grows with the keys of the split, past what fp16 holds
    const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
    half_t* po = part_o + slot * HD;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int i4 = 0; i4 < 4; ++i4)
        *reinterpret_cast<half4_t*>(po + db * 32 + 8 * i4 + 4 * hb) =
            half4_t{(half_t)(o_acc[db][4 * i4 + 0] * inv), (half_t)(o_acc[db][4 * i4 + 1] * inv), (half_t)(o_acc[db][4 * i4 + 2] * inv),
                    (half_t)(o_acc[db][4 * i4 + 3] * inv)};
    return;
  }
  // one split: the rows as they lie in memory, through the wave's part of LDS (other lanes' reads of half_o come first)
  __builtin_amdgcn_wave_barrier();
  unsigned char* mine = lds + wave * (32 * OS * 4);
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i4 = 0; i4 < 4; ++i4)
      *reinterpret_cast<half4_t*>(mine + ql * STR + (db * 32 + 8 * i4 + 4 * hb) * 2) =
          half4_t{(half_t)(o_acc[db][4 * i4 + 0] * inv), (half_t)(o_acc[db][4 * i4 + 1] * inv), (half_t)(o_acc[db][4 * i4 + 2] * inv),
                  (half_t)(o_acc[db][4 * i4 + 3] * inv)};
  __builtin_amdgcn_wave_barrier();
  if (!live) return;
#pragma unroll
  for (int it = 0; it < 32 * VEC_ROW / 64; ++it) {
    const int v = lane + it * 64, row = v / VEC_ROW, c = v % VEC_ROW;
    *reinterpret_cast<half8_t*>(out + ((long)(piece * 32 + row) * H + head) * HD + c * 8) =
        *reinterpret_cast<const half8_t*>(mine + row * STR + c * 16);
  }
}

// Adds the splits of a piece: a thread per eight output elements, every split in use requested at once.
template <int HD>
__global__ __launch_bounds__(256) void causal_add_kernel(const half_t* __restrict__ part_o, const float* __restrict__ part_ml,
                                                         half_t* __restrict__ out, int H, int nsplit, const int32_t* __restrict__ len_dev,
                                                         long cap, int pp, int least) {
  constexpr int VR = HD / 8, MOST = 8;
  const int piece = blockIdx.z, pieces = gridDim.z;
  const int rows = causal_rows(len_dev, piece / pp * pp, pp, pieces, cap);
  const int nact = causal_splits((rows + CAUSAL_TILE - 1) / CAUSAL_TILE, nsplit, least);
  if (nact == 1) return;                           // written by the workgroup itself
  const int id = blockIdx.x * 256 + threadIdx.x;   // (head, row, vector)
  const int hr = id / VR, c = id % VR;
  if (hr >= H * 32) return;
  const int head = hr >> 5, row = hr & 31;
  const long slot = ((long)piece * H + head) * nsplit * 32 + row;
  float m_run = M_FLOOR, l_run = 0.f;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  for (int s0 = 0; s0 < nact; s0 += MOST) {
    float2_t ml[MOST];
    half8_t o[MOST];
#pragma unroll
    for (int k = 0; k < MOST; ++k)
      if (s0 + k < nact) {
        const long at = slot + (long)(s0 + k) * 32;
        ml[k] = *reinterpret_cast<const float2_t*>(part_ml + at * 2);
        o[k] = *reinterpret_cast<const half8_t*>(part_o + at * HD + c * 8);
      }
    float mx = m_run;
#pragma unroll
    for (int k = 0; k < MOST; ++k)
      if (s0 + k < nact) mx = fmaxf(mx, ml[k][0]);
    const float alpha = __builtin_amdgcn_exp2f(m_run - mx);
    m_run = mx;
    l_run *= alpha;
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] *= alpha;
#pragma unroll
    for (int k = 0; k < MOST; ++k)
      if (s0 + k < nact) {
        const float f = __builtin_amdgcn_exp2f(ml[k][0] - mx) * ml[k][1];
        l_run += f;
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = fmaf(f, (float)o[k][e], acc[e]);
      }
  }
  const float inv = l_run > 0.f ? 1.f / l_run : 0.f;
  half8_t r;
#pragma unroll
  for (int e = 0; e < 8; ++e) r[e] = (half_t)(acc[e] * inv);
  *reinterpret_cast<half8_t*>(out + ((long)(piece * 32 + row) * H + head) * HD + c * 8) = r;
}

template <int HD>
int launch_causal(const void* q, const void* kc, const void* vc, const int32_t* len, void* out, int pieces, int H, int G,
                  long cap, int max_len, float scale, void* workspace, hipStream_t st) {
  const int rep = H / G, hp = rep < 4 ? rep : 4, gx = G * ((rep + hp - 1) / hp);
  // With fewer than four heads per group a workgroup can take several pieces, so that its waves share the tiles; the keys can be split.  The
  // division with the least predicted time (us): a workgroup costs its start and its tiles, whatever part of its waves is busy with
  // them, the launch as many of those as there are rounds (fewer where a causal triangle leaves later workgroups short), splits a second
  // launch and their partial results.  Fitted to 2424 shapes timed in all their divisions (32 .. 2048 rows behind 16 .. 32768 keys), 7.4 % rms;
  // its choice is 0.5 % longer than the best of them on average, 3 % at the 95th percentile, where filling the compute units once
  // took 2.6 and 16, and counting on a part of a round 14 and 100 (28 heads, 224 rows behind 8000, 280 workgroups 73 us, 224 51).
  struct Cost {
    double tile, start, add, parts, several;
  };
  constexpr Cost cost = HD > 64 ? Cost{2.27, 0.89, 4.0, 1.34e-6, 0.} : Cost{1.33, 0.43, 2.8, 1.48e-6, 0.058};
  const int rows = pieces * 32, tiles = (max_len + CAUSAL_TILE - 1) / CAUSAL_TILE;
  const double triangle = rows < max_len ? 1.5 * rows / max_len : 1.5;
  int pp = 1, nsplit = 1, least = 1;
  double least_us = 1e30;
  for (int n = 1; n <= 4 / hp && n <= pieces; ++n) {
    const int units = gx * ((pieces + n - 1) / n);
    for (int tpw = tiles, s = 1; s <= MAX_CAUSAL_SPLITS;) {
      const double fill = units * s / 256., whole = (units * s + 255) / 256, rounds = whole > 1. ? whole - triangle * (whole - fill) : 1.;
      const double us = rounds * (cost.start + (cost.tile + (n > 1 ? cost.several : 0.)) * tpw) +
                        (s > 1 ? cost.add + cost.parts * rows * H * HD * s : 0.);
      if (us < least_us) {
        least_us = us;
        pp = n;
        nsplit = s;
        least = units * s > 256 ? 12 : 4;            // (more than one round of workgroups only while the splits are long)
        least = tpw < least ? tpw : least;
      }
      if (tpw == 1) break;
      s = (tiles + tpw - 2) / (tpw - 1);             // the fewest splits with fewer tiles each
      tpw = (tiles + s - 1) / s;
    }
  }
  const int nz = (pieces + pp - 1) / pp;
  float* part_ml = static_cast<float*>(workspace);
  half_t* part_o = reinterpret_cast<half_t*>(part_ml + (size_t)pieces * H * nsplit * 32 * 2);
#define EAGLE_CAUSAL(SEVERAL)                                                                                                              \
  hipLaunchKernelGGL((causal_attn_kernel<HD, HD == 64 ? 2 : 1, SEVERAL>), dim3(gx, nz, nsplit), dim3(512), 0, st,                          \
                     static_cast<const half_t*>(q), static_cast<const half_t*>(kc), static_cast<const half_t*>(vc), len,                   \
                     static_cast<half_t*>(out), part_o, part_ml, H, G, cap, scale * 1.4426950408889634f, pieces, hp, pp, least)
  if (pp > 1) EAGLE_CAUSAL(true);
  else EAGLE_CAUSAL(false);
#undef EAGLE_CAUSAL
  if (nsplit > 1)
    hipLaunchKernelGGL(causal_add_kernel<HD>, dim3((H * 32 * (HD / 8) + 255) / 256, 1, pieces), dim3(256), 0, st, part_o, part_ml,
                       static_cast<half_t*>(out), H, nsplit, len, cap, pp, least);
  return eagle_launch_status();
}

__global__ void rope_table_kernel(const int32_t* __restrict__ pos, const float* __restrict__ inv_freq,
                                  float scale, float* __restrict__ out, int T, int half) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= T * half) return;
  const int i = idx % half;
  const int t = idx / half;
  const float lf = scale * inv_freq[i];
  const float theta = lf * (float)pos[t];
  float sn, cs;
  sincosf(theta, &sn, &cs);
  out[2 * idx] = cs;
  out[2 * idx + 1] = sn;
}

}  // namespace

EAGLE_EXPORT size_t eagle_tree_attention_workspace_bytes(int H, int hd, int max_len) {
  if (H < 1 || hd < 1 || max_len < 1) return 0;
  // 64 key splits of 32 rows: what a piece of a prompt chunk may use (a tree up to 32 splits)
  return (size_t)H * 64 * 32 * (hd + 2) * sizeof(float);
}

EAGLE_EXPORT int eagle_tree_attention_f16(const void* q, const void* k_cache, const void* v_cache,
                                          const uint32_t* tree_mask_bits,
                                          const int32_t* cache_len_dev, void* out, int T, int H,
                                          int G, int hd, long capacity, int max_len, float scale,
                                          void* workspace, size_t workspace_bytes,
                                          eagle_stream_t stream) {
  if (!q || !k_cache || !v_cache || !tree_mask_bits || !cache_len_dev || !out) return EAGLE_ERR_NULL;
  if (T < 1 || T > EAGLE_MAX_TREE || H < 1 || G < 1 || (H % G) != 0 || (H / G) > 8 ||
      (hd != 64 && hd != 128) || max_len < T || max_len > capacity || !(scale > 0.f))
    return EAGLE_ERR_SHAPE;
  if (!eagle_aligned16(q) || !eagle_aligned16(k_cache) || !eagle_aligned16(v_cache) ||
      !eagle_aligned16(out))
    return EAGLE_ERR_ALIGN;
  if (!workspace || !eagle_aligned16(workspace) ||
      workspace_bytes < eagle_tree_attention_workspace_bytes(H, hd, max_len))
    return EAGLE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (hd == 128)
    return launch_tree<128, false>(q, k_cache, v_cache, tree_mask_bits, cache_len_dev, out, T, T, H, G, capacity, max_len, scale,
                                   workspace, st);
  return launch_tree<64, false>(q, k_cache, v_cache, tree_mask_bits, cache_len_dev, out, T, T, H, G, capacity, max_len, scale,
                                workspace, st);
}

EAGLE_EXPORT int eagle_draft_attention_f16(const void* q, const void* k_cache, const void* v_cache,
                                           const uint32_t* mask_words, const int32_t* cache_len_dev,
                                           void* out, int T, int Tk, int H, int G, int hd,
                                           long capacity, int max_len, float scale, void* workspace,
                                           size_t workspace_bytes, eagle_stream_t stream) {
  if (!q || !k_cache || !v_cache || !mask_words || !cache_len_dev || !out) return EAGLE_ERR_NULL;
  if (T < 1 || T > EAGLE_MAX_TREE || Tk < 1 || Tk > 2 * EAGLE_MAX_TREE || H < 1 || G < 1 ||
      (H % G) != 0 || (H / G) > 8 || (hd != 64 && hd != 128) || max_len < Tk || max_len > capacity || !(scale > 0.f))
    return EAGLE_ERR_SHAPE;
  if (!eagle_aligned16(q) || !eagle_aligned16(k_cache) || !eagle_aligned16(v_cache) ||
      !eagle_aligned16(out))
    return EAGLE_ERR_ALIGN;
  if (!workspace || !eagle_aligned16(workspace) ||
      workspace_bytes < eagle_tree_attention_workspace_bytes(H, hd, max_len))
    return EAGLE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (hd == 128)
    return launch_tree<128, true>(q, k_cache, v_cache, mask_words, cache_len_dev, out, T, Tk, H, G, capacity, max_len, scale,
                                  workspace, st);
  return launch_tree<64, true>(q, k_cache, v_cache, mask_words, cache_len_dev, out, T, Tk, H, G, capacity, max_len, scale,
                               workspace, st);
}

EAGLE_EXPORT size_t eagle_tree_attention_wide_workspace_bytes(int T, int H, int hd, int max_len) {
  if (T < 1 || T > EAGLE_MAX_TREE_SLOTS) return 0;
  return (size_t)((T + 31) / 32) * eagle_tree_attention_workspace_bytes(H, hd, max_len);
}

EAGLE_EXPORT int eagle_tree_attention_wide_f16(const void* q, const void* k_cache, const void* v_cache,
                                               const uint32_t* mask_words, const int32_t* cache_len_dev,
                                               void* out, int T, int Tk, int H, int G, int hd,
                                               long capacity, int max_len, float scale, void* workspace,
                                               size_t workspace_bytes, eagle_stream_t stream) {
  if (!q || !k_cache || !v_cache || !mask_words || !cache_len_dev || !out) return EAGLE_ERR_NULL;
  if (T < 1 || T > EAGLE_MAX_TREE_SLOTS || Tk < 1 || Tk > EAGLE_MAX_TREE_SLOTS || H < 1 || G < 1 ||
      (H % G) != 0 || (H / G) > 8 || (hd != 64 && hd != 128) || max_len < Tk || max_len > capacity || !(scale > 0.f))
    return EAGLE_ERR_SHAPE;
  if (!eagle_aligned16(q) || !eagle_aligned16(k_cache) || !eagle_aligned16(v_cache) ||
      !eagle_aligned16(out))
    return EAGLE_ERR_ALIGN;
  if (!workspace || !eagle_aligned16(workspace) ||
      workspace_bytes < eagle_tree_attention_wide_workspace_bytes(T, H, hd, max_len))
    return EAGLE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (hd == 128)
    return launch_tree<128, true>(q, k_cache, v_cache, mask_words, cache_len_dev, out, T, Tk, H, G, capacity, max_len, scale,
                                  workspace, st);
  return launch_tree<64, true>(q, k_cache, v_cache, mask_words, cache_len_dev, out, T, Tk, H, G, capacity, max_len, scale,
                               workspace, st);
}

EAGLE_EXPORT size_t eagle_causal_attention_workspace_bytes(int R, int H, int hd, int max_len) {
  if (R < 32 || (R % 32) != 0) return 0;
  return (size_t)(R / 32) * eagle_tree_attention_workspace_bytes(H, hd, max_len);
}

EAGLE_EXPORT int eagle_causal_attention_f16(const void* q, const void* k_cache, const void* v_cache,
                                            const int32_t* piece_len_dev, void* out, int R, int H, int G,
                                            int hd, long capacity, int max_len, float scale,
                                            void* workspace, size_t workspace_bytes,
                                            eagle_stream_t stream) {
  if (!q || !k_cache || !v_cache || !piece_len_dev || !out) return EAGLE_ERR_NULL;
  if (R < 32 || (R % 32) != 0 || R > EAGLE_MAX_CHUNK || H < 1 || G < 1 || (H % G) != 0 ||
      (H / G) > 8 || (hd != 64 && hd != 128) || max_len < 32 || max_len > capacity || !(scale > 0.f))
    return EAGLE_ERR_SHAPE;
  if (!eagle_aligned16(q) || !eagle_aligned16(k_cache) || !eagle_aligned16(v_cache) ||
      !eagle_aligned16(out))
    return EAGLE_ERR_ALIGN;
  if (!workspace || !eagle_aligned16(workspace) ||
      workspace_bytes < eagle_causal_attention_workspace_bytes(R, H, hd, max_len))
    return EAGLE_ERR_WORKSPACE;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (hd == 128)
    return launch_causal<128>(q, k_cache, v_cache, piece_len_dev, out, R / 32, H, G, capacity, max_len, scale, workspace, st);
  return launch_causal<64>(q, k_cache, v_cache, piece_len_dev, out, R / 32, H, G, capacity, max_len, scale, workspace, st);
}

EAGLE_EXPORT int eagle_rope_table_f32(const int32_t* positions, const float* inv_freqs,
                                      float scaling_factor, int T, int half_dim, float* out,
                                      eagle_stream_t stream) {
  if (!positions || !inv_freqs || !out) return EAGLE_ERR_NULL;
  if (T < 1 || T > EAGLE_MAX_CHUNK || half_dim < 1) return EAGLE_ERR_SHAPE;
  if (!eagle_aligned16(out)) return EAGLE_ERR_ALIGN;
  const int total = T * half_dim;
  hipLaunchKernelGGL(rope_table_kernel, dim3((total + 255) / 256), dim3(256), 0,
                     static_cast<hipStream_t>(stream), positions, inv_freqs, scaling_factor, out, T,
                     half_dim);
  return eagle_launch_status();
}
