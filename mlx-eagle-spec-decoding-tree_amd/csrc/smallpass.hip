// The quantised product for a pass of at most 16 rows through a SMALL model (the drafter's passes
// of the tree loop: 8 rows, layers of a few MB, where every launch is launch latency and the
// number of dependent launches per layer is what counts), with the operators around the product
// folded in so that a decoder layer needs four of these launches and no norm / add launch:
//
//   out = (RMSNorm(x, norm_w) or x) . W^T  (+ bias)              q|k|v
//   out = residual + fp16(x . W^T)                               o and down projections, in place on h
//   out = silu(g) * u,  (g | u) = (RMSNorm(x) or x) . Wgu^T      gate|up, interleaved 16-row tiles
//   q [H,T,hd], cache rows = rope(RMSNorm(x) . Wqkv^T + bias)    q|k|v with rotation and cache append
//
// (mlx_llama.py:195-196, 214-215, 225-249).
//
//   * A workgroup owns one weight tile of 16 rows (a (gate, up) pair for SwiGLU, the two halves of a
//     head that a rotation pairs for rope); its four, eight or sixteen waves deal the 128-column
//     chunks of K among themselves (at most three each) and add their tiles in LDS.  Every request
//     of a wave (weights, scales, its columns of x as the B operand of v_mfma_f32_16x16x32_f16) is
//     in flight together; there is no loop over K.
//   * Up to 8 rows of x leave half of the x operand empty.  Where the workgroups are few, a tile is then 8 weight rows, with the even
//     quantisation groups of K in its first eight columns and the odd ones in the others (and so the rows of x): twice the
//     workgroups, each with half the instructions of a product; half of the products, x of one group with weights of the
//     other, is dropped.  The sums are the same bits: a tile of 16 keeps two sums, of the even and of the odd groups.
//   * The norm is folded into x as it was loaded (whole rows, every lane columns of its own; in the operand layout
//     half the lanes hold nothing when T <= 8): each wave multiplies x with the norm weights and with powers of two that keep
//     its columns in fp16's range, and sums their squares; the powers and the row's 1 / rms go onto the sums at the end, where the
//     waves meet anyway.  No launch, no pass over memory and no barrier for it (8 rows, us in a graph, with the row sums added across
//     the waves before the product / so: gate|up of K 896 4.68 / 4.46, q|k|v with the rotation 3.44 / 3.18, 16 rows of 2048 -> 22016 13.4 / 12.3;
//     4.0 without a norm).  Error against 64 bits: that of w x / rms rounded once, 2.9e-4 of the result, also beside a column of 30000 where
//     the others are 0.004 (with w x / rms itself in fp16 1.6e-3 .. 4e-3 there: subnormal numbers).
//   * The weights are never rounded: the matrix instructions multiply x with the integers q (exact in
//     fp16, through the fp8 conversion) a quantisation group at a time, and with ones for the group's
//     sum of x; scale and bias are applied to the two sums in fp32.
//
// Measured on the way (8 rows, the 0.5B drafter's shapes, launches back to back in a graph):
//   - one wave per tile over the whole K: 2500 instructions on one wave per SIMD, 15 us per launch;
//   - K over the waves, loads under conditions (zero for what a wave does not own): the requests
//     of a wave wait for one another where the branches join; time grows by 1.1 us per chunk;
//   - unconditional loads, 16 bytes per lane straight into the operand layout: the time follows
//     the number of cache lines the load instructions of a compute unit touch (x: 64 per chunk,
//     scales 16 per 2-byte load), 7.8 us for the down projection; shaped as below: 5.7 us;
//   - a whole layer as ONE resident grid with grid-wide barriers between the products: a barrier
//     plus the first load behind it costs what a launch costs (56 us per layer against 33 us for
//     the launches it replaced).
#include "common.h"

namespace {

struct SmallArgs {
  const half_t* x;          // [T, K]
  const half_t* norm_w;     // [K] or nullptr
  const uint32_t* w;        // [N, K / 8]
  const half_t* s;          // [N, K / 64]
  const half_t* b;
  const half_t* bias;       // [N] or nullptr
  const half_t* residual;   // [T, N] or nullptr
  half_t* out;              // [T, N] ([T, N / 2] for SwiGLU)
  float eps, inv_k;         // inv_k = 1 / K
  int T, N, K;
  // rope form: (cos, sin) table [T, hd / 2, 2], rotated q [H, T, hd], caches [G, cap, hd], *len_dev = row of
  // the first new K / V row
  const float* rope_cs;
  half_t* q_out;
  half_t* k_cache;
  half_t* v_cache;
  const int32_t* len_dev;
  int H, G, hd;
  long cap;
};

enum { SMALL_PLAIN = 0, SMALL_SWIGLU = 1, SMALL_ROPE = 2 };

// NW waves per workgroup, at most MAXC chunks of 128 columns per wave (a wave requests MAXC whatever it owns:
// the smallest number that serves K), RP passes of four x rows
// (1: T <= 4, 2: T <= 8, 4: T <= 16).  MODE: one tile per workgroup (plain / residual), a (gate, up) tile pair
// 16 rows apart with the SwiGLU epilogue, or two tiles of one head half a head apart (the two
// halves a rotation pairs) with the rope epilogue.  Lane (r = lane % 16, kq = lane / 16) of a wave
// loads, per chunk, weight row r columns 32 kq .. + 32 (one 16-byte load, four packed words): two lanes
// per quantisation group.  Two half-wave swaps of words deal them so that a word is of one group in all
// four lanes of a row: after them word 2 g + j of lane (r, kq) is columns 64 g + 32 (kq % 2) +
// 16 (kq / 2) + 8 j of the chunk, and x row r is read at the same columns.  x is the A operand, the
// weights are B: the accumulator of lane (r, kq) is x rows 4 kq .. + 4 of weight row r, whose scale and
// bias are one value per lane.
//
// What bounds this kernel is the instructions of a wave, one after the other at about five cycles each (weights that are in the L2
// already save 0.3 us of 5): wave-uniform values are kept scalar, addresses are a uniform base and 32 bits per lane, the
// epilogue is spread over the threads.  8 rows of the 0.5B shapes, us in a graph before / after that: gate|up + norm 5.4 / 4.7, q|k|v 3.9 / 3.5,
// down 4.7 / 4.55, 2048 -> 8192 5.45 / 5.1, one row of 3584 -> 3584 4.4 / 4.0 (from the host a call takes as long: 4.8 and 4.4 .. 4.75, no shorter than before).
// Next to that it is the number of cache lines its load instructions touch per compute
// unit, so every request is shaped for few lines: x is read with whole rows of a chunk per
// instruction (four rows x 256 bytes) and brought into the operand layout through a per-wave LDS
// buffer; the two scales (biases) of a chunk come as one 4-byte load for the three chunks of a
// wave at once and are handed to the lanes that need them with a lane shuffle.
constexpr int SMALL_MAXC = 3;
constexpr int SMALL_RED = 16 + 4;          // floats per x row of a wave's tile
constexpr int SMALL_XROW = 256 + 16;       // bytes per staged x row: 128 columns, padded against bank conflicts

// a load at a uniform address plus 32 bits of a lane's own
template <typename T>
__device__ inline T small_load(const void* base, uint32_t at) {
  return *reinterpret_cast<const T*>(static_cast<const char*>(base) + at);
}

// (four waves per SIMD in the launch bounds: with more registers to give away the compiler puts the products into accumulation registers
// and reads them back, 48 instructions of gate|up; the builds that need more than 128 take two)
template <int NW, int MAXC, int RP, int MODE, bool NORM, bool HALF>
__global__ __launch_bounds__(NW * 64, NW <= 8 && RP == 4 && MAXC == 3 ? 2 : 4) void qmm_small_kernel(SmallArgs a) {
  constexpr int NT = MODE == SMALL_PLAIN ? 1 : 2;
  // a slice per wave: first its x, then (written by the same wave) its weights, then its tiles
  // Whether weights are loaded by whole 64-byte pieces (four lanes of a row next to each other, a quarter of the cache
  // lines per load) and dealt to the lanes through LDS: where a wave has several loads in flight and one tile (8 rows, us when it
  // came, without / with: 2048 -> 8192 5.6 / 5.3, 3072 -> 4096 4.9 / 4.7; gate|up with two tiles a wave 5.4 / 5.5, one chunk 2.4 / 2.5)
  constexpr bool WHOLE = !HALF && MAXC > 1 && NT == 1;
  constexpr int TR = HALF ? 8 : 16;                    // weight rows of a tile
  constexpr int XB = RP * 4 * SMALL_XROW, WB = HALF ? NT * MAXC * 512 : WHOLE ? MAXC * 1024 : 0, TB = NT * 16 * SMALL_RED * 4;
  constexpr int XW = XB > WB ? XB : WB, SLICE = XW > TB ? XW : TB;
  __shared__ __attribute__((aligned(16))) unsigned char slices[NW][SLICE];
  __shared__ float2_t ssq[NORM ? NW : 1][16];          // of a wave and row: the sum of its squares, the power of two taken out
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int r = lane & 15, kq = lane >> 4;
  const int K = a.K, KW = K >> 3, G = K >> 6;
  // chunks dealt over the waves as evenly as they go
  const int chunks = K >> 7;
  const int per = chunks / NW, rem = chunks % NW;
  const int nch = per + (wave < rem ? 1 : 0);
  // every build serves only K of which each wave owns all its chunks but perhaps the last (small_launch)
  auto owned = [&](int c) { return MAXC > 1 && c < MAXC - 1 ? true : c < nch; };
  const int k0 = (wave * per + (wave < rem ? wave : rem)) * 128;
  int row0, second;                       // first row of tile 0, distance of tile 1
  if (MODE == SMALL_ROPE) {
    const int per_head = a.hd / (2 * TR);
    row0 = (blockIdx.x / per_head) * a.hd + (blockIdx.x % per_head) * TR;
    second = a.hd >> 1;
  } else {
    row0 = blockIdx.x * (TR * NT);
    second = TR;
  }

  // ---- every request of the wave at once ----
  // All loads are unconditional (a load under a condition has to be waited for where the branches
  // join, which puts the requests of a wave one behind the other): chunks the wave does not own
  // and rows past T read a valid address again and their values are never used.
  const int kb = nch > 0 ? k0 : 0;
  const int xcol = 4 * (kq & 1) + 2 * (kq >> 1);      // this lane's first 8 columns of a group, in eights
  // x: lane l reads 16 bytes of row 4 p + l / 16 at byte 16 (l % 16) of the chunk's 256
  uint4_t xg[MAXC][RP];
  {
    const int xr = lane >> 4, xc = lane & 15;
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      const int row = 4 * p + xr < a.T ? 4 * p + xr : a.T - 1;
      const uint32_t at = (uint32_t)row * (K * 2) + xc * 16;
#pragma unroll
      for (int c = 0; c < MAXC; ++c) xg[c][p] = small_load<uint4_t>(a.x + kb + (owned(c) ? c : 0) * 128, at);
    }
  }
  half8_t nw[MAXC];
  if (NORM) {
#pragma unroll
    for (int c = 0; c < MAXC; ++c) nw[c] = small_load<half8_t>(a.norm_w + kb + (owned(c) ? c : 0) * 128, (lane & 15) * 16);
  }
  __builtin_amdgcn_sched_barrier(0);
  uint4_t wv[NT][MAXC];
  uint2_t wh[NT][MAXC];
  uint32_t spair[NT], bpair[NT];          // lane (r, c): the two scales (biases) of row r in chunk c
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    // (rows past the end read the last one: N is a multiple of 8, their values are never stored)
    // (HALF: lane (row l / 8, j = l % 8) holds columns 16 j .. + 16 of a chunk, whole 64-byte pieces; N is a multiple of 8)
    const int first = row0 + second * t, last = !HALF && MODE == SMALL_PLAIN ? a.N - 1 - first : 15;
    const int lr = HALF ? r & 7 : r < last ? r : last, wr = WHOLE ? (lane >> 2 < last ? lane >> 2 : last) : lr;
    const uint32_t* wp = a.w + (long)first * KW + (kb >> 3);
    const uint32_t wat = HALF ? (uint32_t)(lane >> 3) * (KW * 4) + (lane & 7) * 8 : (uint32_t)wr * (KW * 4) + (WHOLE ? lane & 3 : kq) * 16;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
      if (HALF)
        wh[t][c] = small_load<uint2_t>(wp + (owned(c) ? c : 0) * 16, wat);
      else
        wv[t][c] = small_load<uint4_t>(wp + (owned(c) ? c : 0) * 16, wat);
    }
    const uint32_t sat = (uint32_t)lr * (G * 2) + (MAXC > 1 && kq < nch ? kq : 0) * 4;
    spair[t] = small_load<uint32_t>(a.s + (long)first * G + (kb >> 6), sat);
    bpair[t] = small_load<uint32_t>(a.b + (long)first * G + (kb >> 6), sat);
  }
  // What the epilogue adds (bias, residual, the rotation's cos / sin, the cache length) is requested here with everything
  // else, not after the product: a load behind the product is a microsecond of latency on the critical path of a
  // kernel that takes four.  Thread (m, n) of the first TR T holds x row m of weight row n of the tile (and of the other).
  const int em = threadIdx.x / TR, en = threadIdx.x % TR;
  const bool epi = em < a.T && (HALF || MODE != SMALL_PLAIN || row0 + en < a.N);
  half_t e_bias0 = (half_t)0.f, e_bias1 = (half_t)0.f, e_res = (half_t)0.f;
  float2_t e_cs = {1.f, 0.f};
  long e_len = 0;
  const int e_head = MODE == SMALL_ROPE ? row0 / a.hd : 0;
  const int e_d = MODE == SMALL_ROPE ? row0 - e_head * a.hd : 0;
  if (epi) {
    if (a.bias) {
      e_bias0 = a.bias[row0 + en];
      if (NT == 2) e_bias1 = a.bias[row0 + second + en];
    }
    if (MODE == SMALL_PLAIN && a.residual) e_res = a.residual[(long)em * a.N + row0 + en];
    if (MODE == SMALL_ROPE && e_head < a.H + a.G)
      e_cs = *reinterpret_cast<const float2_t*>(a.rope_cs + ((long)em * (a.hd >> 1) + e_d + en) * 2);
  }
  if (MODE == SMALL_ROPE) e_len = *a.len_dev;
  __builtin_amdgcn_sched_barrier(0);
  // ---- RMSNorm folded into x, as it was loaded: lane l holds columns 8 (l % 16) .. + 8 of rows 4 p + l / 16.  The product takes
  // x w of each wave's own columns, either factor times a power of two, and is rounded once as w x / rms would be.  The powers and the row's 1 / rms
  // go onto the sums at the end: no wave waits for another's squares before its matrix instructions.  The powers bring the roots of both sums of
  // squares, which bound the factors, to 2^10 .. 2^11 (x) and 2^3.5 .. 2^4.5 (w): no product leaves fp16's range, and what is small beside the
  // largest keeps its bits (the factors themselves are exact down to 2^-24 and 2^-17 of those roots).  With x alone brought near one by its mean
  // square a large column cost the small ones beside it bits: 8 rows of 2048, one 30000 beside 0.05, error 1.3 times that of w x / rms. ----
  if (NORM) {
    auto squares = [&](half8_t v, float sum) {       // exact products, fp32 sum
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const half2_t p2 = half2_t{v[e], v[e + 1]};
        sum = __builtin_amdgcn_fdot2(p2, p2, sum, false);
      }
      return sum;
    };
    // the exponent that brings a root of `sum` below 2^(top / 2), inside fp16's powers, and 2^-k
    auto exponent = [](float sum, int top) {
      const int k = (__builtin_amdgcn_frexp_expf(sum) - top + 1) >> 1;
      return k < -14 ? -14 : k > 14 ? 14 : k;
    };
    auto power8 = [](int k) {
      const half_t d = __builtin_bit_cast(half_t, (unsigned short)((15 - k) << 10));
      return half8_t{d, d, d, d, d, d, d, d};
    };
    float sw = 0.f;
#pragma unroll
    for (int c = 0; c < MAXC; ++c)
      if (owned(c)) sw = squares(nw[c], sw);
    const int kw = exponent(wave_f32(wave_reduce_row(wave_u32(sw), WaveAdd())), 9);
#pragma unroll
    for (int c = 0; c < MAXC; ++c) nw[c] = nw[c] * power8(kw);
#pragma unroll
    for (int p = 0; p < RP; ++p) {
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < MAXC; ++c)
        if (owned(c)) ss = squares(__builtin_bit_cast(half8_t, xg[c][p]), ss);
      ss = wave_f32(wave_reduce_row(wave_u32(ss), WaveAdd()));
      const int k = exponent(ss, 22);
      if ((lane & 15) == 0) ssq[wave][4 * p + (lane >> 4)] = float2_t{ss, wave_f32((uint32_t)(127 + k + kw) << 23)};
      const half8_t d8 = power8(k);
#pragma unroll
      for (int c = 0; c < MAXC; ++c)
        if (owned(c)) xg[c][p] = __builtin_bit_cast(uint4_t, __builtin_bit_cast(half8_t, xg[c][p]) * d8 * nw[c]);
    }
  }
  // x through the wave's LDS buffer into the operand layout, a chunk at a time (rows past 4 RP,
  // which are rows past T, read what is there: their columns of the result are not stored)
  constexpr int XI = HALF ? 2 : 4;
  half8_t xb[MAXC][XI];
  {
    unsigned char* xs = slices[wave];
    const int xr = lane >> 4, xc = lane & 15;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) {
#pragma unroll
      for (int p = 0; p < RP; ++p)
        *reinterpret_cast<half8_t*>(xs + (4 * p + xr) * SMALL_XROW + xc * 16) = eagle_permute8(__builtin_bit_cast(half8_t, xg[c][p]));
      __builtin_amdgcn_wave_barrier();
      const int m = HALF ? r & 7 : r, mr = m < 4 * RP ? m : 0;
#pragma unroll
      for (int i = 0; i < XI; ++i)
        xb[c][i] = *reinterpret_cast<const half8_t*>(xs + mr * SMALL_XROW + (8 * (HALF ? r >> 3 : i >> 1) + xcol + (i & 1)) * 16);
      __builtin_amdgcn_wave_barrier();
    }
  }

  // ---- the wave's part of the tile(s) ----
  // quarter q of row wr at 16 q + (wr + 4 q) % 16, in units of 16 bytes: neither the stores nor the loads meet in a bank
  uint4_t* ws = reinterpret_cast<uint4_t*>(slices[wave]);
  if (WHOLE) {
    __builtin_amdgcn_wave_barrier();
    const int wr = lane >> 2, q = lane & 3;
#pragma unroll
    for (int c = 0; c < MAXC; ++c) ws[c * 64 + 16 * q + ((wr + 4 * q) & 15)] = wv[0][c];
    __builtin_amdgcn_wave_barrier();
  }
  uint2_t* wp2 = reinterpret_cast<uint2_t*>(slices[wave]);
  if (HALF) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int c = 0; c < MAXC; ++c) wp2[(t * MAXC + c) * 64 + lane] = wh[t][c];
    __builtin_amdgcn_wave_barrier();
  }
  const half_t one = (half_t)1.f;
  const half8_t ones = {one, one, one, one, one, one, one, one};
  const float4_t zero = {0.f, 0.f, 0.f, 0.f};
  // a sum for the even and one for the odd quantisation groups, which is also what the two halves of a small tile hold
  constexpr int GI = HALF ? 1 : 2;
  float4_t acc[NT][GI];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int g = 0; g < GI; ++g) acc[t][g] = zero;
#pragma unroll
  for (int c = 0; c < MAXC; ++c) {
    if (owned(c)) {
      float4_t sx[GI];
#pragma unroll
      for (int g = 0; g < GI; ++g) {
        sx[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[c][2 * g], ones, zero, 0, 0, 0);
        sx[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[c][2 * g + 1], ones, sx[g], 0, 0, 0);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        // the pair of chunk c sits in lane (r, c)
        const uint32_t s2 = MAXC > 1 ? __shfl(spair[t], r + 16 * c, 64) : spair[t], b2 = MAXC > 1 ? __shfl(bpair[t], r + 16 * c, 64) : bpair[t];
        uint32_t w02[2], w13[2];
        if (HALF) {
          const uint2_t v = wp2[(t * MAXC + c) * 64 + 8 * (r & 7) + 4 * (r >> 3) + (xcol >> 1)];
          w02[0] = v[0];
          w13[0] = v[1];
        } else if (WHOLE) {
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            const int q = 2 * g + (kq & 1);
            const uint2_t* p = reinterpret_cast<const uint2_t*>(ws + c * 64 + 16 * q + ((r + 4 * q) & 15));
            const uint2_t v = p[kq >> 1];
            w02[g] = v[0];
            w13[g] = v[1];
          }
        } else {
          const auto s02 = __builtin_amdgcn_permlane32_swap(wv[t][c][0], wv[t][c][2], false, false);
          const auto s13 = __builtin_amdgcn_permlane32_swap(wv[t][c][1], wv[t][c][3], false, false);
#pragma unroll
          for (int g = 0; g < 2; ++g) {
            w02[g] = s02[g];
            w13[g] = s13[g];
          }
        }
#pragma unroll
        for (int g = 0; g < GI; ++g) {
          const bool odd = HALF ? r >= 8 : g == 1;
          const float sc = (float)__builtin_bit_cast(half_t, (unsigned short)(odd ? s2 >> 16 : s2 & 0xffffu));
          const float bi = (float)__builtin_bit_cast(half_t, (unsigned short)(odd ? b2 >> 16 : b2 & 0xffffu));
          float4_t d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[c][2 * g], eagle_expand8(w02[g]), zero, 0, 0, 0);
          d = __builtin_amdgcn_mfma_f32_16x16x32_f16(xb[c][2 * g + 1], eagle_expand8(w13[g]), d, 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 4; ++i) acc[t][g][i] = __builtin_fmaf(bi, sx[g][i], __builtin_fmaf(sc, d[i], acc[t][g][i]));
        }
      }
    }
  }
  __builtin_amdgcn_wave_barrier();
  // The waves' tiles meet in LDS, x row m of weight row n at 20 m + n (the four rows of a store in different banks), and
  // every thread of the first TR T finishes one output: one wave that finished all of them was a tail of 200 instructions.
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    float* red = reinterpret_cast<float*>(slices[wave]) + t * (16 * SMALL_RED);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (!HALF)
        red[SMALL_RED * (4 * kq + i) + r] = acc[t][0][i] + acc[t][GI - 1][i];
      else if (r >> 3 == kq >> 1)                       // x of one group with weights of the same
        red[SMALL_RED * (4 * kq + i) + (r & 7)] = acc[t][0][i];
    }
  }
  __syncthreads();
  if (!epi) return;
  float sum[NT];
  float2_t wave_ss[NW];
  if (NORM) {
#pragma unroll
    for (int w = 0; w < NW; ++w) wave_ss[w] = ssq[w][em];
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    sum[t] = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float* red = reinterpret_cast<const float*>(slices[w]) + t * (16 * SMALL_RED);
      const float v = HALF ? red[SMALL_RED * em + en] + red[SMALL_RED * (8 + em) + en] : red[SMALL_RED * em + en];
      sum[t] = NORM ? __builtin_fmaf(v, wave_ss[w][1], sum[t]) : sum[t] + v;
    }
  }
  if (NORM) {
    float tot = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) tot += wave_ss[w][0];
    // (the hardware's reciprocal square root, 1 ulp, as a square root and a division round it too: a fifth of their chain)
    const float rinv = __builtin_amdgcn_rsqf(__builtin_fmaf(tot, a.inv_k, a.eps));
#pragma unroll
    for (int t = 0; t < NT; ++t) sum[t] *= rinv;
  }
  half_t lo = (half_t)sum[0], hi = (half_t)sum[NT - 1];
  if (a.bias) {
    lo = lo + e_bias0;
    hi = hi + e_bias1;
  }
  if (MODE == SMALL_ROPE) {
    // the linear output rounded to fp16 (bias added in fp16), rotated with the table's (cos, sin)
    // exactly as the separate rope launch does; v rows pass through
    const long P = e_len;
    if (P + em >= a.cap) return;                        // the host checks capacity; never write past the buffer
    half_t* dst;
    if (e_head < a.H) {
      dst = a.q_out + ((long)e_head * a.T + em) * a.hd;
    } else {
      const int g = e_head < a.H + a.G ? e_head - a.H : e_head - a.H - a.G;
      dst = (e_head < a.H + a.G ? a.k_cache : a.v_cache) + ((long)g * a.cap + P + em) * a.hd;
    }
    if (e_head < a.H + a.G) {
      const half2_t o = eagle_rotate((float)lo, (float)hi, e_cs[0], e_cs[1]);
      lo = o[0];
      hi = o[1];
    }
    dst[e_d + en] = lo;
    dst[(a.hd >> 1) + e_d + en] = hi;
  } else if (MODE == SMALL_SWIGLU) {
    const float gf = (float)lo;
    const half_t act = (half_t)(gf / (1.0f + expf(-gf)));
    a.out[(long)em * (a.N >> 1) + (row0 >> 1) + en] = (half_t)((float)act * (float)hi);
  } else {
    if (a.residual) lo = (half_t)((float)lo + (float)e_res);
    a.out[(long)em * a.N + row0 + en] = lo;
  }
}

constexpr int SMALL_K16 = 16 * SMALL_MAXC * 128;      // sixteen waves, three chunks each

template <int NW, int MAXC, int MODE, bool NORM>
void small_go(const SmallArgs& a, int grid, hipStream_t st) {
  // Tiles of eight weight rows where that leaves every compute unit at most one workgroup and a wave has more to multiply than
  // one tile's chunk (8 rows, us, tiles of 16 / 8: 4864 -> 896 4.55 / 4.13, 2048 -> 1024 3.00 / 2.86, 6144 -> 2048 5.00 / 4.65, q|k|v of 896
  // 3.34 / 3.27, of 2048 4.98 / 4.45; one chunk 896 -> 896 2.31 / 2.40; past the line 2048 -> 2560 3.46 / 3.85, 4864 -> 2560 4.56 / 6.15)
  if constexpr (MODE == SMALL_ROPE || (MODE == SMALL_PLAIN && MAXC > 1)) {
    const int halves = MODE == SMALL_PLAIN ? a.N / 8 : 2 * grid;
    if (a.T <= 8 && halves <= 256) {
      if (MODE == SMALL_PLAIN && a.T <= 4)
        hipLaunchKernelGGL((qmm_small_kernel<NW, MAXC, 1, MODE, NORM, true>), dim3(halves), dim3(NW * 64), 0, st, a);
      else
        hipLaunchKernelGGL((qmm_small_kernel<NW, MAXC, 2, MODE, NORM, true>), dim3(halves), dim3(NW * 64), 0, st, a);
      return;
    }
  }
  // (up to four rows in one pass: 1 x 3584 -> 3584 4.5 -> 4.3 us when it came)
  if (MODE == SMALL_PLAIN && a.T <= 4)
    hipLaunchKernelGGL((qmm_small_kernel<NW, MAXC, 1, MODE, NORM, false>), dim3(grid), dim3(NW * 64), 0, st, a);
  else if (a.T > 8)
    hipLaunchKernelGGL((qmm_small_kernel<NW, MAXC, 4, MODE, NORM, false>), dim3(grid), dim3(NW * 64), 0, st, a);
  else
    hipLaunchKernelGGL((qmm_small_kernel<NW, MAXC, 2, MODE, NORM, false>), dim3(grid), dim3(NW * 64), 0, st, a);
}

template <int NW, int MAXC, int MODE>
void small_norm(const SmallArgs& a, int grid, hipStream_t st) {
  if (a.norm_w)
    small_go<NW, MAXC, MODE, true>(a, grid, st);
  else
    small_go<NW, MAXC, MODE, false>(a, grid, st);
}

template <int MODE>
void small_launch(const SmallArgs& a, int grid, hipStream_t st) {
  // A load that a wave makes for a chunk it does not own costs what any other does, so the waves are chosen
  // to own whole loads (8 rows, us): 7 x 1 against 4 x 2 for the 7 chunks of K = 896 (o 2.68 / 2.85, 8192 rows
  // 3.28 / 3.51; the other way round for the many workgroups of gate|up, 9728 rows: 6.2 / 5.8), 4 x 2 against
  // 4 x 3 (gate|up 5.8 / 6.3), 16 x 2 against 16 x 3 for K = 3584 (4.9 / 5.7), 13 x 3 against 16 x 3 for
  // K = 4864 (5.08 / 5.18).  By N and K alone: a SwiGLU product gives the bits of the plain one.
  // Products with a norm and without one (o, down, the plain operator) have builds of their own: the norm weights of a wave's chunks take registers.
  // (One build for both left 2 x 2048 -> 28712 three workgroups to a compute unit for four, 10.4 us for 9.2, and cost 896 -> 896 2.5 %.)
  const int chunks = a.K >> 7;
  if (chunks <= 4) return small_norm<4, 1, MODE>(a, grid, st);
  if (chunks <= 7 && a.N <= 8192) return small_norm<7, 1, MODE>(a, grid, st);
  if (chunks <= 8) return small_norm<4, 2, MODE>(a, grid, st);
  if (chunks <= 12) return small_norm<4, 3, MODE>(a, grid, st);
  if (chunks <= 16) return small_norm<8, 2, MODE>(a, grid, st);
  if (chunks <= 24) return small_norm<8, 3, MODE>(a, grid, st);
  if (chunks <= 32) return small_norm<16, 2, MODE>(a, grid, st);
  if (chunks <= 39) return small_norm<13, 3, MODE>(a, grid, st);
  return small_norm<16, 3, MODE>(a, grid, st);
}

// two scales or biases of a row are one load, four values of the bias another
bool small_vectors_aligned(const void* scales, const void* biases, const void* bias) {
  return ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) == 0 &&
         (reinterpret_cast<uintptr_t>(bias) & 7u) == 0;
}

}  // namespace

EAGLE_EXPORT int eagle_qmm_small_supported(int T, int N, int K, int norm, int swiglu) {
  (void)norm;
  return T >= 1 && T <= 16 && N >= (swiglu ? 32 : 8) && (N % (swiglu ? 32 : 8)) == 0 && K >= 128 && (K % 128) == 0 &&
         K <= SMALL_K16;
}

// Where this kernel beats the vector kernel, the streaming kernel and the rows kernel for a plain (or SwiGLU) product:
// measured over K 512 .. 6144, N 512 .. 37888, 1 .. 16 rows, launches back to back over rotating weights.  Its
// workgroups have no loop over N and share nothing, so it holds for so many rounds of 256 workgroups of 16 weight rows, fewer
// the more K and rows of x each has to itself.  Inside and just past the lines, this / the fastest other, us:
//   1 row  (vector kernel)   2048 -> 8192 4.4 / 5.2, 3584 -> 4608 5.1 / 6.1, 3584 -> 18944 11.3 / 11.5; 3584 -> 28672 15.4 / 14.8
//   4 rows                   2048 -> 28672 9.7 / 10.2, 3584 -> 18944 12.1 / 14.7, 6144 -> 8192 10.4 / 11.6; 3072 -> 28672 14.7 / 13.3
//   8 rows                   896 -> 37888 7.2 / 9.1, 2048 -> 18944 8.6 / 9.3, 3584 -> 12288 9.7 / 10.6; 2560 -> 18944 11.6 / 10.7
//   16 rows                  896 -> 28672 6.6 / 6.8, 3584 -> 8192 7.9 / 9.3; 4096 -> 8192 10.0 / 9.3, 3584 -> 12288 13.0 / 10.9
EAGLE_EXPORT int eagle_qmm_small_preferred(int M, int N, int K) {
  if (!eagle_qmm_small_supported(M, N, K, 0, 0)) return 0;
  int rounds;
  if (M <= 4) rounds = K <= 2048 ? 10 : K <= 3584 ? 5 : K <= 4992 ? 3 : 2;      // (x in one pass of rows)
  else if (M <= 8) rounds = K <= 1536 ? 10 : K <= 2048 ? 5 : K <= 3584 ? 3 : 2;
  else rounds = K <= 1024 ? 7 : K <= 1536 ? 5 : K <= 3584 ? 2 : 1;
  return (N + 15) / 16 <= rounds * 256;
}

EAGLE_EXPORT int eagle_qmm_small_w4g64_f16(const void* x, const void* norm_w, float eps, const uint32_t* wq,
                                           const void* scales, const void* biases, const void* bias,
                                           const void* residual, void* out, int T, int N, int K,
                                           int group_size, int bits, int swiglu, eagle_stream_t stream) {
  if (!x || !wq || !scales || !biases || !out) return EAGLE_ERR_NULL;
  if (group_size != 64 || bits != 4) return EAGLE_ERR_UNSUPPORTED;
  if (!eagle_qmm_small_supported(T, N, K, norm_w != nullptr, swiglu)) return EAGLE_ERR_SHAPE;
  if (swiglu && residual) return EAGLE_ERR_UNSUPPORTED;
  const void* aligned[] = {x, norm_w, wq, residual, out};
  for (const void* p : aligned)
    if (p && !eagle_aligned16(p)) return EAGLE_ERR_ALIGN;
  if (!small_vectors_aligned(scales, biases, bias)) return EAGLE_ERR_ALIGN;
  if (x == out) return EAGLE_ERR_UNSUPPORTED;          // other workgroups still read x
  SmallArgs a;
  a.x = static_cast<const half_t*>(x);
  a.norm_w = static_cast<const half_t*>(norm_w);
  a.w = wq;
  a.s = static_cast<const half_t*>(scales);
  a.b = static_cast<const half_t*>(biases);
  a.bias = static_cast<const half_t*>(bias);
  a.residual = static_cast<const half_t*>(residual);
  a.out = static_cast<half_t*>(out);
  a.eps = eps;
  a.inv_k = 1.0f / (float)K;
  a.T = T;
  a.N = N;
  a.K = K;
  a.rope_cs = nullptr;
  a.q_out = a.k_cache = a.v_cache = nullptr;
  a.len_dev = nullptr;
  a.H = a.G = a.hd = 0;
  a.cap = 0;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (swiglu)
    small_launch<SMALL_SWIGLU>(a, N / 32, st);
  else
    small_launch<SMALL_PLAIN>(a, (N + 15) / 16, st);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_qkv_rope_small_supported(int T, int D, int H, int G, int hd) {
  return T >= 1 && T <= 16 && H >= 1 && G >= 1 && (H % G) == 0 && hd >= 32 && (hd % 32) == 0 &&
         D >= 128 && (D % 128) == 0 && D <= SMALL_K16;
}

EAGLE_EXPORT int eagle_qkv_rope_small_w4g64_f16(const void* x, const void* norm_w, float eps,
                                                const uint32_t* wq, const void* scales, const void* biases,
                                                const void* bias, const float* rope_cs, void* q_out,
                                                void* k_cache, void* v_cache, const int32_t* cache_len_dev,
                                                int T, int D, int H, int G, int hd, long capacity,
                                                int group_size, int bits, eagle_stream_t stream) {
  if (!x || !wq || !scales || !biases || !rope_cs || !q_out || !k_cache || !v_cache || !cache_len_dev)
    return EAGLE_ERR_NULL;
  if (group_size != 64 || bits != 4) return EAGLE_ERR_UNSUPPORTED;
  if (!eagle_qkv_rope_small_supported(T, D, H, G, hd) || capacity < T) return EAGLE_ERR_SHAPE;
  const void* aligned[] = {x, norm_w, wq, rope_cs, q_out, k_cache, v_cache};
  for (const void* p : aligned)
    if (p && !eagle_aligned16(p)) return EAGLE_ERR_ALIGN;
  if (!small_vectors_aligned(scales, biases, bias)) return EAGLE_ERR_ALIGN;
  SmallArgs a;
  a.x = static_cast<const half_t*>(x);
  a.norm_w = static_cast<const half_t*>(norm_w);
  a.w = wq;
  a.s = static_cast<const half_t*>(scales);
  a.b = static_cast<const half_t*>(biases);
  a.bias = static_cast<const half_t*>(bias);
  a.residual = nullptr;
  a.out = nullptr;
  a.eps = eps;
  a.inv_k = 1.0f / (float)D;
  a.T = T;
  a.N = (H + 2 * G) * hd;
  a.K = D;
  a.rope_cs = rope_cs;
  a.q_out = static_cast<half_t*>(q_out);
  a.k_cache = static_cast<half_t*>(k_cache);
  a.v_cache = static_cast<half_t*>(v_cache);
  a.len_dev = cache_len_dev;
  a.H = H;
  a.G = G;
  a.hd = hd;
  a.cap = capacity;
  hipStream_t st = static_cast<hipStream_t>(stream);
  small_launch<SMALL_ROPE>(a, (H + 2 * G) * (hd / 32), st);
  return eagle_launch_status();
}
