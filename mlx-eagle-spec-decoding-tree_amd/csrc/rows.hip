// 4-bit group-64 quantised product for 2..2048 rows of x on the weights in the MLX layout, no weight rounded:
// out[m][n] = fp16( sum_k x[m][k] (s[n,k/64] q[n,k] + b[n,k/64]) ) (+ bias[n]), or silu(g) * u of gate and up
// rows interleaved in 16-row tiles.  (Reference: mx.quantized_matmul, mlx_model_fwd_bench.py:65-73; the
// factorisation of kernels/qmv/1b.metal:121-147.)
//
//   * A workgroup of eight waves owns 8 / KP groups of RT 16-row weight tiles over a range of K; KP waves share a
//     group, each with a part of the range.  Wide matrices take many tiles per workgroup (x is read by fewer), narrow
//     ones few tiles and K split over workgroups, whose fp32 partial sums a second launch adds (rows_plan).
//   * Weights go from memory to registers, 16 bytes per lane, a ring of AH chunks of 128 columns ahead; both 64-byte
//     halves of a line are requested together.  Two half-wave swaps deal the words of a lane so that a matrix
//     instruction works in one quantisation group; nibbles become fp16 integers through the fp8 conversion (exact).
//     The group's sum enters the accumulators times its scale in fp32: no weight is rounded.
//   * x (MT tiles of 16 rows) goes through LDS in blocks, two in turn, one barrier per block that leaves the loads
//     in flight.  While it is stored, the sums of x per group are formed; biases times sums are a few matrix
//     instructions at the end, the sums as fp16 hi + lo.
//   * The scales (biases) of a workgroup's rows are read once, whole lines, and kept in LDS.  Read per block of K
//     instead, 16 bytes of a row at a time, every line came from memory as often as it has blocks: 32 x 3584 x 152064
//     90 us, 71 us so; without reading any 67.
//
//   * More than 64 rows (a prompt of the module path) are blocks of 48 or 64 rows of the same kernel, the blocks of one
//     group of weight rows next to each other in the grid, so that an XCD's L2 gives the weights to several of them.
//
// What bounds it: the bytes a compute unit takes in, its weights and all of its x (the loads and the x path alone
// 58 .. 65 us there), then the vector instructions of the expansion.  Against the streaming kernel (us, launches
// back to back over rotating weights): 32 x 3584 x 152064 69.5 / 80, 27 x 18944 x 3584 17.5 / 23, 32 x 2048 x 8192 7.5 / 11.0,
// 64 x 8192 x 8192 23 / 40.  With many rows the vector instructions (expansion per block, a multiply-add per group and
// output) about equal the matrix instructions: 2048 x 37888 x 3584 675 us = 0.82 PFLOP/s, 512 x 3584 x 18944 114 us; the
// GEMM, which rounds the weights to fp16 and expands them once per 256 rows, takes 580 and 93 (128 x 3584 x 37888 58 us
// with the sums of a tile added behind its matrix instructions, 54 under the next tile's).  In a prompt pass, weights
// not in a cache: 732 and (2048 x 3584 x 18944) 372 us against 553 and 263; matrix pipes 37 % busy at 2.05 GHz.
#include "common.h"

#include <type_traits>

namespace {

struct RowsArgs {
  const half_t* x;        // [M, K]
  const uint32_t* w;      // [N, K / 8]
  const half_t* s;        // [N, K / 64]
  const half_t* b;
  const half_t* bias;     // [N] or nullptr
  half_t* out;            // [M, N], [M, N / 2] with SwiGLU
  float* partial;         // [gridDim.y, pitch, N] or nullptr
  int M, N, K, swiglu;
  int both;               // scales and biases fit LDS together
  int pitch;              // rows of x per split in `partial`
  int zb;                 // blocks of 16 MT rows of x
};

constexpr int ROWS_WAVES = 8;
constexpr int ROWS_LDS = 160 * 1024;
constexpr int ROWS_RSRC = 0x00020000;      // buffer descriptor: untyped bytes
constexpr int ROWS_XROW = 256 + 16;        // bytes of a staged x row: a chunk of 128 columns, padded against bank conflicts

// a barrier that leaves the loads from memory in flight
__device__ inline void rows_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// keeps the loads from memory where they are written: everything else may move across
__device__ inline void rows_pin() { __builtin_amdgcn_sched_barrier(0x38f); }

// sum over eight neighbouring lanes
__device__ inline float rows_sum8(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xb1, 0xf, 0xf, false));   // lane ^ 1
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4e, 0xf, 0xf, false));   // lane ^ 2
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xf, 0xf, false));  // 7 - lane
  return v;
}

// bytes of a row's scales in LDS for `units` units of four chunks: an odd multiple of 16, so that sixteen rows
// sit in different banks
__host__ __device__ constexpr int rows_stride(int units) { return (units | 1) * 16; }

constexpr int rows_block(int MT, int KP) { return (MT > 2 ? 2 : 4) / KP > 0 ? (MT > 2 ? 2 : 4) / KP : 1; }

// bytes of LDS: two blocks of x, its sums, scales (and biases); at the end the sums of the K parts
size_t rows_lds_bytes(int RT, int MT, int KP, int nu, bool both) {
  const size_t rows = 16 * MT, B = rows_block(MT, KP), wrows = ROWS_WAVES / KP * RT * 16;
  const size_t stage = 2 * KP * B * rows * ROWS_XROW + KP * 4 * nu * rows * 8 +
                       (both ? 2 : 1) * (size_t)ROWS_WAVES * RT * 16 * rows_stride(nu);
  const size_t epi = KP * rows * (wrows + 4) * 4;
  return stage > epi ? stage : epi;
}

// MANY: more than one block of x rows
template <int RT, int MT, int KP, int AH, bool MANY>
__global__ __launch_bounds__(ROWS_WAVES * 64) void qmm_rows_kernel(RowsArgs a) {
  constexpr int B = rows_block(MT, KP);            // chunks per K part and block of staged x
  constexpr int ROWS = 16 * MT;                    // rows of x
  constexpr int SLOT = ROWS * ROWS_XROW;           // bytes of a staged chunk
  constexpr int BUF = KP * B * SLOT;
  constexpr int NP = KP * B * ROWS * 16 / (ROWS_WAVES * 64);   // 16-byte pieces of x per thread and block
  constexpr int RG = ROWS_WAVES / KP;              // groups of RT tiles side by side
  constexpr int WROWS = RG * RT * 16;              // weight rows per workgroup
  static_assert(NP * ROWS_WAVES * 64 == KP * B * ROWS * 16, "x does not divide over the threads");
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int r = lane & 15, kq = lane >> 4;
  const int kp = wave % KP, rg = wave / KP;
  const int nb = MANY ? blockIdx.x / a.zb : blockIdx.x;                  // weight rows, then block of x
  const int m0 = MANY ? (blockIdx.x - nb * a.zb) * ROWS : 0;
  const int K = a.K, M = MANY && a.M - m0 > ROWS ? ROWS : a.M - m0, N = a.N;
  const int all = K >> 7;
  // K in units of four chunks (512 columns), dealt over the workgroups along y and then over the K parts
  const int units = (all + 3) >> 2;
  const int ulo = (int)((long)units * blockIdx.y / gridDim.y), uhi = (int)((long)units * (blockIdx.y + 1) / gridDim.y);
  auto first = [&](int p) {
    const int c = 4 * (ulo + (uhi - ulo) * p / KP);
    return c < all ? c : all;
  };
  const int NU = (uhi - ulo + KP - 1) / KP;        // units of the longest K part
  const int c0 = first(kp), nch = first(kp + 1) - c0;
  const int XC = 4 * NU;
  half2_t* xsum = reinterpret_cast<half2_t*>(rows_lds + 2 * BUF);      // [KP][XC][ROWS][2]: (hi, lo) of a group's sum
  // scales of this wave's rows for its K part [RT * 16][stride], then the biases if a.both
  const int stride = rows_stride(NU);
  unsigned char* const sbl = rows_lds + 2 * BUF + KP * XC * ROWS * 8 + wave * (RT * 16) * stride * (a.both ? 2 : 1);

  // ---- addresses: buffer loads, a uniform offset per tile and chunk beside one 32-bit lane offset ----
  const int row0 = nb * WROWS + rg * (RT * 16);
  const int G = K >> 6;
  const auto wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(a.w), 0, (int)((long)N * K >> 1), ROWS_RSRC);
  const auto sbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(a.s), 0, N * G * 2, ROWS_RSRC);
  const auto bbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(a.b), 0, N * G * 2, ROWS_RSRC);
  const auto xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t*>(a.x) + (long)m0 * K, 0, M * K * 2, ROWS_RSRC);
  const uint32_t wlane = (uint32_t)r * (K >> 1) + kq * 16;
  uint32_t wbase[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int n = row0 + 16 * t < N - 16 ? row0 + 16 * t : N - 16;     // tiles past the end repeat the last
    wbase[t] = (uint32_t)n * (K >> 1) + c0 * 64;
  }

  // ---- x: a wave instruction moves four rows of a chunk ----
  constexpr int QUADS = ROWS / 4;                  // instructions per chunk
  const int xr4 = lane >> 4, xpc = lane & 15;
  uint4_t xr[NP];
  auto request_x = [&](int blk) {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int at = i * ROWS_WAVES + wave, slot = at / QUADS, part = slot / B;
      const int p0 = first(part), n = first(part + 1) - p0;
      int c = blk * B + slot % B;
      c = c < n ? c : n - 1;
      const int row = at % QUADS * 4 + xr4;
      xr[i] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(
                  xbuf, (row < M ? row : M - 1) * (K * 2) + xpc * 16, (p0 + c) * 256, 0));
    }
  };
  auto store_x = [&](int blk) {
    unsigned char* buf = rows_lds + (blk & 1) * BUF;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int at = i * ROWS_WAVES + wave, slot = at / QUADS, row = at % QUADS * 4 + xr4;
      const half8_t v = __builtin_bit_cast(half8_t, xr[i]);
      *reinterpret_cast<half8_t*>(buf + slot * SLOT + row * ROWS_XROW + xpc * 16) = eagle_permute8(v);
      const half2_t one = {(half_t)1.f, (half_t)1.f};
      float sum = 0.f;
#pragma unroll
      for (int e = 0; e < 8; e += 2) sum = __builtin_amdgcn_fdot2(half2_t{v[e], v[e + 1]}, one, sum, false);
      sum = rows_sum8(sum);
      const int c = blk * B + slot % B;
      // (eight lanes write the same value; a branch here would end the basic block, and the compiler sinks
      // the accumulation of a whole period behind it)
      const half_t top = (half_t)sum;
      xsum[((slot / B * XC + c) * ROWS + row) * 2 + (xpc >> 3)] = half2_t{top, (half_t)(sum - (float)top)};
    }
  };

  // ---- weights: a ring of AH chunks ----
  uint4_t ring[AH][RT];
  auto request_w = [&](int u, int t, int c) {
    const int cc = c < nch ? c : nch - 1;
    ring[u][t] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(wbuf, wlane, wbase[t] + cc * 64, 0));
  };
  // Scales and biases: 16 bytes are a row's groups in four chunks.  A wave reads all that its rows and K part
  // need in one go, whole lines of memory once, and keeps them in LDS.  Values past the part become zero.
  constexpr int SBN = RT * MT < 15 ? 10 : 9;       // loads in one go (the registers of the largest form hold nine)
  const int pieces = RT * 16 * NU;
  const uint32_t inv = (65536u + NU - 1) / NU;
  uint4_t sreg[SBN], breg[SBN];
  auto place = [&](int at, int* row, int* unit) {
    const int i = at < pieces ? at : pieces - 1;   // (past the end: the last one again)
    *row = (int)((uint32_t)i * inv >> 16);
    *unit = i - *row * NU;
  };
  auto request_sb = [&](const auto& buf, uint4_t* reg, int from) {
#pragma unroll
    for (int i = 0; i < SBN; ++i) {
      if (from + i * 64 >= pieces) break;
      int row, unit;
      place(from + i * 64 + lane, &row, &unit);
      int n = row0 + (row & ~15);
      n = (n < N - 16 ? n : N - 16) + (row & 15);
      reg[i] = __builtin_bit_cast(uint4_t, __builtin_amdgcn_raw_buffer_load_b128(buf, (n * G + c0 * 2) * 2 + unit * 16, 0, 0));
    }
  };
  auto store_sb = [&](unsigned char* to, const uint4_t* reg, int from) {
#pragma unroll
    for (int i = 0; i < SBN; ++i) {
      if (from + i * 64 >= pieces) break;
      int row, unit;
      place(from + i * 64 + lane, &row, &unit);
      uint4_t v = reg[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = 4 * unit + e < nch ? v[e] : 0u;
      *reinterpret_cast<uint4_t*>(to + row * stride + unit * 16) = v;
    }
  };
  auto fetch_sb = [&](const auto& buf, unsigned char* to, int from) {
    for (; from < pieces; from += SBN * 64) {
      request_sb(buf, sreg, from);
      store_sb(to, sreg, from);
    }
  };

  request_x(0);
  request_sb(sbuf, sreg, 0);
  if (a.both) request_sb(bbuf, breg, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < AH; u += 2)
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      request_w(u, t, u);
      request_w(u + 1, t, u + 1);
    }
  __builtin_amdgcn_sched_barrier(0);
  store_x(0);
  store_sb(sbl, sreg, 0);
  if (a.both) store_sb(sbl + RT * 16 * stride, breg, 0);
  if (pieces > SBN * 64) {
    fetch_sb(sbuf, sbl, SBN * 64);
    if (a.both) fetch_sb(bbuf, sbl + RT * 16 * stride, SBN * 64);
  }
  rows_barrier();

  const float4_t zero = {0.f, 0.f, 0.f, 0.f};
  float4_t acc[RT][MT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[t][mt] = zero;

  const int xcol = 4 * (kq & 1) + 2 * (kq >> 1);
  const int alane = kp * (B * SLOT) + r * ROWS_XROW + xcol * 16;
  // one chunk: `u` its place among four (static), `last` in the last unit (nothing is requested past its end)
  auto chunk = [&](int u, int c, auto last) {
    const unsigned char* xa = rows_lds + (c / B & 1) * BUF + (c % B) * SLOT + alane;
    uint32_t s2[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) s2[t] = *reinterpret_cast<const uint32_t*>(sbl + (t * 16 + r) * stride + c * 4);
    // word pairs of a lane -> word pairs of a group, in place
    auto regroup = [&](uint4_t& v) {
      const auto w02 = __builtin_amdgcn_permlane32_swap(v[0], v[2], false, false);
      const auto w13 = __builtin_amdgcn_permlane32_swap(v[1], v[3], false, false);
      v = uint4_t{w02[0], w13[0], w02[1], w13[1]};
    };
    auto reload = [&](int t) {                     // both halves of a line together
      if ((u & 1) && (!last() || u - 1 + AH < 4)) {
        rows_pin();
        request_w((u - 1) % AH, t, c - 1 + AH);
        request_w(u % AH, t, c + AH);
        rows_pin();
      }
    };
    auto scale = [&](int t, int g) { return (float)__builtin_bit_cast(half_t, (unsigned short)(g ? s2[t] >> 16 : s2[t] & 0xffffu)); };
    auto load_x = [&](half8_t* xv, int mt, int g) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        xv[i] = *reinterpret_cast<const half8_t*>(xa + mt * (16 * ROWS_XROW) + (8 * g + i) * 16);
    };
    // The matrix instructions of a tile run while the sums of the one before enter the accumulators, both groups of a chunk
    // at once where the registers hold that and it is faster (40 x 3584 x 37888 on three tiles and two parts: tile after tile
    // 34.7 us, group by group with the overlap 33.3, both groups 31.7; one tile: 19.1 by both, 18.7 group by group)
    if (MT <= 2 || (MT == 3 && (RT == 3 ? KP <= 2 : RT == 2 && KP > 1))) {
      half8_t xv[MT][2][2];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int g = 0; g < 2; ++g) load_x(xv[mt][g], mt, g);
      float4_t d[2][2][MT];
      auto add = [&](int t) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const float sg = scale(t, g);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][mt][i] = __builtin_fmaf(sg, d[t & 1][g][mt][i], acc[t][mt][i]);
        }
      };
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        uint4_t v = ring[u % AH][t];
        regroup(v);
        reload(t);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const half8_t q0 = eagle_expand8(v[2 * g]), q1 = eagle_expand8(v[2 * g + 1]);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) d[t & 1][g][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[mt][g][0], q0, zero, 0, 0, 0);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            d[t & 1][g][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[mt][g][1], q1, d[t & 1][g][mt], 0, 0, 0);
        }
        if (t > 0) add(t - 1);
        __builtin_amdgcn_sched_barrier(0);
      }
      add(RT - 1);
    } else {
      // group by group (64 x 3584 x 37888 39.8 us without the overlap, 37.3 with it)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        half8_t xv[MT][2];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) load_x(xv[mt], mt, g);
        float4_t d[2][MT];
        auto add = [&](int t) {
          const float sg = scale(t, g);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[t][mt][i] = __builtin_fmaf(sg, d[t & 1][mt][i], acc[t][mt][i]);
        };
#pragma unroll
        for (int t = 0; t < RT; ++t) {
          if (g == 0) regroup(ring[u % AH][t]);
          const half8_t q0 = eagle_expand8(ring[u % AH][t][2 * g]), q1 = eagle_expand8(ring[u % AH][t][2 * g + 1]);
          if (g == 1) reload(t);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) d[t & 1][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[mt][0], q0, zero, 0, 0, 0);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) d[t & 1][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[mt][1], q1, d[t & 1][mt], 0, 0, 0);
          if (t > 0) add(t - 1);
          __builtin_amdgcn_sched_barrier(0);
        }
        add(RT - 1);
      }
    }
  };
  auto step = [&](int u, int c, auto last) {
    const bool more = !last() || u / B * B + B < 4;          // another block of x follows
    if (u % B == 0 && more) request_x(c / B + 1);
    rows_pin();
    chunk(u, c, last);
    if (last())
      __builtin_amdgcn_sched_barrier(0);       // (nothing is requested between these chunks: keep them apart all the same)
    else
      rows_pin();
    if (u % B == B - 1 && more) {
      store_x(c / B + 1);
      rows_barrier();
    }
  };
  // The last unit by itself: what it would request, no chunk uses.  With the block of x and the ring of weights past the end
  // fetched all the same, a workgroup of one unit spent a round trip to memory and a barrier on them (us before / now, timed in turn:
  // 32 x 3584 x 4608 left as seven partial sums 7.07 / 6.53, 40 rows 8.0 / 7.7; 32 x 3584 x 37888 with SwiGLU 27.3 / 26.5, 40 x 3584 x
  // 152064 80.2 / 78.8, 128 x 3584 x 37888 55.0 / 53.9).
  for (int j = 0; j + 1 < NU; ++j) {
#pragma unroll
    for (int u = 0; u < 4; ++u) step(u, 4 * j + u, std::false_type{});
  }
#pragma unroll
  for (int u = 0; u < 4; ++u) step(u, 4 * (NU - 1) + u, std::true_type{});
  // (or the compiler sinks the accumulation of the unit behind it, into the block that uses the sums, and runs out of registers)
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) asm volatile("" : "+v"(acc[t][mt]));

  // ---- the biases times the sums of x: eight chunks per matrix instruction, each sum as hi + lo ----
  const unsigned char* bl = sbl + RT * 16 * stride;
  if (!a.both) {
    fetch_sb(bbuf, sbl, 0);
    bl = sbl;
  }
  for (int j = 0; j < NU; j += 2) {
    const bool more = j + 1 < NU;                  // (past the end: the sums of the last unit, biases of zero)
    const int ca = 4 * j + kq, cb = more ? ca + 4 : ca;
    half8_t xs[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const half4_t v0 = *reinterpret_cast<const half4_t*>(xsum + ((kp * XC + ca) * ROWS + mt * 16 + r) * 2);
      const half4_t v1 = *reinterpret_cast<const half4_t*>(xsum + ((kp * XC + cb) * ROWS + mt * 16 + r) * 2);
      xs[mt] = half8_t{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const half2_t b0 = *reinterpret_cast<const half2_t*>(bl + (t * 16 + r) * stride + ca * 4);
      half2_t b1 = *reinterpret_cast<const half2_t*>(bl + (t * 16 + r) * stride + cb * 4);
      if (!more) b1 = half2_t{(half_t)0.f, (half_t)0.f};
      const half8_t bv = {b0[0], b0[0], b0[1], b0[1], b1[0], b1[0], b1[1], b1[1]};
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[t][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xs[mt], bv, acc[t][mt], 0, 0, 0);
    }
  }

  // ---- through LDS: [KP][ROWS][WROWS], then eight outputs per thread ----
  constexpr int OROW = WROWS + 4;
  float* red = reinterpret_cast<float*>(rows_lds);
  rows_barrier();
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        red[(long)(kp * ROWS + mt * 16 + 4 * kq + i) * OROW + rg * (RT * 16) + t * 16 + r] = acc[t][mt][i];
  rows_barrier();
  const int base = nb * WROWS;
  auto sum8 = [&](int m, int at, float* v) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = 0.f;
#pragma unroll
    for (int k = 0; k < KP; ++k) {
      const float* p = red + (long)(k * ROWS + m) * OROW + at;
      const float4_t p0 = *reinterpret_cast<const float4_t*>(p), p1 = *reinterpret_cast<const float4_t*>(p + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] += p0[e];
        v[4 + e] += p1[e];
      }
    }
  };
  const bool swi = a.swiglu && !a.partial;
  const int per_row = swi ? WROWS / 16 : WROWS / 8;
  for (int idx = tid; idx < M * per_row; idx += ROWS_WAVES * 64) {
    const int m = idx / per_row, o = idx % per_row;
    const int at = swi ? (o >> 1) * 32 + (o & 1) * 8 : o * 8;
    if (base + (at & ~15) >= N) continue;
    const int tile = base + (at & ~15) < N - 16 ? base + (at & ~15) : N - 16;
    const int n = tile + (at & 15);
    float v[8];
    sum8(m, at, v);
    if (a.partial) {
      float* p = a.partial + ((long)blockIdx.y * a.pitch + m0 + m) * N + n;
      *reinterpret_cast<float4_t*>(p) = float4_t{v[0], v[1], v[2], v[3]};
      *reinterpret_cast<float4_t*>(p + 4) = float4_t{v[4], v[5], v[6], v[7]};
      continue;
    }
    half8_t h;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      h[e] = (half_t)v[e];
      if (a.bias) h[e] = h[e] + a.bias[n + e];
    }
    if (swi) {
      float w[8];
      sum8(m, at + 16, w);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        half_t u = (half_t)w[e];
        if (a.bias) u = u + a.bias[n + 16 + e];
        const float gf = (float)h[e];
        const half_t act = (half_t)(gf / (1.0f + expf(-gf)));
        h[e] = (half_t)((float)act * (float)u);
      }
      *reinterpret_cast<half8_t*>(a.out + (long)(m0 + m) * (N >> 1) + ((n >> 5) << 4) + (n & 15)) = h;
    } else {
      *reinterpret_cast<half8_t*>(a.out + (long)(m0 + m) * N + n) = h;
    }
  }
}

template <int RT, int MT, int KP, int AH, bool MANY>
int rows_launch(const RowsArgs& a, int splits, hipStream_t st) {
  constexpr int WROWS = ROWS_WAVES / KP * RT * 16;
  const int units = ((a.K >> 7) + 3) / 4, most = (units + splits - 1) / splits, nu = (most + KP - 1) / KP;
  RowsArgs b = a;
  b.zb = (a.M + 16 * MT - 1) / (16 * MT);
  b.both = rows_lds_bytes(RT, MT, KP, nu, true) <= ROWS_LDS;
  const size_t lds = rows_lds_bytes(RT, MT, KP, nu, b.both);
  if (lds > ROWS_LDS) return EAGLE_ERR_SHAPE;
  static bool ready = false;             // (set twice by two first calls at once: the same value)
  if (!ready) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&qmm_rows_kernel<RT, MT, KP, AH, MANY>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, ROWS_LDS) != hipSuccess)
      return EAGLE_ERR_HIP;
    ready = true;
  }
  hipLaunchKernelGGL((qmm_rows_kernel<RT, MT, KP, AH, MANY>), dim3((a.N + WROWS - 1) / WROWS * b.zb, splits), dim3(ROWS_WAVES * 64), lds, st, b);
  return eagle_launch_status();
}

// The partial sums of a split product added in split order: fp16 (+ bias), or silu(g) * u of interleaved gate|up
// rows.  Eight outputs per thread, every load in flight before the first add.
template <bool SWI>
__global__ __launch_bounds__(256) void rows_sum_kernel(const float* __restrict__ partial, int splits, const half_t* __restrict__ bias,
                                                       half_t* __restrict__ out, int M, int N) {
  const int per_row = (SWI ? N >> 1 : N) >> 3;
  const int idx = blockIdx.x * 256 + threadIdx.x;
  if (idx >= M * per_row) return;
  const int m = idx / per_row, o8 = (idx % per_row) * 8;
  const int n = SWI ? (o8 >> 4) * 32 + (o8 & 15) : o8;
  const size_t stride = (size_t)M * N;
  half8_t r = eagle_slab_sum8(partial, splits, stride, (size_t)m * N + n, nullptr);
  half8_t u;
  if (SWI) u = eagle_slab_sum8(partial, splits, stride, (size_t)m * N + n + 16, nullptr);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (bias) r[e] = r[e] + bias[n + e];
    if (SWI) {
      half_t ue = u[e];
      if (bias) ue = ue + bias[n + 16 + e];
      const float gf = (float)r[e];
      const half_t act = (half_t)(gf / (1.0f + expf(-gf)));
      r[e] = (half_t)((float)act * (float)ue);
    }
  }
  *reinterpret_cast<half8_t*>(out + (size_t)m * (SWI ? N >> 1 : N) + o8) = r;
}

struct RowsForm {
  int rt, mt, kp;
  int (*launch)(const RowsArgs&, int, hipStream_t);
  int (*launch_many)(const RowsArgs&, int, hipStream_t);      // more than 64 rows (blocks of 48 or 64), or nullptr
};
template <int RT, int MT, int KP, int AH>
constexpr RowsForm rows_form() {
  if constexpr (MT >= 3)
    return {RT, MT, KP, rows_launch<RT, MT, KP, AH, false>, rows_launch<RT, MT, KP, AH, true>};
  else
    return {RT, MT, KP, rows_launch<RT, MT, KP, AH, false>, nullptr};
}
const RowsForm rows_forms[] = {
#define ROWS_FORM(RT, MT, KP, AH) rows_form<RT, MT, KP, AH>()
    ROWS_FORM(1, 1, 1, 4), ROWS_FORM(1, 1, 2, 4), ROWS_FORM(1, 1, 4, 4), ROWS_FORM(2, 1, 1, 4), ROWS_FORM(3, 1, 1, 4),
    ROWS_FORM(3, 1, 4, 2), ROWS_FORM(5, 1, 1, 2), ROWS_FORM(5, 1, 4, 2),
    ROWS_FORM(1, 2, 1, 4), ROWS_FORM(1, 2, 2, 4), ROWS_FORM(1, 2, 4, 4), ROWS_FORM(2, 2, 1, 4), ROWS_FORM(2, 2, 2, 4),
    ROWS_FORM(3, 2, 1, 4), ROWS_FORM(3, 2, 4, 2), ROWS_FORM(5, 2, 1, 2), ROWS_FORM(5, 2, 4, 2),
    ROWS_FORM(1, 3, 1, 4), ROWS_FORM(1, 3, 2, 4), ROWS_FORM(2, 3, 1, 4), ROWS_FORM(2, 3, 2, 2), ROWS_FORM(3, 3, 1, 2),
    ROWS_FORM(3, 3, 2, 2), ROWS_FORM(3, 3, 4, 2), ROWS_FORM(5, 3, 1, 2), ROWS_FORM(5, 3, 2, 2),
    ROWS_FORM(1, 4, 1, 4), ROWS_FORM(1, 4, 2, 4), ROWS_FORM(2, 4, 1, 4), ROWS_FORM(2, 4, 2, 2), ROWS_FORM(3, 4, 1, 2),
    ROWS_FORM(3, 4, 2, 2),
#undef ROWS_FORM
};
constexpr int ROWS_FORMS = sizeof(rows_forms) / sizeof(rows_forms[0]);

struct RowsPlan {
  int form, splits;
  bool behind;         // the streaming kernel is expected to be faster
};

// The division of the work with the least predicted time (us), from a model fitted to timings of every form, launches
// back to back over rotating weights.  A compute unit takes
// its workgroups one after the other; each costs its start, its share of the weights and its x at the rates a
// unit ingests them (40 and 72 GB/s), and 0.22 us per unit of four chunks, tile and 16 rows of x.  What the whole
// grid reads counts a little, a split as much as its second launch and the partial sums (the sums alone where
// the consumer of the product adds them).  For 65 .. 2048 rows the same formula over the blocks of x.  Its choice against
// the best of all forms and splits of 1400 and 12600 random products: 17 .. 64 rows 1.2 % longer on
// average, 8 % at the 95th percentile; 65 .. 2048 rows 1.2 and 7.5.  Up to 16 rows (one tile, other constants: a unit costs its
// weights and the barriers of its K parts rather than its matrix instructions, a split more than the few rows say) 1.0 and 7.3,
// where the constants of the others gave 3.2 and 14 (4 x 8192 -> 3584 two tiles a wave in 16 splits 12.0 us, one in 8 9.9).  Splits of up to
// three rows count as those of four (2 x 11008 -> 18944 chose another division: 36.1 us, 33.1).
enum { ROWS_WHOLE = 0, ROWS_SPLIT = 1, ROWS_PARTIAL = 2 };
struct RowsCost {
  double start, w, x, unit, parts, whole, second, sums, rows;
};
constexpr RowsCost rows_cost_one = {2.11, 0.0309, 0.0107, 0.0448, 0.419, 0.0018, 2.60, 1.353, 5.};
constexpr RowsCost rows_cost = {1.03, 0.0246, 0.0138, 0.221, 0., 0.0107, 2.93, 0.49, 0.};

// Up to 16 rows of x, K up to 2048 or 70 .. 250 M weights: whether the streaming kernel is faster than this one by the form (rt tiles, kp
// parts, no splits).  That kernel deals the tiles of 16 weight rows evenly over the compute units, where this one has whole rounds of 128 .. 640
// weight rows a workgroup: at 100000 weight rows half of the second round idles (3 x 1152 -> 102016 22.8 us, 18.9; 10 x 640 -> 99944 17.2, 14.9;
// 4 x 2816 -> 34496 17.9, 16.9), while 28672 or 152064 fill theirs (8 x 512 -> 152064 12.4, 18.3; 8 x 3584 -> 28672 14.3, 17.2).  Both times (us) from
// fits to 1779 such products of 16000 weight rows up, 2.7 and 3 % rms: the streaming kernel's by its waves, one per 256 columns, and the tiles of
// a workgroup, which come in steps of four.  This kernel is more than 3 % behind in 345 of them, with the rule in 76 (8 %: 93, 6), and the rule
// loses more than 3 % in 20.  (The streaming kernel's result is further from the exact one before it is rounded: 0.02 .. 0.5 % more error after.)
bool rows_behind_streaming(int M, int N, int K, int rt, int kp) {
  const double size = (double)N * K;
  if (M > 16 || N <= 16000 || K > 3584 || (K > 2048 && (size <= 7e7 || size >= 2.5e8))) return false;
  const int waves = (K + 255) >> 8, all = (N + 15) >> 4, tiles = (all + 255) / 256, steps = (tiles + 3) / 4;
  static const double start[] = {4.02, 5.08, 5.86}, tile[] = {0.313, 0.454, 0.864}, step[] = {0.094, 0.282, 0.343}, more[] = {0.152, 0.343, 0.444};
  static const int least[] = {2, 5, 9};
  const int b = waves <= 4 ? 0 : waves <= 8 ? 1 : 2;
  const double stream = start[b] + (tile[b] + (K % 256 ? 0.028 : 0.) + 0.0037 * M) * tiles + (step[b] + more[b] * (waves - least[b])) * steps;
  const int units = ((K >> 7) + 3) / 4, nu = (units + kp - 1) / kp, wrows = ROWS_WAVES / kp * rt * 16;
  const int blocks = (N + wrows - 1) / wrows, rounds = (blocks + 255) / 256;
  const double rows = 1.32 + rounds * (1.94 + 0.396 * rt + (0.517 + 0.0065 * M) * nu * rt + 0.197 * nu * kp + (K % 512 ? 0.104 * rt : 0.)) +
                      blocks / 256. * 0.519 * nu * rt + 0.027e-6 * size;
  return stream < 0.98 * rows;
}

RowsPlan rows_find_plan(int M, int N, int K, int mode) {
  const int units = ((K >> 7) + 3) / 4;
  const int least_zb = (M + 63) / 64, mt = (M + 16 * least_zb - 1) / (16 * least_zb), zb = (M + 16 * mt - 1) / (16 * mt);
  const RowsCost& cost = mt == 1 ? rows_cost_one : rows_cost;
  RowsPlan best = {-1, 1, false};
  double least = 1e30;
  for (int f = 0; f < ROWS_FORMS; ++f) {
    const RowsForm& form = rows_forms[f];
    if (form.mt != mt) continue;
    const int wrows = ROWS_WAVES / form.kp * form.rt * 16;
    const long blocks = (long)((N + wrows - 1) / wrows) * zb;
    int last = 0;
    for (int z = 1; z <= (mode == ROWS_WHOLE ? 1 : 32) && units / z >= form.kp; ++z) {
      const int nu = ((units + z - 1) / z + form.kp - 1) / form.kp;
      if (nu == last) continue;                    // more workgroups, none of them shorter
      last = nu;
      if (rows_lds_bytes(form.rt, mt, form.kp, nu, false) > ROWS_LDS) continue;
      const double rounds = (double)((blocks * z + 255) / 256);
      const double w = wrows * (double)nu * form.kp * (512 * 0.5625 / 1e3), x = 16. * mt * nu * form.kp * (1024 / 1e3);
      double t = rounds * (cost.start + cost.w * w + cost.x * x + (cost.unit * form.rt * mt + cost.parts * (form.kp - 1)) * nu) +
                 cost.whole * (blocks * z / 256.) * (w + 0.5 * x);
      if (z > 1) t += (mode == ROWS_SPLIT ? cost.second : 0.) + cost.sums * 4e-6 * z * ((M > 4 ? M : 4) + cost.rows) * N;
      if (t < least) {
        least = t;
        best = {f, z, false};
      }
    }
  }
  if (best.form >= 0 && best.splits == 1) best.behind = rows_behind_streaming(M, N, K, rows_forms[best.form].rt, rows_forms[best.form].kp);
  return best;
}

RowsPlan rows_plan(int M, int N, int K, int mode) {
  struct Known {
    int M = 0, N = 0, K = 0, mode = 0;
    RowsPlan plan;
  };
  static thread_local Known known[64];
  Known& k = known[((unsigned)M * 2654435761u ^ (unsigned)N * 40503u ^ (unsigned)K * 9176u ^ (unsigned)mode << 9) >> 7 & 63];
  if (k.M != M || k.N != N || k.K != K || k.mode != mode) {
    k.plan = rows_find_plan(M, N, K, mode);
    k.M = M;
    k.N = N;
    k.K = K;
    k.mode = mode;
  }
  return k.plan;
}

}  // namespace

EAGLE_EXPORT int eagle_qmm_rows_supported(int M, int N, int K, int swiglu) {
  return M >= 1 && M <= EAGLE_MAX_CHUNK && N >= 16 && (N % (swiglu ? 32 : 8)) == 0 && K >= 128 && (K % 128) == 0 &&
         (long)N * K < (1L << 33) && rows_plan(M, N, K, ROWS_SPLIT).form >= 0;
}

// Where it beats the other forms (us, against the streaming kernel unless noted).  33 rows on: everywhere (two
// passes of the streaming kernel; 48 x 3584 x 18944 23 / 38, 64 x 896 x 512 8.1 / 10.8).  17 .. 32 rows: from about
// 4 MB of weights or K above 4608 (2048 -> 3584 7.4 / 9.1, 896 -> 8192 6.3 / 6.8, 8192 -> 512 9.9 / 12.2, but 2560 ->
// 512 7.7 / 5.7).  Up to 16 rows, past the lines of the small-row kernel: everywhere but where
// rows_behind_streaming expects it to be slower (2048 -> 18944 9.2 / 10.8, 4096 -> 32768 16.8 / 21.5, 4864 -> 18944 17.1 / 19.0).  Of 2943
// products with K 4096 .. 8192 and 70 .. 250 M weights 151 are more than 3 % behind, 11 % at most, nearly all at K above 6912 (4 x 8192 -> 11488
// 19.3 / 17.5), the mean is 0.87; fits to both times do not tell those apart.  Of 3312 with K 8193 .. 11264 332, 25 % at most (4 x 11008 -> 16928
// 34.1 / 27.3), the mean is 0.94: there a division of K into 22 units is uneven whatever the splits.
// The forms for one or a few rows come first where they apply (the caller asks them before).  Above 64 rows the GEMM is
// faster; who must not round a weight asks for this kernel.
EAGLE_EXPORT int eagle_qmm_rows_preferred(int M, int N, int K) {
  if (M < 1 || M > 2 * EAGLE_MAX_M) return 0;
  if (M > 16 && M <= 32 && (double)N * K < 7e6 && K <= 4608) return 0;
  return eagle_qmm_rows_supported(M, N, K, 0) && !rows_plan(M, N, K, ROWS_SPLIT).behind;
}

EAGLE_EXPORT size_t eagle_qmm_rows_workspace_bytes(int M, int N, int K) {
  if (!eagle_qmm_rows_supported(M, N, K, 0)) return 0;
  const RowsPlan p = rows_plan(M, N, K, ROWS_SPLIT);
  return p.splits > 1 ? (size_t)p.splits * M * N * sizeof(float) : 0;
}

EAGLE_EXPORT int eagle_qmm_rows_w4g64_f16(const void* x, const uint32_t* wq, const void* scales, const void* biases, const void* bias,
                                          void* out, int M, int N, int K, int group_size, int bits, int swiglu, void* workspace,
                                          size_t workspace_bytes, eagle_stream_t stream) {
  if (!x || !wq || !scales || !biases || !out) return EAGLE_ERR_NULL;
  if (group_size != 64 || bits != 4) return EAGLE_ERR_UNSUPPORTED;
  if (!eagle_qmm_rows_supported(M, N, K, swiglu)) return EAGLE_ERR_SHAPE;
  const void* aligned[] = {x, wq, out, workspace};
  for (const void* p : aligned)
    if (p && !eagle_aligned16(p)) return EAGLE_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) return EAGLE_ERR_ALIGN;
  if (x == out) return EAGLE_ERR_UNSUPPORTED;          // other workgroups still read x
  const RowsPlan p = rows_plan(M, N, K, workspace ? ROWS_SPLIT : ROWS_WHOLE);
  if (p.form < 0) return EAGLE_ERR_SHAPE;
  if (p.splits > 1 && workspace_bytes < (size_t)p.splits * M * N * sizeof(float)) return EAGLE_ERR_WORKSPACE;
  RowsArgs a;
  a.x = static_cast<const half_t*>(x);
  a.w = wq;
  a.s = static_cast<const half_t*>(scales);
  a.b = static_cast<const half_t*>(biases);
  a.bias = static_cast<const half_t*>(bias);
  a.out = static_cast<half_t*>(out);
  a.partial = p.splits > 1 ? static_cast<float*>(workspace) : nullptr;
  a.M = M;
  a.N = N;
  a.K = K;
  a.swiglu = swiglu != 0;
  a.both = 0;
  a.pitch = M;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const RowsForm& form = rows_forms[p.form];
  const int rc = (M > 2 * EAGLE_MAX_M ? form.launch_many : form.launch)(a, p.splits, st);
  if (rc != EAGLE_OK || p.splits == 1) return rc;
  const dim3 grid((unsigned)(((long)M * ((swiglu ? N / 2 : N) / 8) + 255) / 256));
  if (swiglu)
    hipLaunchKernelGGL(rows_sum_kernel<true>, grid, dim3(256), 0, st, a.partial, p.splits, a.bias, a.out, M, N);
  else
    hipLaunchKernelGGL(rows_sum_kernel<false>, grid, dim3(256), 0, st, a.partial, p.splits, a.bias, a.out, M, N);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_qmm_rows_partial_splits(int M, int N, int K) {
  return M <= 2 * EAGLE_MAX_M && eagle_qmm_rows_supported(M, N, K, 0) ? rows_plan(M, N, K, ROWS_PARTIAL).splits : 0;
}

EAGLE_EXPORT int eagle_qmm_rows_partial_w4g64(const void* x, const uint32_t* wq, const void* scales, const void* biases, float* partial,
                                              size_t partial_bytes, int M, int N, int K, int group_size, int bits,
                                              eagle_stream_t stream) {
  if (!x || !wq || !scales || !biases || !partial) return EAGLE_ERR_NULL;
  if (group_size != 64 || bits != 4) return EAGLE_ERR_UNSUPPORTED;
  const int splits = eagle_qmm_rows_partial_splits(M, N, K);
  if (splits < 1) return EAGLE_ERR_SHAPE;
  if (!eagle_aligned16(x) || !eagle_aligned16(wq) || !eagle_aligned16(partial)) return EAGLE_ERR_ALIGN;
  if ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 3u) return EAGLE_ERR_ALIGN;
  RowsArgs a = {};
  a.x = static_cast<const half_t*>(x);
  a.w = wq;
  a.s = static_cast<const half_t*>(scales);
  a.b = static_cast<const half_t*>(biases);
  a.partial = partial;
  a.M = M;
  a.N = N;
  a.K = K;
  a.pitch = eagle_slab_rows(M);
  if (partial_bytes < (size_t)splits * a.pitch * N * sizeof(float)) return EAGLE_ERR_WORKSPACE;
  return rows_forms[rows_plan(M, N, K, ROWS_PARTIAL).form].launch(a, splits, static_cast<hipStream_t>(stream));
}
