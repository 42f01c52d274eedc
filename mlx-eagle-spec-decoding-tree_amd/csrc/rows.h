// The kernel of the product described in rows.hip, its launch, and the forms that rows.hip chooses among: a table per
// number of 16-row tiles of x, each in a source of its own (rows_1.hip .. rows_4.hip) so that they compile at once.
#pragma once
#include "common.h"

#include <type_traits>

// What rows.hip and the sources of forms share; the kernel and its launches are each source's own.
namespace eagle_rows {

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
  int pairs;              // K is dealt in pairs of chunks (1), or chunk by chunk (0)
  int units;              // of the longest K part
  uint32_t inv;           // 2^31 over the number of K parts, rounded up
};

constexpr int ROWS_WAVES = 8;
constexpr int ROWS_LDS = 160 * 1024;
constexpr int ROWS_RSRC = 0x00020000;      // buffer descriptor: untyped bytes
constexpr int ROWS_XROW = 256 + 16;        // bytes of a staged x row: a chunk of 128 columns, padded against bank conflicts

// bytes of a row's scales in LDS for `units` units of four chunks: an odd multiple of 16, so that sixteen rows
// sit in different banks
__host__ __device__ constexpr int rows_stride(int units) { return (units | 1) * 16; }

constexpr int rows_block(int MT, int KP) { return (MT > 2 ? 2 : 4) / KP > 0 ? (MT > 2 ? 2 : 4) / KP : 1; }

// bytes of LDS: two blocks of x, its sums, scales (and biases); at the end the sums of the K parts
inline size_t rows_lds_bytes(int RT, int RT2, int MT, int KP, int nu, bool both) {
  const size_t rows = 16 * MT, B = rows_block(MT, KP), wrows = ROWS_WAVES / KP / 2 * (RT + RT2) * 16;
  const size_t stage = 2 * KP * B * rows * ROWS_XROW + KP * 4 * nu * rows * 8 +
                       (both ? 2 : 1) * (size_t)ROWS_WAVES * RT * 16 * rows_stride(nu);
  const size_t epi = KP * rows * (wrows + 4) * 4;
  return stage > epi ? stage : epi;
}

// chunks in the last unit of the longest K part (of all workgroups along y and all parts)
inline int rows_last(int K, int parts) { return (((K >> 7) + parts - 1) / parts - 1) % 4 + 1; }

struct RowsForm {
  int rt, rt2, mt, kp;
  int (*launch)(const RowsArgs&, int, hipStream_t);
  int (*launch_half)(const RowsArgs&, int, hipStream_t);      // the last unit of a K part has at most two chunks
  int (*launch_many)(const RowsArgs&, int, hipStream_t);      // more than 64 rows (blocks of 48 or 64), or nullptr
  int (*launch_many_half)(const RowsArgs&, int, hipStream_t);
  int run(const RowsArgs& a, int splits, hipStream_t st) const {
    const bool half = rows_last(a.K, splits * kp) <= 2;
    return (a.M > 2 * EAGLE_MAX_M ? half ? launch_many_half : launch_many : half ? launch_half : launch)(a, splits, st);
  }
  int wrows() const { return ROWS_WAVES / kp / 2 * (rt + rt2) * 16; }
};
struct RowsTable {
  const RowsForm* forms;
  int count;
};
RowsTable forms_1();
RowsTable forms_2();
RowsTable forms_3();
RowsTable forms_4();

namespace {

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

// The part of a workgroup's wave: RT tiles from row0 on (the waves of a workgroup may differ in RT), then its sums in LDS.
template <int RT, int MOST, int WROWS, int MT, int KP, int AH, bool MANY, int REM>
__device__ inline void rows_wave(const RowsArgs& a, int nb, int m0, int wave, int kp, int row0) {
  constexpr int B = rows_block(MT, KP);            // chunks per K part and block of staged x
  constexpr int ROWS = 16 * MT;                    // rows of x
  constexpr int SLOT = ROWS * ROWS_XROW;           // bytes of a staged chunk
  constexpr int BUF = KP * B * SLOT;
  constexpr int NP = KP * B * ROWS * 16 / (ROWS_WAVES * 64);   // 16-byte pieces of x per thread and block
  static_assert(NP * ROWS_WAVES * 64 == KP * B * ROWS * 16, "x does not divide over the threads");
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
  const int lane = threadIdx.x & 63;
  const int r = lane & 15, kq = lane >> 4;
  const int K = a.K, M = MANY && a.M - m0 > ROWS ? ROWS : a.M - m0, N = a.N;
  const int all = K >> 7;
  // chunks of 128 columns, dealt over the K parts of all workgroups along y; worked off in units of four, the last of REM.
  // In pairs (the two halves of a line; the longest part has the units it has chunk by chunk), unless a.pairs is 0
  auto first = [&](int p) {
    // (exact while pairs times the square of the parts is below 2^31: 128 parts, K of 2^24.  Divided here, the first requests waited for some forty
    // instructions, and the compiler kept more addresses through the loop: nine vector instructions a unit with ten tiles, 32 x 3584 -> 152064
    // 0.3 to 0.6 % slower)
    const unsigned n = (unsigned)((all + a.pairs) >> a.pairs) * (blockIdx.y * KP + p);
    const int c = (int)((unsigned long)n * a.inv >> 31) << a.pairs;
    return c < all ? c : all;
  };
  // (Three tiles of x: the counters that the compiler makes of the addresses when the kernel works the units out itself are the faster loop, 34 x 4352 ->
  // 76632 48.6 us, 51.6 from the host; with one, two and four tiles the other way round, 32 x 3584 -> 152064 67.7, 67.2.)
  const int NU = MT == 3 ? ((all + (int)gridDim.y * KP - 1) / ((int)gridDim.y * KP) + 3) >> 2 : a.units;
  const int c0 = first(kp), nch = first(kp + 1) - c0;
  const int XC = 4 * NU;
  half2_t* xsum = reinterpret_cast<half2_t*>(rows_lds + 2 * BUF);      // [KP][XC][ROWS][2]: (hi, lo) of a group's sum
  // scales of this wave's rows for its K part [RT * 16][stride], then the biases if a.both
  const int stride = rows_stride(NU);
  unsigned char* const sbl = rows_lds + 2 * BUF + KP * XC * ROWS * 8 + wave * (MOST * 16) * stride * (a.both ? 2 : 1);

  // ---- addresses: buffer loads, a uniform offset per tile and chunk beside one 32-bit lane offset ----
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
      if ((u & 1) && (!last() || u - 1 + AH < REM)) {
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
    const bool more = !last() || u / B * B + B < REM;        // another block of x follows
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
  // fetched all the same, a workgroup of one unit spent a round trip to memory and a barrier on them (us with / without, timed in turn with equal shares
  // of the waves and whole last units:
  // 32 x 3584 x 4608 left as seven partial sums 7.07 / 6.53, 40 rows 8.0 / 7.7; 32 x 3584 x 37888 with SwiGLU 27.3 / 26.5, 40 x 3584 x
  // 152064 80.2 / 78.8, 128 x 3584 x 37888 55.0 / 53.9).
  for (int j = 0; j + 1 < NU; ++j) {
#pragma unroll
    for (int u = 0; u < 4; ++u) step(u, 4 * j + u, std::false_type{});
  }
#pragma unroll
  for (int u = 0; u < REM; ++u) step(u, 4 * (NU - 1) + u, std::true_type{});
  // The chunks that a short last unit leaves in the ring count as used: with the ring's last place read in the loop alone, the compiler fetched it
  // into other registers and copied it at the end of each unit, behind a wait for every load in flight
#pragma unroll
  for (int u = REM; u < AH; ++u)
#pragma unroll
    for (int t = 0; t < RT; ++t) asm volatile("" ::"v"(ring[u][t]));
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
    // (a last unit of two chunks: no sums of the others, whose biases are zero)
    const int held = 4 * (NU - 1) + REM - 1, xa = ca < held ? ca : held, xb = cb < held ? cb : held;
    half8_t xs[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const half4_t v0 = *reinterpret_cast<const half4_t*>(xsum + ((kp * XC + xa) * ROWS + mt * 16 + r) * 2);
      const half4_t v1 = *reinterpret_cast<const half4_t*>(xsum + ((kp * XC + xb) * ROWS + mt * 16 + r) * 2);
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
        red[(long)(kp * ROWS + mt * 16 + 4 * kq + i) * OROW + row0 - nb * WROWS + t * 16 + r] = acc[t][mt][i];
}

// MANY: more than one block of x rows.  RT2: tiles of the second half of the waves, which share the SIMDs with the first.
template <int RT, int RT2, int MT, int KP, int AH, bool MANY, int REM>
__global__ __launch_bounds__(ROWS_WAVES * 64) void qmm_rows_kernel(RowsArgs a) {
  constexpr int ROWS = 16 * MT;
  constexpr int RG = ROWS_WAVES / KP;              // groups of tiles side by side
  constexpr int WROWS = RG / 2 * (RT + RT2) * 16;  // weight rows per workgroup
  static_assert(WROWS % 32 == 0, "SwiGLU pairs the tiles of a workgroup");
  constexpr int OROW = WROWS + 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rg = wave / KP, kp = wave % KP;
  const int nb = MANY ? blockIdx.x / a.zb : blockIdx.x;                  // weight rows, then block of x
  const int m0 = MANY ? (blockIdx.x - nb * a.zb) * ROWS : 0;
  const int M = MANY && a.M - m0 > ROWS ? ROWS : a.M - m0, N = a.N;
  const int row0 = nb * WROWS + (rg < RG / 2 ? rg * RT : RG / 2 * RT + (rg - RG / 2) * RT2) * 16;
  if (RT == RT2 || rg < RG / 2)
    rows_wave<RT, RT, WROWS, MT, KP, AH, MANY, REM>(a, nb, m0, wave, kp, row0);
  else
    rows_wave<RT2, RT, WROWS, MT, KP, AH, MANY, REM>(a, nb, m0, wave, kp, row0);
  const float* red = reinterpret_cast<const float*>(rows_lds);
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

template <int RT, int RT2, int MT, int KP, int AH, bool MANY, int REM>
static int rows_launch(const RowsArgs& a, int splits, hipStream_t st) {
  constexpr int WROWS = ROWS_WAVES / KP / 2 * (RT + RT2) * 16;
  const int parts = splits * KP, nu = (((a.K >> 7) + parts - 1) / parts + 3) / 4;
  RowsArgs b = a;
  b.units = nu;
  b.inv = ((1u << 31) + parts - 1) / parts;
  b.zb = (a.M + 16 * MT - 1) / (16 * MT);
  b.both = rows_lds_bytes(RT, RT2, MT, KP, nu, true) <= ROWS_LDS;
  const size_t lds = rows_lds_bytes(RT, RT2, MT, KP, nu, b.both);
  if (lds > ROWS_LDS) return EAGLE_ERR_SHAPE;
  static bool ready = false;             // (set twice by two first calls at once: the same value)
  if (!ready) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(&qmm_rows_kernel<RT, RT2, MT, KP, AH, MANY, REM>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, ROWS_LDS) != hipSuccess)
      return EAGLE_ERR_HIP;
    ready = true;
  }
  hipLaunchKernelGGL((qmm_rows_kernel<RT, RT2, MT, KP, AH, MANY, REM>), dim3((a.N + WROWS - 1) / WROWS * b.zb, splits), dim3(ROWS_WAVES * 64), lds, st, b);
  return eagle_launch_status();
}

template <int RT, int RT2, int MT, int KP, int AH>
constexpr RowsForm rows_form() {
  constexpr auto whole = rows_launch<RT, RT2, MT, KP, AH, false, 4>, half = rows_launch<RT, RT2, MT, KP, AH, false, 2>;
  if constexpr (MT >= 3)
    return {RT, RT2, MT, KP, whole, half, rows_launch<RT, RT2, MT, KP, AH, true, 4>, rows_launch<RT, RT2, MT, KP, AH, true, 2>};
  else
    return {RT, RT2, MT, KP, whole, half, nullptr, nullptr};
}

}  // namespace
}  // namespace eagle_rows
