// 4-bit group-64 quantised product for 2..2048 rows of x on the weights in the MLX layout, no weight rounded:
// out[m][n] = fp16( sum_k x[m][k] (s[n,k/64] q[n,k] + b[n,k/64]) ) (+ bias[n]), or silu(g) * u of gate and up
// rows interleaved in 16-row tiles.  (Reference: mx.quantized_matmul, mlx_model_fwd_bench.py:65-73; the
// factorisation of kernels/qmv/1b.metal:121-147.)
//
//   * A workgroup of eight waves owns 8 / KP groups of RT 16-row weight tiles over a range of K; KP waves share a
//     group, each with a part of the range.  The second half of the waves, which sits on the SIMDs of the first, may take a tile
//     less, and the parts of K are dealt in chunks of 128 columns: a SIMD then has five tiles instead of four or six, and a part of fourteen chunks is
//     three and a half units of the loop, not four (32 x 3584 -> 37888 with SwiGLU 28.1 us -> 24.0, 40 rows 32.0 -> 29.2, 64 rows 38.9 -> 32.8;
//     40 x 18944 -> 3584 left as partial sums 19.6 -> 18.7).  Wide matrices take many tiles per workgroup (x is read by fewer), narrow
//     ones few tiles and K split over workgroups, whose fp32 partial sums a second launch adds (rows_plan).
//   * A product whose parts are added here deals K in pairs of chunks, the two 64-byte halves of a line: a part that begins with a second half
//     requests no line whole, and the line at each seam twice (8 x 10240 -> 21064 in three parts 35.5 us chunk by chunk, 30.7 in pairs; 3 x 13568 ->
//     17888 39.2, 34.4; 40 x 18944 -> 3584 23.0, 22.4).  One that is left as partial sums deals single chunks: alone it gains as much, but in the
//     middle of a tree pass's weights the longer parts cost more (40 tokens 2519 us, 2533 in pairs).
//   * Weights go from memory to registers, 16 bytes per lane, a ring of AH chunks of 128 columns ahead; both 64-byte
//     halves of a line are requested together (of two lines, where a part begins at an odd chunk).  Two half-wave swaps deal the words of a lane so that a matrix
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
// with the sums of a tile added behind its matrix instructions, 54 under the next tile's, 49 with unequal shares of the waves).  In a prompt pass, weights
// not in a cache: 732 and (2048 x 3584 x 18944) 372 us against 553 and 263; matrix pipes 37 % busy at 2.05 GHz.
#include "rows.h"

using namespace eagle_rows;

namespace {

// The partial sums of a split product added in split order: fp16 (+ bias), or silu(g) * u of interleaved gate|up
// rows.  Four outputs per thread and one wave per workgroup, every load in flight before the first add.  What a compute unit takes in of
// its partial sums bounds it: with eight outputs and 256 threads 27 x 18944 -> 3584 had 48 workgroups with 73 KB each (the product with it 17.4 us,
// 16.9 with 378).
constexpr int SUM_WAVE = 64;
__device__ inline float4_t rows_sum4(const float* __restrict__ p, int splits, size_t stride) {
  float4_t sum = {0.f, 0.f, 0.f, 0.f};
  for (int z = 0; z < splits; z += 12) {
    float4_t a[12];
#pragma unroll
    for (int k = 0; k < 12; ++k)
      if (z + k < splits) a[k] = *reinterpret_cast<const float4_t*>(p + (size_t)(z + k) * stride);
#pragma unroll
    for (int k = 0; k < 12; ++k)
      if (z + k < splits) sum += a[k];
  }
  return sum;
}
template <bool SWI>
__global__ __launch_bounds__(SUM_WAVE) void rows_sum_kernel(const float* __restrict__ partial, int splits, const half_t* __restrict__ bias,
                                                            half_t* __restrict__ out, int M, int N) {
  const int per_row = (SWI ? N >> 1 : N) >> 2;
  const int idx = blockIdx.x * SUM_WAVE + threadIdx.x;
  if (idx >= M * per_row) return;
  const int m = idx / per_row, o4 = (idx % per_row) * 4;
  const int n = SWI ? (o4 >> 4) * 32 + (o4 & 15) : o4;
  const size_t stride = (size_t)M * N;
  const float* p = partial + (size_t)m * N + n;
  const float4_t g = rows_sum4(p, splits, stride), u = SWI ? rows_sum4(p + 16, splits, stride) : g;
  half4_t r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    r[e] = (half_t)g[e];
    if (bias) r[e] = r[e] + bias[n + e];
    if (SWI) {
      half_t ue = (half_t)u[e];
      if (bias) ue = ue + bias[n + 16 + e];
      const float gf = (float)r[e];
      const half_t act = (half_t)(gf / (1.0f + expf(-gf)));
      r[e] = (half_t)((float)act * (float)ue);
    }
  }
  *reinterpret_cast<half4_t*>(out + (size_t)m * (SWI ? N >> 1 : N) + o4) = r;
}

struct RowsPlan {
  const RowsForm* form;
  int splits;
  bool behind;         // the streaming kernel takes this product instead
};

// The division of the work with the least predicted time (us), from a model fitted to timings of every form, launches
// back to back over rotating weights in a graph.  A compute unit takes its workgroups one after the other; each costs its start, its
// share of the weights and its x, with more K parts more barriers.  What the whole grid reads counts a little, a split as much as
// its second launch and the partial sums (the sums alone where the consumer of the product adds them).  Constants by the
// rows: up to 16, 17 .. 32, 33 .. 48, more; above 64 the last over the blocks of x.  The second launch counts 0.6 us less from 17 rows on than the fit
// gave for its first kernel: of 9900 products of 17 .. 64 rows that take another division for it the mean is 0.94, 0.94 and 0.98 of the time, one in ten
// loses more than 3 %, 21 at most (46 x 2432 -> 5720).  The choice against the best of the divisions within 1.35 of the least predicted time, this kernel
// and this launch, 16950 products (141000 timings): 0.7, 0.8, 1.1 and 0.8 % longer on average, 5, 6, 7 and 6 at the 95th percentile; of 1620
// products of 65 .. 512 rows (13500 timings) 1.0 and 6.  Splits of up to three rows count as those of four (2 x 11008 -> 18944 chose another division: 36.1 us, 33.1).
enum { ROWS_WHOLE = 0, ROWS_SPLIT = 1, ROWS_PARTIAL = 2 };
struct RowsCost {
  double start, w, x, unit, parts, whole, second, sums, rows;
};
constexpr RowsCost rows_cost_one = {2.11, 0.0309, 0.0107, 0.0448, 0.419, 0.0018, 2.60, 1.353, 5.};
constexpr RowsCost rows_cost_two = {3.89, 0.0416, 0.0058, 0., 0.293, 0.0068, 2.62, 0.459, 0.};
constexpr RowsCost rows_cost_three = {4.23, 0.0484, 0.0104, 0., 0.0887, 0.0070, 2.86, 0.336, 0.};
constexpr RowsCost rows_cost = {1.03, 0.0246, 0.0138, 0.221, 0., 0.0107, 2.33, 0.49, 0.};

// What the norm or rope launch that adds the partial sums takes for them, us per MB: 40 rows of 18944 -> 3584 are left as nine instead of thirteen
// (19.1 us either way; the norm behind them reads 5.2 instead of 7.5 MB: 4.1 for 5.3 us).  Timed over 1 .. 16 parts that launch takes 0.24 .. 0.6 a MB as a
// norm (64 .. 18 rows of 3584; nearly nothing up to five parts, most past nine) and 0.1 .. 0.23 as a rotation (18 .. 64 rows of 4608).  The line lies low
// on purpose: at 0.37 32 x 3584 -> 4608, which a rotation adds, would lose 1.3 us on the product for 0.9 behind it.
constexpr double rows_read = 0.18;

// Up to 16 rows of x, K up to 2048 or 70 .. 250 M weights: whether the streaming kernel is faster than this one by the form (rt tiles, kp
// parts, no splits).  That kernel deals the tiles of 16 weight rows evenly over the compute units, where this one has whole rounds of 128 .. 640
// weight rows a workgroup: at 100000 weight rows half of the second round idles (3 x 1152 -> 102016 22.8 us, 18.9; 10 x 640 -> 99944 17.2, 14.9;
// 4 x 2816 -> 34496 17.9, 16.9), while 28672 or 152064 fill theirs (8 x 512 -> 152064 12.4, 18.3; 8 x 3584 -> 28672 14.3, 17.2).  Both times (us) from
// fits to 1779 such products of 16000 weight rows up, 2.7 and 3 % rms: the streaming kernel's by its waves, one per 256 columns, and the tiles of
// a workgroup, which come in steps of four.  This kernel is more than 3 % behind in 345 of them, with the rule in 76 (8 %: 93, 6), and the rule
// loses more than 3 % in 20.  (The streaming kernel's result is further from the exact one before it is rounded: 0.02 .. 0.5 % more error after.)
// The rule looks at the division into equal shares and whole units only.  (Where the plan has unequal shares instead, this kernel takes 0.97 of the
// streaming kernel's time over 3076 products that the rule sends there, 1.04 at the 95th percentile: not changed.)
bool rows_behind_streaming(int M, int N, int K, const RowsForm& form) {
  const double size = (double)N * K;
  if (M > 16 || N <= 16000 || K > 3584 || (K > 2048 && (size <= 7e7 || size >= 2.5e8))) return false;
  const int waves = (K + 255) >> 8, all = (N + 15) >> 4, tiles = (all + 255) / 256, steps = (tiles + 3) / 4;
  static const double start[] = {4.02, 5.08, 5.86}, tile[] = {0.313, 0.454, 0.864}, step[] = {0.094, 0.282, 0.343}, more[] = {0.152, 0.343, 0.444};
  static const int least[] = {2, 5, 9};
  const int b = waves <= 4 ? 0 : waves <= 8 ? 1 : 2;
  const double stream = start[b] + (tile[b] + (K % 256 ? 0.028 : 0.) + 0.0037 * M) * tiles + (step[b] + more[b] * (waves - least[b])) * steps;
  const int rt = form.rt, units = ((K >> 7) + 3) / 4, kp = form.kp, nu = (units + kp - 1) / kp, wrows = form.wrows();
  const int blocks = (N + wrows - 1) / wrows, rounds = (blocks + 255) / 256;
  const double rows = 1.32 + rounds * (1.94 + 0.396 * rt + (0.517 + 0.0065 * M) * nu * rt + 0.197 * nu * kp + (K % 512 ? 0.104 * rt : 0.)) +
                      blocks / 256. * 0.519 * nu * rt + 0.027e-6 * size;
  return stream < 0.98 * rows;
}

RowsPlan rows_find_plan(int M, int N, int K, int mode) {
  const int chunks = K >> 7, units = (chunks + 3) / 4;
  const int least_zb = (M + 63) / 64, mt = (M + 16 * least_zb - 1) / (16 * least_zb), zb = (M + 16 * mt - 1) / (16 * mt);
  const RowsCost& cost = mt == 1 ? rows_cost_one : mt == 2 ? rows_cost_two : M <= 48 ? rows_cost_three : rows_cost;
  RowsPlan best = {nullptr, 1, false}, even = best;
  double least = 1e30, least_even = 1e30;
  const RowsTable table = mt == 1 ? forms_1() : mt == 2 ? forms_2() : mt == 3 ? forms_3() : forms_4();
  for (int f = 0; f < table.count; ++f) {
    const RowsForm& form = table.forms[f];
    const int wrows = form.wrows();
    const double rt = 0.5 * (form.rt + form.rt2);
    const long blocks = (long)((N + wrows - 1) / wrows) * zb;
    auto time = [&](int z, double nu) {
      const double rounds = (double)((blocks * z + 255) / 256);
      const double w = wrows * nu * form.kp * (512 * 0.5625 / 1e3), x = 16. * mt * nu * form.kp * (1024 / 1e3);
      const double t = rounds * (cost.start + cost.w * w + cost.x * x + (cost.unit * rt * mt + cost.parts * (form.kp - 1)) * nu) +
                       cost.whole * (blocks * z / 256.) * (w + 0.5 * x);
      return z == 1 ? t : t + (mode == ROWS_SPLIT ? cost.second : 0.) + (cost.sums + (mode == ROWS_PARTIAL ? rows_read : 0.)) * 4e-6 * z * ((M > 4 ? M : 4) + cost.rows) * N;
    };
    double last = 0.;
    for (int z = 1; z <= (mode == ROWS_WHOLE ? 1 : 32) && units / z >= form.kp; ++z) {
      const int whole = ((chunks + z * form.kp - 1) / (z * form.kp) + 3) / 4;
      const double nu = whole - (rows_last(K, z * form.kp) <= 2 ? 0.5 : 0.);
      if (nu == last) continue;                    // more workgroups, none of them shorter
      last = nu;
      if (rows_lds_bytes(form.rt, form.rt2, mt, form.kp, whole, false) > ROWS_LDS) continue;
      const double t = time(z, nu), t_even = time(z, whole);
      if (t < least) {
        least = t;
        best = {&form, z, false};
      }
      if (form.rt == form.rt2 && t_even < least_even) {
        least_even = t_even;
        even = {&form, z, false};
      }
    }
  }
  if (even.form && even.splits == 1) best.behind = rows_behind_streaming(M, N, K, *even.form);
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
         (long)N * K < (1L << 33) && rows_plan(M, N, K, ROWS_SPLIT).form != nullptr;
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
  if (!p.form) return EAGLE_ERR_SHAPE;
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
  a.pairs = 1;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const int rc = p.form->run(a, p.splits, st);
  if (rc != EAGLE_OK || p.splits == 1) return rc;
  const dim3 grid((unsigned)(((long)M * ((swiglu ? N / 2 : N) / 4) + SUM_WAVE - 1) / SUM_WAVE));
  if (swiglu)
    hipLaunchKernelGGL(rows_sum_kernel<true>, grid, dim3(SUM_WAVE), 0, st, a.partial, p.splits, a.bias, a.out, M, N);
  else
    hipLaunchKernelGGL(rows_sum_kernel<false>, grid, dim3(SUM_WAVE), 0, st, a.partial, p.splits, a.bias, a.out, M, N);
  return eagle_launch_status();
}

EAGLE_EXPORT int eagle_qmm_rows_plan(int M, int N, int K, int mode, int* plan6) {
  if (!plan6) return EAGLE_ERR_NULL;
  if (mode < ROWS_WHOLE || mode > ROWS_PARTIAL) return EAGLE_ERR_UNSUPPORTED;
  if (!eagle_qmm_rows_supported(M, N, K, 0) || (mode == ROWS_PARTIAL && M > 2 * EAGLE_MAX_M)) return EAGLE_ERR_SHAPE;
  const RowsPlan p = rows_plan(M, N, K, mode);
  if (!p.form) return EAGLE_ERR_SHAPE;
  const int plan[] = {p.form->rt, p.form->rt2, p.form->mt, p.form->kp, p.splits, rows_last(K, p.splits * p.form->kp) <= 2 ? 2 : 4};
  for (int i = 0; i < 6; ++i) plan6[i] = plan[i];
  return EAGLE_OK;
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
  a.pairs = 0;
  if (partial_bytes < (size_t)splits * a.pitch * N * sizeof(float)) return EAGLE_ERR_WORKSPACE;
  return rows_plan(M, N, K, ROWS_PARTIAL).form->run(a, splits, static_cast<hipStream_t>(stream));
}
