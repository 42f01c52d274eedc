// Shared declarations for the gfx950 kernels behind include/eagle_mi355x.h.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/eagle_mi355x.h"

#define EAGLE_EXPORT extern "C" __attribute__((visibility("default")))

typedef _Float16 half_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef float float16_t __attribute__((ext_vector_type(16)));
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint2_t __attribute__((ext_vector_type(2)));

static inline bool eagle_aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

static inline int eagle_launch_status() {
  return hipGetLastError() == hipSuccess ? EAGLE_OK : EAGLE_ERR_HIP;
}

// Wave-wide reductions over 64 lanes without the shuffles through LDS: halves and rows of sixteen lanes by lane swaps, then
// rotations within a row.  Every lane gets the result; sums are formed in the order of a butterfly from 32 lanes down (the
// same bits).  A norm over 32 x 3584 with seven slabs took 4.32 us with shuffles and takes 4.16 so, over 2048 x 3584 13.9
// and 12.65.
template <int ROR>
__device__ inline uint32_t wave_row_ror(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + ROR, 0xf, 0xf, true);
}
// over the lanes 32 and 16 apart, and over the sixteen lanes of a row
template <typename Op>
__device__ inline uint32_t wave_reduce32(uint32_t v, Op op) {
  const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);
  return op(a[0], a[1]);
}
template <typename Op>
__device__ inline uint32_t wave_reduce16(uint32_t v, Op op) {
  const auto a = __builtin_amdgcn_permlane16_swap(v, v, false, false);
  return op(a[0], a[1]);
}
template <typename Op>
__device__ inline uint32_t wave_reduce_row(uint32_t v, Op op) {
  v = op(v, wave_row_ror<8>(v));
  v = op(v, wave_row_ror<4>(v));
  v = op(v, wave_row_ror<2>(v));
  return op(v, wave_row_ror<1>(v));
}
template <typename Op>
__device__ inline uint32_t wave_reduce(uint32_t v, Op op) {
  return wave_reduce_row(wave_reduce16(wave_reduce32(v, op), op), op);
}
__device__ inline float wave_f32(uint32_t v) { return __builtin_bit_cast(float, v); }
__device__ inline uint32_t wave_u32(float v) { return __builtin_bit_cast(uint32_t, v); }
struct WaveAdd {
  __device__ uint32_t operator()(uint32_t a, uint32_t b) const { return wave_u32(wave_f32(a) + wave_f32(b)); }
};
struct WaveMax {
  __device__ uint32_t operator()(uint32_t a, uint32_t b) const { return wave_u32(fmaxf(wave_f32(a), wave_f32(b))); }
};
__device__ inline float wave_sum(float v) { return wave_f32(wave_reduce(wave_u32(v), WaveAdd())); }
__device__ inline float wave_max(float v) { return wave_f32(wave_reduce(wave_u32(v), WaveMax())); }

// Eight nibbles -> fp16 q, exact, in the order q0 q2 q4 q6 q1 q3 q5 q7.  A byte that holds a nibble is, read as OCP e4m3,
// q * 2^-9 (subnormals up to 7, the first exponents up to 15), so the fp8 conversion gives the fp16 values of q two at a
// time: seven instructions per packed word.
__device__ inline half8_t eagle_expand8(uint32_t w) {
  const uint32_t lo = w & 0x0f0f0f0fu, hi = (w >> 4) & 0x0f0f0f0fu;
  union { half2_t h2[4]; half8_t h8; } o;
  o.h2[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.f, false);
  o.h2[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.f, true);
  o.h2[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.f, false);
  o.h2[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.f, true);
  return o.h8;
}
// eight values of x in that order
__device__ inline half8_t eagle_permute8(half8_t v) { return half8_t{v[0], v[2], v[4], v[6], v[1], v[3], v[5], v[7]}; }

// A pair (x1, x2) turned by an angle: a fused multiply-add on a product rounded to fp32, then fp16.  Every rotation in the library is this one, so
// that they agree bit for bit.  The sums are held in fp32 registers: folded into mixed-precision instructions by the compiler's choice
// they were rounded once to fp16, other elements of the same kernel twice (three values of a million differ).
__device__ inline half2_t eagle_rotate(float x1, float x2, float co, float sn) {
  float lo = __builtin_fmaf(x1, co, -(x2 * sn)), hi = __builtin_fmaf(x1, sn, x2 * co);
  asm("" : "+v"(lo), "+v"(hi));
  return half2_t{(half_t)lo, (half_t)hi};
}

// Rows of a partial tile of the slab form: 32 for up to 32 rows of x, 64 for 33..64.
__host__ __device__ inline int eagle_slab_rows(int M) { return M > 32 ? 64 : 32; }

// Eight consecutive values of a matmul result that is held as fp32 partial sums of K slabs
// (eagle_qmm_slab_partial_w4g64): fp16 of the sum in slab order, then the fp16 bias.  `at` is
// the element offset inside a slab, `stride` the elements per slab.  Up to twelve slabs are requested before
// the first add, and none twice (a norm over 32 x 3584 with ten slabs: 5.1 us with eight at a time, 4.7 so; seven 4.3, 4.2).
__device__ inline half8_t eagle_slab_sum8(const float* __restrict__ partial, int nslab, size_t stride,
                                          size_t at, const half_t* __restrict__ bias8) {
  float4_t lo = float4_t{0.f, 0.f, 0.f, 0.f}, hi = lo;
  const float* p = partial + at;
  for (int z = 0; z < nslab; z += 12) {
    float4_t a[12], c[12];
#pragma unroll
    for (int k = 0; k < 12; ++k)
      if (z + k < nslab) {
        a[k] = *reinterpret_cast<const float4_t*>(p + (size_t)(z + k) * stride);
        c[k] = *reinterpret_cast<const float4_t*>(p + (size_t)(z + k) * stride + 4);
      }
#pragma unroll
    for (int k = 0; k < 12; ++k)
      if (z + k < nslab) {
        lo += a[k];
        hi += c[k];
      }
  }
  half8_t v = half8_t{(half_t)lo[0], (half_t)lo[1], (half_t)lo[2], (half_t)lo[3],
                      (half_t)hi[0], (half_t)hi[1], (half_t)hi[2], (half_t)hi[3]};
  if (bias8) {
    const half8_t b8 = *reinterpret_cast<const half8_t*>(bias8);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = v[e] + b8[e];
  }
  return v;
}
