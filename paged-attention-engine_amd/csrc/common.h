// Shared device helpers for the gfx950 kernels: storage types, conversions,
// wavefront reductions and the error convention of the C entry points.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_bf16.h>
#include <stdint.h>

#define PAE_WAVE 64

// dtype codes shared with the Python side
#define PAE_F32 0
#define PAE_BF16 1

typedef __hip_bfloat16 bf16_t;

// Every entry point returns 0 on success.  On refusal it returns a negative code
// and leaves a message that pae_last_error() hands to the caller.
extern "C" const char* pae_last_error();
int pae_fail(const char* fmt, ...);
int pae_check_launch(const char* what);

#define PAE_REQUIRE(cond, ...)                 \
  do {                                         \
    if (!(cond)) return pae_fail(__VA_ARGS__); \
  } while (0)

__device__ __forceinline__ float to_f32(float x) { return x; }
__device__ __forceinline__ float to_f32(bf16_t x) { return __bfloat162float(x); }

template <typename T>
__device__ __forceinline__ T from_f32(float x);
template <>
__device__ __forceinline__ float from_f32<float>(float x) { return x; }
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float x) { return __float2bfloat16(x); }

// Value of x after a round trip through storage type T (round-to-nearest-even).
template <typename T>
__device__ __forceinline__ float round_to(float x) { return to_f32(from_f32<T>(x)); }

// A vector parameter (norm weight, bias) may be stored in float32 even when
// activations are bfloat16: `is_f32` says which.
__device__ __forceinline__ float load_param(const void* p, int is_f32, int64_t i) {
  return is_f32 ? ((const float*)p)[i] : __bfloat162float(((const bf16_t*)p)[i]);
}

// Activations by code (0 gelu by erf, 1 gelu by tanh, 2 silu, 3 the square of relu), in float32.
#define PAE_LAST_ACTIVATION 3
__device__ __forceinline__ float act_of(float z, int kind) {
  if (kind == 0) return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f));
  if (kind == 1) return 0.5f * z * (1.0f + tanhf(0.79788456080286536f * (z + 0.044715f * z * z * z)));
  if (kind == 3) return z > 0.f ? z * z : 0.f;
  return z / (1.0f + expf(-z));
}

// The same where the result is rounded to bfloat16, by the unit's own exponential and reciprocal with what they round away put back.  Their error
// against 64 bits before that rounding is no larger than act_of's (normally distributed z, 2-norm of the error over that of the results, act_of
// and here: SiLU 3.94e-8 and 3.94e-8, GELU by tanh 3.75e-8 and 2.72e-8, by erf 3.85e-8 and 2.92e-8), in 13, 13 and 24 vector instructions beside
// those two instead of 24, about 40 and about 40.  The epilogue of a product's 256 x 256 tile forms 64 a lane while no matrix core works: us with act_of and
// with these, SiLU with the gate in it 2,048 x 17,920 x 1,536 104.7 and 100.6, 8,192 of it 363 and 347, 6,030 x 37,888 x 3,584 1,182 and 1,161; GELU by tanh 8,192 x
// 17,920 x 1,536 403 and 367 (with tiles one after another as well); by erf 2,048 x 8,960 x 1,536 68.3 and 60.6, 300 rows 21.1 and 17.5.  (SiLU without what puts
// the roundings back: 96.4, 334 and 1,130, 1e-6 of the result off at z = -8 and 8e-6 at -88.)

// z / d for d from 1 on, infinity too: q z's product with the reciprocal r, `left` what that leaves of z.  The reciprocal is taken of a 2^32nd: of up
// to 2^128 it is a number below 2^-126, which the unit does not give.
__device__ __forceinline__ float over_one(float d) { return __builtin_amdgcn_rcpf(d * 0x1p-32f) * 0x1p-32f; }
__device__ __forceinline__ float quotient(float left, float r, float q, float z, float d) { return __builtin_amdgcn_div_fixupf(fmaf(left, r, q), d, z); }
__device__ __forceinline__ float silu_to_bf16(float z) {
  const float c = __builtin_amdgcn_fmed3f(z, -126.f, 126.f), n = rintf(c * -1.44269504088896341f);
  const float f = fmaf(c, -1.925963033500e-8f, fmaf(c, -1.44269504088896341f, -n));  // log2(e) in two parts
  const float d = 1.0f + ldexpf(__builtin_amdgcn_exp2f(f), (int)n), r = over_one(d), q = z * r;
  return quotient(fmaf(-q, d, z), r, q, z, d);
}
// Half of 1 + tanh(u) is 1 / (1 + exp(-2 u)).  (The tanh's form takes 1 + tanh apart where it is small: at z = -4 it is 4e-4 of the result off.)  What
// is rounded off the sum counts in what is left.
__device__ __forceinline__ float gelu_tanh_to_bf16(float z) {
  const float e = __builtin_amdgcn_exp2f(-2.30220819813f * fmaf(0.044715f * z * z, z, z)), d = 1.0f + e, r = over_one(d), q = z * r;
  return quotient(fmaf(-q, (1.0f - d) + e, fmaf(-q, d, z)), r, q, z, d);
}
// By the complementary error function of x = |z| / sqrt(2): erfc(x) = exp(-x^2) (1 + s q(s)), s = 0.35 x / (1 + 0.35 x), q of degree 8 fitted to
// exp(x^2) erfc(x) over 0 <= x <= 9.4 for the least largest relative error (Lawson's iteration), 1.5e-8, 1.4e-7 with the numbers below.  What is rounded
// in q counts by s: at z = 0 nothing of it does.
__device__ __forceinline__ float gelu_to_bf16(float z) {
  const float a = fminf(fabsf(z), 1e30f);  // (at infinity, where half is 0, a product with it would be no number)
  const float x = 0.247487373f * a, s = x * __builtin_amdgcn_rcpf(1.0f + x);
  float q = -0.0339356177f;
  q = fmaf(q, s, 0.101851627f);
  q = fmaf(q, s, -0.0206512567f);
  q = fmaf(q, s, -0.23625496f);
  q = fmaf(q, s, 0.0798865706f);
  q = fmaf(q, s, 0.972347021f);
  q = fmaf(q, s, -2.22093511f);
  q = fmaf(q, s, 2.46963143f);
  q = fmaf(q, s, -1.61196935f);
  const float half = fmaf(q, s, 0.5f) * __builtin_amdgcn_exp2f(z * z * -0.72134752044448170f);
  return z < 0.f ? z * half : fmaf(-a, half, z);
}
template <typename T>
__device__ __forceinline__ float act_to(float z, int kind) {
  if (sizeof(T) == 2) {
    if (kind == 0) return gelu_to_bf16(z);
    if (kind == 1) return gelu_tanh_to_bf16(z);
    if (kind == 2) return silu_to_bf16(z);
  }
  return act_of(z, kind);
}

// Reductions over a wavefront by a butterfly: every lane meets the lane 32, 16, 8, 4, 2 and 1 away, in this
// order, and all lanes end with the same value.  No step goes through LDS (a shuffle does, about 100 clocks
// each): the halves and the rows of 16 lanes change places by v_permlane32_swap and v_permlane16_swap; within a
// row the lanes are rotated by 8, 4, 2 and 1, which brings the partner or a lane that by then holds the
// partner's value.
template <int ROTATE>
__device__ __forceinline__ float row_rotated(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x120 + ROTATE, 0xf, 0xf, true));
}

template <typename Op>
__device__ __forceinline__ float wave_reduce(float v, Op op) {
  const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(halves[0]), __uint_as_float(halves[1]));
  const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = op(__uint_as_float(rows[0]), __uint_as_float(rows[1]));
  v = op(v, row_rotated<8>(v));
  v = op(v, row_rotated<4>(v));
  v = op(v, row_rotated<2>(v));
  return op(v, row_rotated<1>(v));
}

__device__ __forceinline__ float wave_sum(float v) {
  return wave_reduce(v, [](float a, float b) { return a + b; });
}

__device__ __forceinline__ float wave_max(float v) {
  return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); });
}

// Sum over a block of `NW` wavefronts in a fixed order: lanes by butterfly,
// then wave partials 0..NW-1 in sequence.  `scratch` holds NW floats in LDS.
template <int NW>
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x / PAE_WAVE;
  if ((threadIdx.x & (PAE_WAVE - 1)) == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) total += scratch[w];
  __syncthreads();
  return total;
}
