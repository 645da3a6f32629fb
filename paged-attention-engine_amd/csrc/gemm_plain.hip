// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]): the plain matrix product of the
// float32 path, also available for bfloat16 operands with float32 accumulation.
//
// W is stored (out_features, in_features) row-major as in the checkpoint, the
// layout F.linear takes in the reference (engine/model.py:303-305,315,318-320).
//
// Products run on the bfloat16 matrix cores (v_mfma_f32_16x16x32_bf16).  A float32 number is the sum of three bfloat16 numbers that hold
// its 24 bits, and of the nine products of two numbers' parts the six that reach a float32 product's last bit are
// added in float32; the three left out are below 2^-24 of the product, half a unit of its last place, of either sign (root mean square of
// normal operands 2^-27.4).  bfloat16 numbers are one part and take one product.  The
// float32 instructions (v_mfma_f32_16x16x4_f32), which these replace, add up four products at a time and give 154 TFLOP/s on the
// whole chip; six of the others do the work at up to 230.  A slab's products are a sum of their own before they join the others'.  Error
// against 64 bits (root mean square, share of the result's; normal operands): k 1,536 4.1e-7 before, 1.0e-7 now; 8,960 4.1e-7 and
// 1.6e-7; 18,944 4.2e-7 and 2.1e-7; bfloat16 operands 1.7e-7 and 0.9e-7.  (Rows with one or two numbers only are further off than before, 3.5e-8
// against 2.5e-8 and 3.3e-8 against 3.1e-8: the last of the six instructions does not always round to the nearest.  Adding it up apart from
// the others mends that and takes tiles of 128 x 256 6 to 9 % longer.)
//
// k is cut into slabs of 32, one set of instructions each, and into blocks of 512 whose sums are then added up in
// order (with rows of 30,000 terms one running sum loses a digit more than the block sums do).  Every kernel here adds in this
// order, so that the value of an output element does not depend on M, on the tile it falls in, on how
// the blocks are shared out or on which other rows share the launch.
//
// Why three kernels.  Up to 32 rows the weights' way from memory is the time: `few` gives 16 weight
// rows to a workgroup whose wavefronts take a block of k each, or a part of one where they are few (a wavefront reads 16
// rows x 64 bytes an instruction).  With more rows the matrix cores are: `tiles` takes the numbers apart once and stages the
// parts of 32 of k through LDS, two buffers that take turns.  Where a launch has too
// few tiles for the chip the blocks of k are shared out over workgroups as well: the
// block sums go to scratch memory and `sum` adds them in order.
// Measured, weights from HBM, 2,048 / 1,536 / 17,920 x 1,536 and 1,536 x 8,960, with the float32 instruction in tiles of 64 x 64 and now:
//   3 rows     6.9, 6.8, 26.3 (4.2 TB/s), 23 us      8.0, 7.9, 26.7, 22 us
//   64 rows    18, 18, 78, 65                        17, 18, 46, 26
//   300 rows   27, 27, 173, 96                       25, 24, 135, 85
//   601 rows   51, 39, 332 (100 TFLOP/s), 188        43, 33, 264 (125 TFLOP/s), 131
//   2,048      117, 90, 985, 488                     101, 79, 703 (160), 369
// The nearest second part and the factor 2^16 are two of the 8.5 instructions that take a number apart: without them 601 rows take 253
// and 127 us instead of 264 and 131.
// Tried: W's rows from memory straight to the registers they are multiplied from (a wavefront's load then touches 16 lines, and what
// a slab needs took 2.4 us to arrive); numbers taken apart with conversions and dot products (see half_parts_of); loads under a condition
// (see load8_anyhow);
// all six products straight into the running sums (601 x 17,920 x 1,536 226 us, but an error of 3.4e-7 that leans to one side: a model's
// logits were 1.8e-6 off instead of 1.5e-6).  In `few`
// the compiler moves the loads of a batch down to where they are used unless it is told not to (sched_barrier): 18.8
// against 15.3 us a launch in the step.
#include "common.h"
#include "api.h"

#define GP_BLOCK 512  // k of a block whose sum is formed before it joins the total
#define GP_SLAB 32    // k of one instruction
#define GP_UP 65536.f  // float32 operands are taken times this, and sums of products divided by its square
#define GP_FEW_ROWS 32  // (64 where rows are read number by number)
#define GP_FEW_WAVES 8
#define GP_FEW_MOST 12  // wavefronts of up to 16 rows, where blocks of k are spread
#define GP_STAGED_ROWS 8
#define GP_TILE 64    // parts of a product are cut in multiples of it
#define GP_UNITS 256  // compute units

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Eight numbers of a row's slab as they lie in memory: lane group (or thread of four) q holds the fours at 4 q and at 16 + 4 q, so that
// the four that read a row side by side ask for 64 bytes in a row.  Which of an instruction's k a number stands at is free as
// long as both sides agree.
template <typename T>
struct Eight;
template <>
struct Eight<float> {
  f32x4 v[2];
};
template <>
struct Eight<bf16_t> {
  uint2 v[2];
};
// Group q's of the slab at k; rows may be read four numbers at a time.
__device__ __forceinline__ void load8(Eight<float>& e, const float* row, int k, int q) {
  e.v[0] = *(const f32x4*)(row + k + q * 4);
  e.v[1] = *(const f32x4*)(row + k + 16 + q * 4);
}
__device__ __forceinline__ void load8(Eight<bf16_t>& e, const bf16_t* row, int k, int q) {
  e.v[0] = *(const uint2*)(row + k + q * 4);
  e.v[1] = *(const uint2*)(row + k + 16 + q * 4);
}
// The same of a row that ends at `end`, four numbers at a time (FOURS: `end` is a multiple of four) or one, without a condition around
// a load (one makes the compiler wait for every load on its way): what lies from `end` on is
// read elsewhere in the row, and `cut` makes it zero when it is there.
template <bool FOURS>
__device__ __forceinline__ void load8_anyhow(Eight<float>& e, const float* row, int k, int q, int end) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int at = k + 16 * h + q * 4;
    if (FOURS) {
      e.v[h] = *(const f32x4*)(row + min(at, end - 4));
    } else {
#pragma unroll
      for (int u = 0; u < 4; ++u) e.v[h][u] = row[min(at + u, end - 1)];
    }
  }
}
template <bool FOURS>
__device__ __forceinline__ void load8_anyhow(Eight<bf16_t>& e, const bf16_t* row, int k, int q, int end) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int at = k + 16 * h + q * 4;
    if (FOURS) {
      e.v[h] = *(const uint2*)(row + min(at, end - 4));
    } else {
      uint32_t w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = ((const uint16_t*)row)[min(at + u, end - 1)];
      e.v[h] = uint2{w[0] | w[1] << 16, w[2] | w[3] << 16};
    }
  }
}
__device__ __forceinline__ void cut(Eight<float>& e, int k, int q, int end) {
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (k + u / 4 * 16 + q * 4 + u % 4 >= end) e.v[u / 4][u % 4] = 0.f;
}
__device__ __forceinline__ void cut(Eight<bf16_t>& e, int k, int q, int end) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int left = end - (k + 16 * h + q * 4);  // numbers of the four that there are
    e.v[h].x &= left >= 2 ? ~0u : left == 1 ? 0xffffu : 0u;
    e.v[h].y &= left >= 4 ? ~0u : left == 3 ? 0xffffu : 0u;
  }
}

// The eight, times 2^16, as sums of bfloat16 numbers, largest part first: three of them hold a float32's 24 bits.  Times 2^16 the
// smallest float32 is 2^-133, as is the smallest bfloat16, so that no number is too small for its parts (as they are, numbers below 2^-110 would
// lose digits); sums of products are divided by 2^32 at the end.  The first two are the
// nearest, so that the products left out (of a second and a third part, and of two third parts) have either sign and are
// below 2^-24 of the product; with the second part cut off instead they have the product's sign where a row meets itself, and reach
// 2^-23.  The differences are exact.  Additions and masks and not v_cvt_pk_bf16_f32 and v_dot2c_f32_bf16, which do it in half the
// instructions: beside a matrix instruction of 17 clocks two of the former are free, but one of the latter makes it 35.
template <typename T>
struct Parts {
  static constexpr int P = sizeof(T) == 4 ? 3 : 1;
  u32x4 p[P];
};
__device__ __forceinline__ uint32_t upper_halves(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
// Half h of the eight: four numbers.
__device__ __forceinline__ void half_parts_of(Parts<float>& o, const Eight<float>& e, int h) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float a = e.v[h][2 * i] * GP_UP, b = e.v[h][2 * i + 1] * GP_UP;
    const uint32_t a0 = __float_as_uint(a) + 0x8000u, b0 = __float_as_uint(b) + 0x8000u;
    const float ra = a - __uint_as_float(a0 & 0xffff0000u), rb = b - __uint_as_float(b0 & 0xffff0000u);
    const uint32_t a1 = __float_as_uint(ra) + 0x8000u, b1 = __float_as_uint(rb) + 0x8000u;
    const float a2 = ra - __uint_as_float(a1 & 0xffff0000u), b2 = rb - __uint_as_float(b1 & 0xffff0000u);
    o.p[0][2 * h + i] = upper_halves(a0, b0);
    o.p[1][2 * h + i] = upper_halves(a1, b1);
    o.p[2][2 * h + i] = upper_halves(__float_as_uint(a2), __float_as_uint(b2));
  }
}
__device__ __forceinline__ void half_parts_of(Parts<bf16_t>& o, const Eight<bf16_t>& e, int h) {
  o.p[0][2 * h] = e.v[h].x;
  o.p[0][2 * h + 1] = e.v[h].y;
}
template <typename T>
__device__ __forceinline__ void parts_of(Parts<T>& o, const Eight<T>& e) {
  half_parts_of(o, e, 0);
  half_parts_of(o, e, 1);
}

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 w, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, w), c, 0, 0, 0);
}

// A slab's sum, which then joins the others'.  float32: the six products of parts that reach its 24 bits, small ones first.
__device__ __forceinline__ f32x4 slab(const Parts<float>& a, const Parts<float>& w) {
  f32x4 t = mfma(a.p[2], w.p[0], f32x4{0.f, 0.f, 0.f, 0.f});
  t = mfma(a.p[0], w.p[2], t);
  t = mfma(a.p[1], w.p[1], t);
  t = mfma(a.p[1], w.p[0], t);
  t = mfma(a.p[0], w.p[1], t);
  return mfma(a.p[0], w.p[0], t);
}
__device__ __forceinline__ f32x4 slab(const Parts<bf16_t>& a, const Parts<bf16_t>& w) { return mfma(a.p[0], w.p[0], f32x4{0.f, 0.f, 0.f, 0.f}); }

// A sum of products of numbers times GP_UP, of the numbers themselves.
template <typename T>
__device__ __forceinline__ float sized(float v) { return sizeof(T) == 4 ? v * (1.f / GP_UP / GP_UP) : v; }

// A result that is not finite is formed again from the numbers themselves: an infinity has no parts (its remainder is no
// number), nor have numbers from 2^112 on, and sums from 2^96 on are infinite times 2^32.  A number by itself, as
// it should never be needed; the blocks' sums are added as ever.
__device__ __forceinline__ bool is_finite(float v) { return fabsf(v) <= 3.402823466e38f; }
__device__ __attribute__((noinline)) float formed_again(const float* a, const float* w, int K) {
  float total = 0.f;
  for (int k = 0; k < K && total == total; k += GP_BLOCK) {
    float sum = 0.f;
    const int end = min(K, k + GP_BLOCK);
    for (int i = k; i < end && sum == sum; ++i) sum = fmaf(a[i], w[i], sum);
    total += sum;
  }
  return total;
}

// Up to 16 * MT rows: blockIdx.x 16 weight rows, blockIdx.y the product of the batch, blockIdx.z a share of
// the blocks of k.  VEC: rows may be read four numbers at a time.  A block of k is one wavefront's; SPREAD: of
// `parts` wavefronts, an equal range of its slabs each, whose sums meet in LDS one by one and are added in the order of k, the order
// of a running sum.  STAGED: the rows' parts are made once for all wavefronts and lie in LDS.
#define GP_SLABS (GP_BLOCK / GP_SLAB)
__host__ __device__ constexpr int few_slots(bool spread) { return spread ? GP_SLABS : 1; }  // sums of a block in LDS
template <typename TA, typename TC, int MT, bool VEC, bool SPREAD, bool STAGED>
__global__ __launch_bounds__(64 * (SPREAD && MT <= 2 ? GP_FEW_MOST : GP_FEW_WAVES), 2) void gemm_plain_few_kernel(
    TC* __restrict__ C, int64_t ldc, const TA* __restrict__ A, int64_t lda, const TA* __restrict__ W,
    const void* __restrict__ bias, int b_is_f32, int M, int N, int K, int64_t batch_c, int64_t batch_a,
    int64_t batch_w, float* __restrict__ scratch, int parts) {
  C += blockIdx.y * batch_c;
  A += blockIdx.y * batch_a;
  W += blockIdx.y * batch_w;
  extern __shared__ f32x4 sums_lds[];  // [block][slot][MT][lane]; STAGED: behind it u32x4 [block][slab][part][row][eight]
  constexpr int SLOTS = few_slots(SPREAD), P = Parts<TA>::P;
  if (!SPREAD) parts = 1;
  const int waves = blockDim.x / PAE_WAVE, here = waves / parts;  // blocks side by side
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  const int place = wave / parts, part_slabs = GP_SLABS / parts, slab0 = (wave - place * parts) * part_slabs;
  const int lane = threadIdx.x % PAE_WAVE, r = lane % 16, kq = lane / 16;
  const int n0 = blockIdx.x * 16;
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  const int step = here * gridDim.z;
  u32x4* a_lds = (u32x4*)(sums_lds + here * SLOTS * MT * PAE_WAVE);
  // rows past the end are read as the last one and dropped
  const TA* w_row = W + (int64_t)min(n0 + r, N - 1) * K;
  const TA* a_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) a_row[i] = A + (int64_t)min(i * 16 + r, M - 1) * lda;
  constexpr int U = MT == 1 ? 2 : 1;  // slabs whose loads are on their way together, twice
  constexpr int TOTALS = (16 * MT * 16) / PAE_WAVE;
  float total[TOTALS];  // thread t: outputs t, t + threads, ...
#pragma unroll
  for (int i = 0; i < TOTALS; ++i) total[i] = 0.f;

  for (int first = 0; first < blocks; first += step) {  // the same trips for every wavefront
    const int round = first + blockIdx.z * here, block = round + place;
    int k = 0, end = 0;
    if (block < blocks) {
      k = block * GP_BLOCK + slab0 * GP_SLAB;
      end = min(K, k + part_slabs * GP_SLAB);
    }
    struct Batch {
      Eight<TA> w[U], a[U][STAGED ? 1 : MT];
    } b0, b1;
    constexpr int STEP = GP_SLAB * U;
    int batches = VEC ? max(0, end - k) / STEP : 0;
    auto fetch = [&](Batch& b, int at) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        load8(b.w[u], w_row, at + u * GP_SLAB, kq);
        if constexpr (!STAGED) {
#pragma unroll
          for (int i = 0; i < MT; ++i) load8(b.a[u][i], a_row[i], at + u * GP_SLAB, kq);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if (batches > 0) fetch(b0, k);
    if constexpr (STAGED) {
      const int k0 = round * GP_BLOCK, slabs = (min(K, k0 + here * GP_BLOCK) - k0 + GP_SLAB - 1) / GP_SLAB;
      for (int e = threadIdx.x; e < M * slabs * 4; e += blockDim.x) {
        const int row = e / (slabs * 4), slab = e / 4 - row * slabs, q = e % 4;
        Eight<TA> raw;
        load8_anyhow<VEC>(raw, A + (int64_t)row * lda, k0 + slab * GP_SLAB, q, K);
        cut(raw, k0 + slab * GP_SLAB, q, K);
        Parts<TA> made;
        parts_of(made, raw);
#pragma unroll
        for (int p = 0; p < P; ++p) a_lds[((slab * P + p) * M + row) * 4 + q] = made.p[p];
      }
      __syncthreads();
    }
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4* to = sums_lds + (place * SLOTS + slab0) * (MT * PAE_WAVE) + lane;
    const u32x4* staged = a_lds + (place * GP_SLABS + slab0) * (P * 4 * M) + min(r, M - 1) * 4 + kq;
    auto join = [&](const Parts<TA>& w, const Eight<TA>* a) {
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        Parts<TA> made;
        if constexpr (STAGED) {
#pragma unroll
          for (int p = 0; p < P; ++p) made.p[p] = staged[p * 4 * M];
        } else {
          parts_of(made, a[i]);
        }
        if constexpr (!SPREAD) acc[i] += slab(made, w);
        else to[i * PAE_WAVE] = f32x4{0.f, 0.f, 0.f, 0.f} + slab(made, w);
      }
      if (SPREAD) to += MT * PAE_WAVE;
      if (STAGED) staged += P * 4 * M;
    };
    if (batches > 0) {
      // two batches take turns; no load stands under a condition of its own
      auto multiply = [&](const Batch& b) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          Parts<TA> w;
          parts_of(w, b.w[u]);
          join(w, b.a[u]);
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      while (batches >= 3) {
        fetch(b1, k + STEP);
        multiply(b0);
        fetch(b0, k + 2 * STEP);
        multiply(b1);
        k += 2 * STEP;
        batches -= 2;
      }
      if (batches == 2) {
        fetch(b1, k + STEP);
        multiply(b0);
        multiply(b1);
      } else {
        multiply(b0);
      }
      k += batches * STEP;
    }
    for (; k < end; k += GP_SLAB) {
      Eight<TA> w_raw, a_raw[MT];
      load8_anyhow<VEC>(w_raw, w_row, k, kq, K);
      if constexpr (!STAGED) {
#pragma unroll
        for (int i = 0; i < MT; ++i) load8_anyhow<VEC>(a_raw[i], a_row[i], k, kq, K);
#pragma unroll
        for (int i = 0; i < MT; ++i) cut(a_raw[i], k, kq, K);
      }
      cut(w_raw, k, kq, K);
      Parts<TA> w;
      parts_of(w, w_raw);
      join(w, a_raw);
    }
    if constexpr (!SPREAD) {
      if (scratch) {  // this block's sums to memory; another kernel adds them up
        if (block < blocks && n0 + r < N) {
#pragma unroll
          for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int m = i * 16 + kq * 4 + e;
              if (m < M) scratch[((int64_t)block * M + m) * N + n0 + r] = acc[i][e];
            }
        }
        if (STAGED) __syncthreads();
        continue;
      }
      if (block < blocks) {
#pragma unroll
        for (int i = 0; i < MT; ++i) to[i * PAE_WAVE] = acc[i];
      }
    }
    __syncthreads();
    // output o of lane (o / 64 % 4, o % 16), element o / 16 % 4
    auto place_of = [&](int o) { return (o / 256 * PAE_WAVE + o / 64 % 4 * 16 + o % 16) * 4 + o / 16 % 4; };
    float* sums = (float*)sums_lds;
    const int there = min(here, blocks - round);
    if constexpr (SPREAD) {  // the blocks' sums, a thread an output; they take the place of the first slabs'
      for (int o = threadIdx.x; o < there * MT * 256; o += blockDim.x) {
        const int v = o / (MT * 256), left = K - (round + v) * GP_BLOCK;
        float* from = sums + v * (SLOTS * MT * 256) + place_of(o % (MT * 256));
        float slab_sum[GP_SLABS], sum = 0.f;
#pragma unroll
        for (int j = 0; j < GP_SLABS; ++j) slab_sum[j] = from[j * (MT * 256)];
#pragma unroll
        for (int j = 0; j < GP_SLABS; ++j) sum += j * GP_SLAB < left ? slab_sum[j] : 0.f;
        *from = sum;
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < TOTALS; ++i) {
      const int o = threadIdx.x + i * blockDim.x, m = o / 16, n = n0 + o % 16;
      if (o >= MT * 256) continue;
      const float* from = sums + place_of(o);
      for (int v = 0; v < there; ++v) {
        const float sum = from[v * (SLOTS * MT * 256)];
        if (!scratch) total[i] += sum;
        else if (m < M && n < N) scratch[((int64_t)(round + v) * M + m) * N + n] = sum;  // another kernel adds them up
      }
    }
    if (first + step < blocks) __syncthreads();
  }
  if (scratch) return;
#pragma unroll
  for (int i = 0; i < TOTALS; ++i) {
    const int o = threadIdx.x + i * blockDim.x, m = o / 16, n = n0 + o % 16;
    if (o < MT * 256 && m < M && n < N) {
      float v = sized<TA>(total[i]);
      if constexpr (P > 1) {
        if (!is_finite(v)) v = formed_again(A + m * lda, W + (int64_t)n * K, K);
      }
      if (bias) v += load_param(bias, b_is_f32, n);
      C[(int64_t)m * ldc + n] = from_f32<TC>(v);
    }
  }
}

// Tiles of BM rows of A by BN of W, WM x WN wavefronts.  blockIdx.x: the tiles, those of one column of tiles (the same weights)
// next to each other on one die; blockIdx.y: the product of the batch; blockIdx.z: a share of the blocks of k.
// What bounds it is the matrix cores' six instructions a slab of float32 and, not far behind, LDS, which takes in 192 bytes a row
// and slab and gives them to WN or WM wavefronts; a thread takes three eights a slab apart (34 instructions a half; one eight in
// tiles of 64 x 64) between its products.  A row of 32 numbers of one part, 64 bytes, lies in LDS as four eights, at places turned by the row so
// that the 16 rows that a wavefront reads an eight of fall into different banks.
template <typename TA, typename TC, int BM, int BN, int WM, int WN, bool VEC, bool SHARED>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_plain_tiles_kernel(
    TC* __restrict__ C, int64_t ldc, const TA* __restrict__ A, int64_t lda, const TA* __restrict__ W,
    const void* __restrict__ bias, int b_is_f32, int M, int N, int K, int64_t batch_c, int64_t batch_a,
    int64_t batch_w, float* __restrict__ scratch) {
  C += blockIdx.y * batch_c;
  A += blockIdx.y * batch_a;
  W += blockIdx.y * batch_w;
  constexpr int THREADS = 64 * WM * WN, P = Parts<TA>::P, MT = BM / WM / 16, NT = BN / WN / 16;
  constexpr int E = (BM + BN) * 4 / THREADS;  // eights that a thread brings
  static_assert((BM + BN) * 4 % THREADS == 0, "whole eights");
  extern __shared__ u32x4 parts_lds[];  // [2][P][BM + BN][4]
  const int tid = threadIdx.x, lane = tid % PAE_WAVE, r = lane % 16, kq = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / PAE_WAVE);
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles = gridDim.x;
  // workgroups i, i + 8, i + 16, ... run on one die: they take neighbouring tiles
  const int per = tiles / 8, rest = tiles % 8, die = blockIdx.x % 8;
  const int tile = die * per + min(die, rest) + blockIdx.x / 8;
  const int m_tile = (tile % tiles_m) * BM, n_tile = (tile / tiles_m) * BN;
  const int m0 = m_tile + wave / WN * (BM / WM), n0 = n_tile + wave % WN * (BN / WN);
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  const int share = (blocks + gridDim.z - 1) / gridDim.z;
  const int block0 = blockIdx.z * share, block1 = min(blocks, block0 + share);
  if (block0 >= block1) return;

  const TA* src[E];
  int dst[E];
#pragma unroll
  for (int u = 0; u < E; ++u) {
    const int c = tid + u * THREADS, row = c / 4;
    src[u] = row < BM ? A + (int64_t)min(m_tile + row, M - 1) * lda : W + (int64_t)min(n_tile + row - BM, N - 1) * K;
    dst[u] = row * 4 + ((c % 4) ^ ((row >> 1) & 3));
  }
  const int at = r * 4 + (kq ^ ((r >> 1) & 3));  // of the lane's eight within 16 rows
  const int a_at = wave / WN * (BM / WM) * 4 + at, w_at = (BM + wave % WN * (BN / WN)) * 4 + at;

  f32x4 acc[MT][NT], total[SHARED ? 1 : MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = total[SHARED ? 0 : i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  Eight<TA> raw[E];
  const int k_begin = block0 * GP_BLOCK;
  auto fetch = [&](int u, int k) { load8_anyhow<VEC>(raw[u], src[u], k, tid % 4, K); };
  auto parts_at = [&](int buf, int p) { return parts_lds + (buf * P + p) * ((BM + BN) * 4); };
  auto store = [&](const Parts<TA>& part, int u, int buf) {
#pragma unroll
    for (int p = 0; p < P; ++p) parts_at(buf, p)[dst[u]] = part.p[p];
  };
#pragma unroll
  for (int u = 0; u < E; ++u) fetch(u, k_begin);
#pragma unroll
  for (int u = 0; u < E; ++u) {
    Parts<TA> part;
    if (k_begin + GP_SLAB > K) cut(raw[u], k_begin, tid % 4, K);
    parts_of(part, raw[u]);
    store(part, u, 0);
    fetch(u, k_begin + GP_SLAB);
  }
  __syncthreads();
  int buf = 0;
  for (int block = block0; block < block1; ++block) {
    const int end = min(K, (block + 1) * GP_BLOCK);
    for (int k = block * GP_BLOCK; k < end; k += GP_SLAB) {
      // the products, and between them the parts of the next slab's numbers (behind the last slab: of what nobody reads)
      Parts<TA> a[2], w[NT], part;
      f32x4 sum[2][NT];
      auto read_a = [&](int i) {
#pragma unroll
        for (int p = 0; p < P; ++p) a[i % 2].p[p] = parts_at(buf, p)[a_at + i * 64];
      };
      read_a(0);
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int p = 0; p < P; ++p) w[j].p[p] = parts_at(buf, p)[w_at + j * 64];
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        if (i + 1 < MT) read_a(i + 1);
        constexpr int HALVES = 2 * E;
#pragma unroll
        for (int h = i * HALVES / MT; h < (i + 1) * HALVES / MT; ++h) {
          if (h % 2 == 0 && k + 2 * GP_SLAB > K) cut(raw[h / 2], k + GP_SLAB, tid % 4, K);
          half_parts_of(part, raw[h / 2], h % 2);
#pragma unroll
          for (int p = 0; p < P; ++p)  // here and not where the compiler would have it: in one piece behind the products
            asm volatile("" : "+v"(part.p[p][h % 2 * 2]), "+v"(part.p[p][h % 2 * 2 + 1]));
          if (h % 2) {
            store(part, h / 2, buf ^ 1);
            fetch(h / 2, k + 2 * GP_SLAB);
          }
        }
#pragma unroll
        for (int j = 0; j < NT; ++j) sum[i % 2][j] = slab(a[i % 2], w[j]);
        if (i > 0) {  // the sums before these, which are done by now
#pragma unroll
          for (int j = 0; j < NT; ++j) acc[i > 0 ? i - 1 : 0][j] += sum[(i + 1) % 2][j];
        }
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[MT - 1][j] += sum[(MT - 1) % 2][j];
      __syncthreads();
      buf ^= 1;
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (SHARED) {
          const int n = n0 + j * 16 + r, m = m0 + i * 16 + kq * 4;
          float* p = scratch + ((int64_t)block * M + m) * N + n;
#pragma unroll
          for (int e = 0; e < 4; ++e, p += N)
            if (m + e < M && n < N) *p = acc[i][j][e];
        } else {
          total[SHARED ? 0 : i][j] += acc[i][j];
        }
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  if (SHARED) return;
  bool whole = true;
#pragma unroll
  for (int j = 0; j < NT; ++j) {
    const int n = n0 + j * 16 + r;
    if (n >= N) continue;
    const float b = bias ? load_param(bias, b_is_f32, n) : 0.f;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + i * 16 + kq * 4 + e;
        if (m >= M) continue;
        float v = sized<TA>(total[SHARED ? 0 : i][j][e]);
        whole = whole && is_finite(v);
        if (bias) v += b;
        C[(int64_t)m * ldc + n] = from_f32<TC>(v);
      }
  }
  if constexpr (P > 1) {
    if (whole) return;
    for (int o = 0; o < MT * NT * 4; ++o) {  // the sums are gone from the registers: what was stored is looked at
      const int n = n0 + o % NT * 16 + r, m = m0 + o / (NT * 4) * 16 + kq * 4 + o / NT % 4;
      if (m >= M || n >= N || is_finite(C[(int64_t)m * ldc + n])) continue;
      float v = formed_again(A + m * lda, W + (int64_t)n * K, K);
      if (bias) v += load_param(bias, b_is_f32, n);
      C[(int64_t)m * ldc + n] = v;
    }
  }
}

// The block sums [blocks][M][N] added up in order.
template <typename TA, typename TC>
__global__ __launch_bounds__(256) void gemm_plain_sum_kernel(TC* __restrict__ C, int64_t ldc, const TA* __restrict__ A,
                                                             int64_t lda, const TA* __restrict__ W,
                                                             const float* __restrict__ scratch,
                                                             const void* __restrict__ bias, int b_is_f32, int M,
                                                             int N, int K) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  const int m = blockIdx.y;
  if (n >= N) return;
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  const int64_t stride = (int64_t)M * N;
  const float* p = scratch + (int64_t)m * N + n;
  float total = 0.f;
  int b = 0;
  for (; b + 8 <= blocks; b += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(b + u) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) total += v[u];
  }
  for (; b < blocks; ++b) total += p[b * stride];
  total = sized<TA>(total);
  if constexpr (Parts<TA>::P > 1) {
    if (!is_finite(total)) total = formed_again(A + m * lda, W + (int64_t)n * K, K);
  }
  if (bias) total += load_param(bias, b_is_f32, n);
  C[(int64_t)m * ldc + n] = from_f32<TC>(total);
}

// How a product of many rows is cut: into tiles of 128 x 256, which have the most products to a byte of LDS, or of 64 x 64, of which three
// workgroups a compute unit hide each other's waits, and over how many workgroups the blocks of k of a tile are shared.
//
// The least of the times (us) that the two shapes and every number of shares would take, from times of both at 18 sizes of weights (16 to 17,920
// features, 512 to 18,944 of k) by 20 row counts from 33 to 4,096 and up to eight numbers of shares, which this meets within 11 % (root mean
// square) and whose fastest it is on average 1 % behind: a large tile has a unit to itself and takes 36 a block of k, small ones 11.6 a
// block alone, 15.4 two to a unit and 20.5 three to a unit; where rows are read number by number 73 and 24, 43 and 63.  Shares cost the
// launch that adds their sums, and the sums a way to memory and back.  Large / small, each with its best number of shares: 65 x 17,920 x 1,536 54 / 64 us, 1,500 x 17,920 x 1,536 542 / 676, 300 x
// 17,920 x 1,536 137 / 145, 601 x 1,536 x 8,960 129 / 145, 4,096 x 1,536 x 8,960 717 / 853; 65 x 1,536 x 8,960 49 / 38, 1,024 x 896 x 4,864 123 / 85,
// 601 x 1,536 x 1,536 47 / 32, 65 x 64 x 1,536 42 / 14.
struct GpTiles {
  int rows, cols, splits;
};
static int64_t tiles_of(int M, int N, int rows, int cols) { return (int64_t)((M + rows - 1) / rows) * ((N + cols - 1) / cols); }
static GpTiles tiles_plan(int M, int N, int K, bool shared) {
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  const int64_t large = tiles_of(M, N, 128, 256), small = tiles_of(M, N, 64, 64);
  struct Cost {
    double large, small[4];
  };
  static const Cost by_fours = {35.9, {0.0, 11.6, 15.4, 20.5}}, one_by_one = {73.0, {0.0, 24.0, 43.0, 63.0}};
  const Cost& cost = K % 4 ? one_by_one : by_fours;
  GpTiles best = {64, 64, 1};
  double least = 1e30;
  for (int z = 1, last = 0; z <= (shared ? blocks : 1); ++z) {
    const int each = (blocks + z - 1) / z;  // blocks of a workgroup
    if (each == last) continue;             // no more shares than they take
    last = each;
    if (z > 1 && large * (z - 1) > 4 * GP_UNITS && small * (z - 1) > 6 * GP_UNITS) break;  // more rounds of both
    const double each_k = each * GP_BLOCK < K ? each : K / (double)GP_BLOCK;
    const double sums = z > 1 ? 1.9 + 8.0 * blocks * M * N / 7.6e6 : 0.0;
    const int64_t rest = (small * z) % (3 * GP_UNITS);
    const double by_large = 5.8 + (large * z + GP_UNITS - 1) / GP_UNITS * cost.large * each_k + sums;
    const double by_small = 0.7 + ((small * z) / (3 * GP_UNITS) * cost.small[3] + cost.small[(rest + GP_UNITS - 1) / GP_UNITS]) * each_k + sums;
    if (by_large < least) least = by_large, best = GpTiles{128, 256, z};
    if (by_small < least) least = by_small, best = GpTiles{64, 64, z};
  }
  return best;
}
// Over how many workgroups the blocks of k of one tile are shared.  A share costs its sums a way to memory and back and the launch that adds
// them (about 4 us), so that up to 32 rows a workgroup's wavefronts take up to GP_FEW_WAVES blocks side by side first.
// Few rows: a compute unit works through its workgroups in rounds, and shares pay where they leave fewer rounds of the whole
// k.  Measured without shares / with them: 3 rows of 11,008 by 128 sixteens of weight rows (2 rounds of a third) 36.1 / 30.1 us, of
// 16,384 by 192 (3 of a quarter) 50.0 / 44.3, of 8,192 by 192 (2 of a half) 27.0 / 28.6, of 11,008 by 256 (3 of a third) 44.8 / 49.3.
static int splits_of(int M, int N, int K) {
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  if (M <= 0 || blocks == 1) return 1;
  if (M <= GP_FEW_ROWS) {
    if (blocks <= GP_FEW_WAVES) return 1;
    const int64_t sixteens = (N + 15) / 16, shares = (blocks + GP_FEW_WAVES - 1) / GP_FEW_WAVES;
    const int64_t rounds = (sixteens + GP_UNITS - 1) / GP_UNITS, rounds_of_shares = (sixteens * shares + GP_UNITS - 1) / GP_UNITS;
    return rounds_of_shares < rounds * shares && shares <= 65535 ? (int)shares : 1;
  }
  return tiles_plan(M, N, K, true).splits;
}

// Rows and columns of C that one pass of launches makes.  A product with shared blocks of k keeps their sums, whatever the
// number of shares: up to GP_SCRATCH floats (128 MiB) at once, more rows or columns than that one after the other, the longer side of C
// cut into equal parts (all at once, a product of 2,000 x 512 x 18,944 would keep 152 MB; cut it takes 428 us instead of 380; one of
// 200 x 3,584 x 18,944 keeps 106 MB).  And a grid's threads along x are counted in 32 bits.
#define GP_SCRATCH (32 << 20)
struct GpPart {
  int rows, cols;
};
static GpPart part_of(int M, int N, int K, bool shared) {
  const int64_t blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  auto cut = [](int whole, int64_t most) {  // equal parts of at most `most`, in multiples of a tile
    const int64_t tiles = (whole + GP_TILE - 1) / GP_TILE, fit = most / GP_TILE > 0 ? most / GP_TILE : 1, parts = (tiles + fit - 1) / fit;
    return parts == 1 ? whole : (int)((tiles + parts - 1) / parts * GP_TILE);
  };
  GpPart part = {M, cut(N, 1 << 26)};
  if (shared && splits_of(M, N, K) > 1 && blocks * M * N > GP_SCRATCH) {
    if (N >= M) part.cols = cut(N, GP_SCRATCH / (blocks * M));
    else part.rows = cut(M, GP_SCRATCH / (blocks * N));
  }
  part.rows = cut(part.rows, (int64_t)0x7fffff / ((part.cols + GP_TILE - 1) / GP_TILE) * GP_TILE);
  return part;
}

// part_of, for who wants to look: part[0] rows by part[1] columns.
extern "C" void pae_gemm_plain_part(int M, int N, int K, int shared, int* part) {
  const GpPart p = part_of(M, N, K, shared != 0);
  part[0] = p.rows;
  part[1] = p.cols;
}

// Floats of scratch memory that pae_gemm_plain_shared is best called with (0: none).
extern "C" int64_t pae_gemm_plain_scratch(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || splits_of(M, N, K) == 1) return 0;
  const GpPart part = part_of(M, N, K, true);
  return (int64_t)((K + GP_BLOCK - 1) / GP_BLOCK) * part.rows * part.cols;
}

// How few rows are worked on.  What a wavefront does for a slab is mostly taking numbers apart (8.5 instructions a number, eight of W
// and eight of A for each lane), and small products leave most places for wavefronts empty.  So where a unit has room for it, a block's slabs are
// spread over up to 8 wavefronts, and up to 8 rows, of which a wavefront alone would take 16 apart, are taken apart once for all.
// Without either / spread / spread and staged, us: 3 x 512 x 512 7.5, 4.9, 4.6; 1 x 896 x 896 8.1, 6.2, 5.9; 1 x 1,536 x 1,536 8.5, 8.2, 6.9; 8
// rows 8.6, 8.9, 8.3.  Staged alone: 1 x 17,920 x 1,536 25.2 / 23.8, 3 x 1,536 x 8,960 24.4 / 22.1.
// The lines: more than two blocks side by side (three and four with staged rows, or where rows are read number by number and what
// counts is loads on their way: 1 x 1,537 x 1,538 18.0 / 12.9) are enough for the four SIMDs (16 x 1,536 x 1,536 9.2, spread 9.8; 16 x 896 x 4,864 15.1,
// 16.4); a thread of a workgroup stages four eights at most (8 x 9,728 x 896 13.0, staged 14.4; 6 x 3,584 x 3,584 14.6, staged 15.9); 128 of k are four
// slabs (1 x 1,536 x 64 3.6, staged 3.8, spread 4.2).  `here` blocks lie side by side in each of `groups` workgroups.
struct GpFew {
  int parts;  // wavefronts a block is spread over
  bool staged;
};
static GpFew few_of(int here, int mt, int M, int K, int64_t groups, bool three_parts, bool vec) {
  const int rounds = (int)(groups < 16 * GP_UNITS ? (groups + GP_UNITS - 1) / GP_UNITS : 16), side = 16 / here > 1 ? 16 / here : 1;
  const int fit = rounds < side ? rounds : side;  // workgroups that a unit holds side by side
  GpFew few = {1, false};
  const bool may_stage = three_parts && mt == 1 && M <= GP_STAGED_ROWS && K > 128;
  for (int staged = may_stage; staged >= 0; --staged) {
    int parts = 1;
    if (K > 128 && here <= (staged || !vec ? 4 : 2) && fit * here * (GP_SLABS * mt + (staged ? 3 * M : 0)) <= 160)
      while (parts < 8 && here * parts * 2 <= GP_FEW_MOST && fit * here * parts * 2 <= 16) parts *= 2;
    few = GpFew{parts, staged != 0};
    if (staged && M <= 4 * parts && fit * here * ((parts > 1 ? GP_SLABS : 1) + 3 * M) <= 160) break;
  }
  return few;
}

template <typename TA, typename TC, bool VEC>
static int launch_plain(void* C, int64_t ldc, int64_t batch_c, const void* A, int64_t lda, int64_t batch_a,
                        const void* W, int64_t batch_w, const void* bias, int b_is_f32, int M, int N, int K, int batch,
                        float* scratch, int splits, hipStream_t stream) {
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
#define GP_ARGS                                                                                                  \
  (TC*)C, ldc, (const TA*)A, lda, (const TA*)W, bias, b_is_f32, M, N, K, batch_c, batch_a, batch_w, scratch
  // Over 32 rows the tiles are faster (33 x 17,920 x 1,536 59 us against 48, 33 x 1,536 x 8,960 49 against 24, 33 x 1,536 x 1,536 16 against
  // 14.5), except that rows read number by number stay with `few` up to 64 where there is more than a block of k (64 x 1,537 x 2,049 42 us)
  if (M <= (VEC || blocks == 1 ? GP_FEW_ROWS : 2 * GP_FEW_ROWS)) {
    const int each = (blocks + splits - 1) / splits;
    const int here = each < GP_FEW_WAVES ? each : GP_FEW_WAVES;
    const dim3 grid((N + 15) / 16, batch, splits);
#define GP_FEW_KERNEL(MT, SPREAD, STAGED)                                                                                 \
  do {                                                                                                                    \
    auto kernel = gemm_plain_few_kernel<TA, TC, MT, VEC, SPREAD, STAGED>;                                                 \
    const int lds = here * (few_slots(SPREAD) * MT + (STAGED ? 3 * M : 0)) * 1024;                                        \
    if (lds > 65536) {                                                                                                    \
      const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
      PAE_REQUIRE(allowed == hipSuccess, "gemm: no %d bytes of LDS", lds);                                                \
    }                                                                                                                     \
    kernel<<<grid, here * few.parts * PAE_WAVE, lds, stream>>>(GP_ARGS, few.parts);                                       \
  } while (0)
#define GP_FEW(MT)                                                                                                        \
  do {                                                                                                                    \
    constexpr bool CAN = MT == 1 && Parts<TA>::P == 3;                                                                    \
    const GpFew few = few_of(here, MT, M, K, (int64_t)grid.x * batch * splits, Parts<TA>::P == 3, VEC);                        \
    if (few.parts > 1 && few.staged) GP_FEW_KERNEL(MT, true, CAN);                                                        \
    else if (few.parts > 1) GP_FEW_KERNEL(MT, true, false);                                                               \
    else if (few.staged) GP_FEW_KERNEL(MT, false, CAN);                                                                   \
    else GP_FEW_KERNEL(MT, false, false);                                                                                 \
  } while (0)
    if (M <= 16) GP_FEW(1);
    else if (VEC || M <= 32) GP_FEW(2);
    else if constexpr (!VEC) GP_FEW(4);
#undef GP_FEW
#undef GP_FEW_KERNEL
  } else {
    const GpTiles shape = tiles_plan(M, N, K, splits > 1);
    const dim3 grid((unsigned)tiles_of(M, N, shape.rows, shape.cols), batch, splits);
    constexpr int ROW = 2 * Parts<TA>::P * 64;  // bytes of LDS
#define GP_TILES(BM, BN, WM, WN, SHARED)                                                                                  \
  do {                                                                                                                    \
    auto kernel = gemm_plain_tiles_kernel<TA, TC, BM, BN, WM, WN, VEC, SHARED>;                                           \
    const hipError_t allowed =                                                                                            \
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (BM + BN) * ROW);            \
    PAE_REQUIRE(allowed == hipSuccess, "gemm: no %d bytes of LDS", (BM + BN) * ROW);                                      \
    kernel<<<grid, 64 * WM * WN, (BM + BN) * ROW, stream>>>(GP_ARGS);                                                     \
  } while (0)
    if (shape.rows == 128) {
      if (scratch) GP_TILES(128, 256, 1, 8, true);
      else GP_TILES(128, 256, 1, 8, false);
    } else {
      if (scratch) GP_TILES(64, 64, 2, 4, true);
      else GP_TILES(64, 64, 2, 4, false);
    }
#undef GP_TILES
  }
#undef GP_ARGS
  if (scratch) {
    const int bad = pae_check_launch("gemm_plain");
    if (bad) return bad;
    gemm_plain_sum_kernel<TA, TC><<<dim3((N + 255) / 256, M), 256, 0, stream>>>((TC*)C, ldc, (const TA*)A, lda, (const TA*)W, scratch,
                                                                                bias, b_is_f32, M, N, K);
  }
  return pae_check_launch("gemm_plain");
}

// in_dtype: operands; out_dtype: C.  Supported: f32->f32, bf16->bf16, bf16->f32.
// `batch` products at once (one per head, say): product b reads A + b batch_a and W + b batch_w and
// writes C + b batch_c, with the same leading dimensions; no bias then.  `scratch`: pae_gemm_plain_scratch floats for one product,
// whose k may then be shared over workgroups, or null.
extern "C" int pae_gemm_plain_shared(int in_dtype, int out_dtype, void* C, int64_t ldc, int64_t batch_c, const void* A,
                                     int64_t lda, int64_t batch_a, const void* W, int64_t batch_w, const void* bias,
                                     int b_is_f32, int M, int N, int K, int batch, float* scratch, hipStream_t stream) {
  PAE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  PAE_REQUIRE(batch >= 1 && batch <= 65535 && (batch == 1 || !bias), "gemm: %d products at once (1..65535, no bias)", batch);
  PAE_REQUIRE(lda >= K && ldc >= N, "gemm: leading dimensions lda=%lld ldc=%lld too small for K=%d N=%d",
              (long long)lda, (long long)ldc, K, N);
  PAE_REQUIRE(batch == 1 || !scratch, "gemm: shares of k go with one product at a time, not with %d", batch);
  if (M == 0) return 0;
  PAE_REQUIRE(M <= 65535 * 64, "gemm: M=%d exceeds the grid", M);
  PAE_REQUIRE((in_dtype == PAE_F32 && out_dtype == PAE_F32) || (in_dtype == PAE_BF16 && (out_dtype == PAE_BF16 || out_dtype == PAE_F32)),
              "gemm: unsupported dtype pair in=%d out=%d", in_dtype, out_dtype);
  // four numbers at a time: 16 bytes in float32, 8 in bfloat16
  const int elem = in_dtype == PAE_F32 ? 4 : 2, out_elem = out_dtype == PAE_F32 ? 4 : 2;
  const bool vec = K % 4 == 0 && lda % 4 == 0 && (batch == 1 || (batch_a % 4 == 0 && batch_w % 4 == 0)) &&
                   (uintptr_t)A % (4 * elem) == 0 && (uintptr_t)W % (4 * elem) == 0;
  const GpPart part = part_of(M, N, K, scratch != nullptr);
  for (int64_t n0 = 0; n0 < N; n0 += part.cols)
    for (int64_t m0 = 0; m0 < M; m0 += part.rows) {
      const int rows = (int)(M - m0 < part.rows ? M - m0 : part.rows), cols = (int)(N - n0 < part.cols ? N - n0 : part.cols);
      char* c = (char*)C + (m0 * ldc + n0) * out_elem;
      const char* a = (const char*)A + m0 * lda * elem;
      const char* w = (const char*)W + n0 * K * elem;
      const char* b = bias ? (const char*)bias + n0 * (b_is_f32 ? 4 : 2) : nullptr;
      const int splits = scratch ? splits_of(rows, cols, K) : 1;
      float* sums = splits > 1 ? scratch : nullptr;
#define GP_GO(TA, TC)                                                                                                    \
  (vec ? launch_plain<TA, TC, true>(c, ldc, batch_c, a, lda, batch_a, w, batch_w, b, b_is_f32, rows, cols, K, batch, sums, \
                                    splits, stream)                                                                      \
       : launch_plain<TA, TC, false>(c, ldc, batch_c, a, lda, batch_a, w, batch_w, b, b_is_f32, rows, cols, K, batch,    \
                                     sums, splits, stream))
      const int rc = in_dtype == PAE_F32 ? GP_GO(float, float) : out_dtype == PAE_BF16 ? GP_GO(bf16_t, bf16_t) : GP_GO(bf16_t, float);
#undef GP_GO
      if (rc) return rc;
    }
  return 0;
}

extern "C" int pae_gemm_plain_batched(int in_dtype, int out_dtype, void* C, int64_t ldc, int64_t batch_c, const void* A,
                                      int64_t lda, int64_t batch_a, const void* W, int64_t batch_w, const void* bias,
                                      int b_is_f32, int M, int N, int K, int batch, hipStream_t stream) {
  return pae_gemm_plain_shared(in_dtype, out_dtype, C, ldc, batch_c, A, lda, batch_a, W, batch_w, bias, b_is_f32, M, N, K,
                               batch, nullptr, stream);
}
