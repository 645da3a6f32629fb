// A row that is the sum of several rows in memory (branches' outputs in the activation type or float32, partial sums of split
// products, a bias that every row adds), for kernels with one workgroup of 256 a row, a thread owning four
// consecutive columns in every 1,024.
//
// On a few rows such a kernel's time is its trips to memory, one behind the other: a piece's type and number are known at
// run time only, and a load whose value is converted under a condition is waited for there.  So all pieces are
// asked for at once as raw bits, the weights with them, and converted and added when all are there.  Up to
// PIECES pieces and 4,096 columns; the general kernels take the rest.  Kernels are built for up to FEW pieces and for up to PIECES
// (MOST): room for all seven is registers, 156 to 172 of them at four trips, which many rows of few pieces then lack wavefronts for.
#pragma once
#include "common.h"

namespace row_pieces {

constexpr int PIECES = 7, FEW = 2;

struct Pieces {
  const void* ptr[PIECES];
  int64_t row_stride[PIECES];  // elements from a row to the next (0: one row that all add)
  float scale[PIECES];         // of the term that ends with this piece (the pieces of a term are added, then scaled) ...
  int ends[PIECES];            // ... if it does
  int is_f32[PIECES];
  int count;
};

// Fills `out` from terms of `parts` pieces each; false if they are too many.
inline bool flatten(Pieces& out, int terms, const void* const* ptr, const int* is_f32, const int* parts,
                    const int64_t* part_stride, const int64_t* row_stride, const float* scale) {
  out.count = 0;
  for (int k = 0; k < PIECES; ++k) {
    out.ptr[k] = nullptr;
    out.row_stride[k] = 0;
    out.scale[k] = 0.f;
    out.ends[k] = out.is_f32[k] = 0;
  }
  for (int j = 0; j < terms; ++j)
    for (int p = 0; p < parts[j]; ++p) {
      if (out.count == PIECES) return false;
      const int k = out.count++;
      out.ptr[k] = is_f32[j] ? (const void*)((const float*)ptr[j] + p * part_stride[j]) : ptr[j];
      out.row_stride[k] = row_stride[j];
      out.is_f32[k] = is_f32[j];
      out.ends[k] = p + 1 == parts[j];
      out.scale[k] = scale[j];
    }
  return true;
}

// Four numbers as they lie in memory: float32, or bfloat16 in the first two words.
__device__ __forceinline__ uint4 ask(const void* p, int64_t at, bool f32) {
  if (f32) return *reinterpret_cast<const uint4*>((const float*)p + at);
  const uint2 v = *reinterpret_cast<const uint2*>((const bf16_t*)p + at);
  return make_uint4(v.x, v.y, 0, 0);
}

__device__ __forceinline__ void numbers(const uint4 raw, bool f32, float (&v)[4]) {
  v[0] = __uint_as_float(f32 ? raw.x : raw.x << 16);
  v[1] = __uint_as_float(f32 ? raw.y : raw.x & 0xffff0000u);
  v[2] = __uint_as_float(f32 ? raw.z : raw.y << 16);
  v[3] = __uint_as_float(f32 ? raw.w : raw.y & 0xffff0000u);
}

__device__ __forceinline__ void put4(float* p, const float (&v)[4]) { *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ void put4(bf16_t* p, const float (&v)[4]) {
  bf16_t h[4] = {__float2bfloat16(v[0]), __float2bfloat16(v[1]), __float2bfloat16(v[2]), __float2bfloat16(v[3])};
  *reinterpret_cast<uint2*>(p) = *reinterpret_cast<const uint2*>(h);
}

// The pieces of a row's columns i .. i + 3 as raw bits.  T: the activation type.
template <typename T, int MOST>
__device__ __forceinline__ void ask_all(const Pieces& pieces, int64_t row, int i, uint4 (&raw)[MOST]) {
#pragma unroll
  for (int k = 0; k < MOST; ++k)
    if (k < pieces.count) raw[k] = ask(pieces.ptr[k], row * pieces.row_stride[k] + i, sizeof(T) == 4 || pieces.is_f32[k]);
}

// sum[e] += scale_j * (the pieces of term j, added in order), terms in order.
template <typename T, int MOST>
__device__ __forceinline__ void add_all(const Pieces& pieces, const uint4 (&raw)[MOST], float (&sum)[4]) {
  float term[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < MOST; ++k)
    if (k < pieces.count) {
      float v[4];
      numbers(raw[k], sizeof(T) == 4 || pieces.is_f32[k], v);
#pragma unroll
      for (int e = 0; e < 4; ++e) term[e] += v[e];
      if (pieces.ends[k]) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          sum[e] += pieces.scale[k] * term[e];
          term[e] = 0.f;
        }
      }
    }
}

}  // namespace row_pieces
