// The delta rule and gated linear attention over a step of single tokens, in one launch: see recurrent_tokens.hip.
#pragma once
#include "common.h"

struct TokensStep {
  const void* proj;  // rows of the activations' type: [q: G heads of D | k: G heads of D | v: H heads of V]
  int64_t row_stride;
  const int4* runs;  // (first row, rows, tokens before, 0) of every sequence
  const int* slots;
  float* state;      // [slot][H][V][D]
  int64_t state_slot_stride;
  int G, H, D, V;
  const void* decay_in;  // rows of H (delta, a decay a head) or H D numbers
  int64_t decay_stride;
  const void* gate;      // rows of H V numbers
  int64_t gate_stride;
  int gate_sigmoid;
  const void* norm_w;    // [V]
  int w_is_f32;
  float norm_eps;
  void* out;             // [rows][H V]
  // the delta rule
  const float* conv_w;   // [C][taps]
  float* conv_tail;      // [slot][taps - 1][C]
  int64_t tail_slot_stride;
  int taps;
  const float* a_log;
  const float* dt_bias;
  float unit_eps;
  const void* beta_in;
  int64_t beta_stride;
  // gated linear attention
  const void* decay_bias;
  int bias_is_f32;
  float inv_tau;
};

enum { TOKENS_DELTA, TOKENS_CHANNEL_DELTA, TOKENS_LINEAR };

// Whether a step goes in one launch, and that launch.
bool takes_tokens_step(int num_tokens, int num_seqs, int G, int H, int D, int V, const float* state, int64_t slot_stride);
void launch_tokens_step(int kind, int dtype, const TokensStep& p, int num_seqs, hipStream_t stream);

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float softplus_f(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ __forceinline__ float gla_log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// Sum over a group of L = 4, 8 or 16 neighbouring lanes, in every one of them.
template <int L>
__device__ __forceinline__ float group_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xF, 0xF, true));  // lanes (1, 0, 3, 2) of a quad
  v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x4E, 0xF, 0xF, true));  // lanes (2, 3, 0, 1)
  if (L >= 8) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x141, 0xF, 0xF, true));   // 8 lanes mirrored
  if (L >= 16) v += __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x140, 0xF, 0xF, true));  // 16 lanes mirrored
  return v;
}
