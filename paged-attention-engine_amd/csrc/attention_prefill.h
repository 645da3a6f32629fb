// The operands of the prefill attention kernels (attention_mfma.hip, attention_prefill.hip).
#pragma once
#include "common.h"

#define PREFILL_RUN 128    // tokens of a run at most
#define RESCALE_STEP 8.0f  // how far (in units of log2) a score may pass its column's reference before the sums are rescaled

struct PrefillArgs {
  bf16_t* out;
  int64_t out_stride;
  const bf16_t* q;
  int64_t q_stride;
  const bf16_t* k;
  const bf16_t* v;
  const int* tiles;  // (table row of the sequence, first flat token, number of tokens <= PREFILL_RUN)
  int num_tiles;
  const int* positions;
  const int* block_tables;
  int max_blocks, nh, nkv;
  float scale_log2;
  int window;
  float cap_over_scale, scale_over_cap;
  const float* sinks;
  int chunked;
  const float* slopes;
  float inv_scale;
  const bf16_t* gate;
  int64_t gate_stride;
  const bf16_t* head_gate;
  int64_t head_gate_stride;
};

// attention_prefill.hip: the key and value widths it is built for, and the launch with `groups` (2 or 4) of 32 tokens a workgroup.
bool attn_prefill_shared_takes(int hd, int vd, int page_size);
int attn_prefill_shared(const PrefillArgs& p, int hd, int vd, bool biased, int groups, hipStream_t stream);
