// Products of 17 to 64 rows with their operands streamed through LDS: see gemm_stream.hip.
#pragma once
#include "skinny_device.h"

struct StreamProduct {
  int epilogue;
  void* out;
  int64_t ldc;
  const bf16_t* a;
  int64_t lda;
  const bf16_t* w;
  const void* bias;
  int b_is_f32, M, N, K, k_per_split;
  int64_t part_stride;
  SkinnyRope rope;
  SkinnyTickets tickets;
  SkinnyNorm norm;
};

// Tiles of 16 weight rows a workgroup takes of this product in `splits` k ranges; 0: the other kernels take it.
int stream_tiles(int epilogue, const void* a, const void* w, int M, int N, int K, int64_t lda, int splits);
int launch_stream(const StreamProduct& p, int tiles, int splits, hipStream_t stream);
// Slots and floats of scratch that `splits` ticketed k ranges need (the most over the tiles a workgroup may take).
int stream_ticket_slots(int M, int N);
int64_t stream_ticket_floats(int M, int N, int splits);
