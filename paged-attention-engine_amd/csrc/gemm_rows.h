// Products of up to 16 rows of A by W streamed once from memory: what gemm_rows.hip takes from gemm_skinny.hip's launcher.
#pragma once
#include "skinny_device.h"

struct RowsProduct {
  int epilogue;
  void* out;
  int64_t ldc;
  const bf16_t* A;
  int64_t lda;
  const bf16_t* W;
  const void* bias;
  int b_is_f32, M, N, K;
  int splits;             // k ranges
  int64_t part_stride;
  SkinnyRope rope;
  SkinnyTickets tickets;
  SkinnyNorm norm;
};

// M <= 16, or (float32 sums) more: 16 or 8 rows a workgroup, shared out over grid.z.
int launch_rows(const RowsProduct& p, hipStream_t stream);

// The part of it that takes eight weight rows a workgroup: `side_by_side` k ranges in a workgroup (1, 2 or 4).
void launch_rows_halves(const RowsProduct& p, int side_by_side, int k_per_range, dim3 grid, hipStream_t stream);
