// C[M, N] = A[M, K] * W[N, K]^T for up to 16 rows of A: the products of decode steps, which are bound by reading W once from HBM.
//
// What bounds them, and the layout that follows.  Memory gives its rate to loads of whole lines: a load instruction here reads 256
// contiguous bytes of each of four weight rows, 16 bytes a lane (16 rows by 64 bytes, which is the matrix instruction's own shape,
// reads 55 MB in 12.9 us, this in 10.5).  Such a fragment is multiplied as it comes, without a lane changing places: to the
// instruction (16 x 16 x 32) it is a tile of 16 "rows", each one of the four weight rows by one of four parts of the step's k
// (part p holds the 16-byte pieces p, p + 4, p + 8, p + 12), and A's fragment is laid out likewise, four rows by four parts.  Of the
// 16 x 16 products only those of equal parts mean something, a quarter; the instruction has the time (up to 16 rows take four of
// them a kilobyte of weights, of the 26 that fit), and a lane finds the four parts of its (weight row, row of A) in its quad.
//
// A workgroup takes 4 R weight rows (16, or 8 where few weight rows would leave compute units idle: what one unit takes in, about
// 30 KB a microsecond, bounds a product of few rows) and all of k: four wavefronts take its 128-wide steps in turn, or, with few
// weight rows, two times four wavefronts half of k each.  Sums are added part by part, then wavefront by wavefront, then range by
// range: an order that depends on N and K alone, so that a row's sums are the same bits whatever it is batched with.
//
// In a recorded graph, weights from HBM, microseconds at 1 / 8 / 16 rows, before (a kernel that loaded 16 rows by 64 bytes and moved
// every fragment to the instruction's order through LDS) and now:
//   0.5B gate/up with the gate    7.0 /  7.2 /  9.0    6.5 /  6.9 /  7.9      0.5B down      6.8 /  7.0 /  7.2    4.9 /  5.9 /  7.2
//   1.5B gate/up                 13.7 / 15.5 / 18.1   12.1 / 13.1 / 14.6      1.5B down     10.1 / 10.8 / 11.8    7.6 /  9.1 / 11.3
//   1.5B QKV                      5.8 /  6.1 /  6.8    5.0 /  5.3 /  5.9      1.5B O         4.7 /  5.0 /  5.7    3.7 /  4.0 /  4.7
//   3B gate/up                   20.8 / 22.9 / 24.6   17.9 / 20.4 / 23.2      3B QKV         6.6 /  7.0 /  7.6    6.0 /  6.6 /  7.4
//   7B gate/up                   52.2 / 59.2 / 64.2   48.2 / 49.8 / 60.5      7B down       33.5 / 39.0 / 44.8   26.1 / 27.0 / 32.4
//   14B gate/up                  57.9 / 69.2 / 78.1   50.8 / 53.0 / 69.0      72B gate/up    181 /  198 /  230    163 /  172 /  196
// (55 MB, the 1.5B gate/up's weights, are read in 10.9 us by a kernel that does nothing else.  At 16 rows the fragments of A are as many
// as the weights', which is what is left there.)
#pragma once
#include "common.h"
#include "api.h"
#include "gemm_rows.h"

#include <type_traits>

// R: fragments of four weight rows a wavefront (R = 2: half of a tile of 16); MG: groups of four rows of A; NW: wavefronts, four to a
// k range; U: steps asked for together.  Two batches of U steps take turns; ONE: a wavefront has at most U steps, all asked for at once.
// Wavefronts a SIMD are asked for where the compiler would give sums registers twice over (16 rows: 196, two wavefronts, instead of 136 to 160;
// at 16 rows 7B gate/up 68.3 -> 60.5 us, 0.5B 9.4 -> 7.9, 72B 218 -> 197).
template <int R, int MG, int EPI, int NW, int U, bool ONE>
__global__ __launch_bounds__(64 * NW, NW > 4 ? NW / 4 : U == 4 ? 2 : MG == 4 || (ONE && MG >= 2) ? 3 : 1) void gemm_rows_kernel(RowsProduct p, int k_per_range) {
  static_assert((R == 4 || R == 2) && (NW == 4 || NW == 8 || NW == 16), "a tile of 16 weight rows or half of one; one range, two or four");
  constexpr bool PAIRS = EPI == EPI_SWIGLU || EPI == EPI_ROPE;  // the epilogue joins row r of a tile with row r + 8
  constexpr bool AHEAD = EPI == EPI_RESIDUAL || EPI == EPI_ROPE;
  __shared__ float s_part[NW][R * MG][16];
  __shared__ float s_scale[16];
  int M = p.M;
  // Rows of A shared out: this workgroup's 4 MG.  (Only float32 sums are asked for so.  The residual's and the rotation's arguments are then fetched with
  // the others at the start and not, one trip more, behind the products: 1.5B O at 1 row 3.9 -> 3.7 us; the gate's kernel is better off without, 0.5B at
  // 8 rows 6.9 -> 6.7.)
  if ((AHEAD || EPI == EPI_F32) && gridDim.z > 1) {
    const int m0 = blockIdx.z * 4 * MG;
    p.A += (int64_t)m0 * p.lda;
    p.out = EPI == EPI_ROPE ? (void*)((bf16_t*)p.out + (int64_t)m0 * p.ldc) : (void*)((float*)p.out + (int64_t)m0 * p.ldc);
    M = min(4 * MG, M - m0);
    if (p.norm.row_stats) p.norm.row_stats += (int64_t)m0 * p.norm.row_stat_tiles;
    if (EPI == EPI_RESIDUAL) {
      p.norm.next_rows += (int64_t)m0 * p.norm.ld_next;
      p.norm.next_stats += (int64_t)m0 * p.norm.next_stat_tiles;
    }
    if (EPI == EPI_ROPE) {
      p.rope.positions += m0;
      if (p.rope.tok_seq) p.rope.tok_seq += m0;
      if (p.rope.cos_sin) p.rope.cos_sin += (int64_t)m0 * p.rope.rot;
    }
  }
  const int N = p.N, K = p.K;
  const int tid = threadIdx.x, lane = tid % PAE_WAVE, wave = tid / PAE_WAVE;
  const int tile = R == 4 ? blockIdx.x : blockIdx.x / 2, half = R == 4 ? 0 : blockIdx.x % 2;
  const int row = piece_row(lane), piece = piece_of(lane);
  // place in its tile of row `row` of fragment r
  auto place = [&](int r) { return R == 4 ? 4 * r + row : PAIRS ? 8 * r + 4 * half + row : 8 * half + 4 * r + row; };
  const bf16_t* wrow[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    int n = 16 * tile + place(r);
    if (EPI == EPI_ROPE) {
      const int per_head = p.rope.hd / 16;
      n = tile / per_head * p.rope.hd + rope_feature(tile % per_head, place(r), p.rope.rot);
    }
    wrow[r] = p.W + (int64_t)(n < N ? n : N - 1) * K;  // rows past N are loaded from the last row and never stored
  }
  const bf16_t* arow[MG];
#pragma unroll
  for (int g = 0; g < MG; ++g) {
    const int m = 4 * g + row;
    arow[g] = p.A + (int64_t)(m < M ? m : M - 1) * p.lda;
  }
  const int k_lo = (NW > 4 ? wave / 4 : blockIdx.y) * k_per_range, k_hi = min(K, k_lo + k_per_range);
  f32x4 acc[R][MG];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int g = 0; g < MG; ++g) acc[r][g] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // Loads are unconditional, from clamped addresses (the compiler counts the loads in flight behind the one it waits for, and where one
  // may or may not have been issued it waits for all); a lane past the end of the range zeroes its weights, and, where a wavefront's last batch may
  // hold whole steps behind it, its numbers of A (zero times an infinite one would be no number).
  constexpr int KW = 128 * 4, STEP = KW * U;
  const bf16x8 zero = {};
  struct Batch {
    bf16x8 wf[U][R], af[U][MG];
  };
  auto load = [&](Batch& b, int kb) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = kb + KW * u + 8 * piece;
      const int kc = k < K - 8 ? k : K - 8;
#pragma unroll
      for (int r = 0; r < R; ++r) b.wf[u][r] = *reinterpret_cast<const bf16x8*>(wrow[r] + kc);
#pragma unroll
      for (int g = 0; g < MG; ++g) b.af[u][g] = *reinterpret_cast<const bf16x8*>(arow[g] + kc);
    }
  };
  auto multiply = [&](const Batch& b, int kb, auto last) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = kb + KW * u + 8 * piece < k_hi;  // K and the bounds are multiples of 8: a lane's eight numbers are all in or all out
      bf16x8 a[MG];
#pragma unroll
      for (int g = 0; g < MG; ++g) a[g] = in || U == 1 || !decltype(last)::value ? b.af[u][g] : zero;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const bf16x8 w = in ? b.wf[u][r] : zero;
#pragma unroll
        for (int g = 0; g < MG; ++g) acc[r][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a[g], acc[r][g], 0, 0, 0);
      }
    }
  };
  const std::false_type inside;
  const std::true_type last;
  int kb = k_lo + 128 * (wave % 4);  // the same in every lane of a wavefront: the branches on it are uniform
  // what the epilogue reads beside the sums, and the rows' shares of the sums of squares, are asked for before the first batch is waited for
  EpilogueAhead<1> ahead;
  const int g4 = lane / 16;
  const bool live = R == 4 || (PAIRS ? g4 % 2 : g4 / 2) == half;  // this lane's four weight rows are the workgroup's
  Batch b0;
  if (AHEAD && wave == 0) ask_row<1, EPI>(ahead, M, p.rope);
  row_scales_to_lds<1>(s_scale, p.norm, M, K, tid, [&] { load(b0, kb); });
  if (AHEAD && wave == 0) ask_epilogue<1, EPI, false>(ahead, tile, p.out, p.ldc, M, N, p.rope, p.norm, live);
  if (ONE) {
    multiply(b0, kb, last);
  } else {
    Batch b1;
    int batches = kb < k_hi ? (k_hi - kb + STEP - 1) / STEP : 0;  // of this wavefront
    while (batches >= 3) {
      load(b1, kb + STEP);
      multiply(b0, kb, inside);
      load(b0, kb + 2 * STEP);
      multiply(b1, kb + STEP, inside);
      kb += 2 * STEP;
      batches -= 2;
    }
    if (batches == 2) {
      load(b1, kb + STEP);
      multiply(b0, kb, inside);
      multiply(b1, kb + STEP, last);
    } else if (batches == 1) {
      multiply(b0, kb, last);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int g = 0; g < MG; ++g) {
      const float sum = sum_of_parts(acc[r][g]);
      if (lane % 4 == 0) s_part[wave][r * MG + g][lane / 4] = sum;  // [weight row of the four][row of the four]
    }
  __syncthreads();
  if (wave > 0) return;

  // lane (m = lane % 16, g4): the sums of weight rows 4 g4 + i of the tile with row m of A, as the epilogues want them
  const int m = lane % 16, frag = R == 4 ? g4 : PAIRS ? g4 / 2 : g4 % 2;
  const int group = m / 4 < MG ? m / 4 : 0;  // (rows past the groups are not stored)
  f32x4 sums[1][1];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = 4 * i + m % 4;
    float total = 0.f;
#pragma unroll
    for (int range = 0; range < NW / 4; ++range) {
      float sum = s_part[4 * range][frag * MG + group][at];
#pragma unroll
      for (int w = 1; w < 4; ++w) sum += s_part[4 * range + w][frag * MG + group][at];
      total = range == 0 ? sum : total + sum;
    }
    sums[0][0][i] = total;
  }
  const float scale[1] = {s_scale[m]};
  if (EPI != EPI_F32 && NW == 4 && p.tickets.counters) {
    if (!add_up_k_ranges<1>(sums[0], blockIdx.z * gridDim.x + blockIdx.x, blockIdx.y, gridDim.y, p.tickets)) return;
  }
  skinny_epilogue<1, 1, EPI>(sums, tile, -1, p.out, p.ldc, p.bias, p.b_is_f32, M, N, blockIdx.y, p.part_stride, p.rope, p.norm, scale,
                             AHEAD ? &ahead : nullptr, live);
}

// One wavefront's steps of a range decide how its loads are asked for: two to four steps at once, more in batches of U that take turns.
// (Four at once, k of 1,537 to 2,048, us at 1 / 8 / 16 rows: 22,016 weight rows 18.2 / 21.1 / 25.5 -> 17.7 / 20.4 / 23.6, 2,560 6.5 / 7.2 / 8.3 -> 6.0 / 6.6 / 7.4;
// three, at 8 rows, 17,920 weight rows 14.0 -> 13.2.)
template <int R, int MG, int NW, int U, int EPI>
void launch_rows_as(const RowsProduct& p, int k_per_range, dim3 grid, hipStream_t stream) {
  const int steps = (k_per_range + 511) / 512;
  if (steps == 2) {
    gemm_rows_kernel<R, MG, EPI, NW, 2, true><<<grid, 64 * NW, 0, stream>>>(p, k_per_range);
    return;
  }
  if constexpr (NW == 4) {
    if (steps == 3 || steps == 4) {
      if (steps == 3) gemm_rows_kernel<R, MG, EPI, NW, 3, true><<<grid, 64 * NW, 0, stream>>>(p, k_per_range);
      else gemm_rows_kernel<R, MG, EPI, NW, 4, true><<<grid, 64 * NW, 0, stream>>>(p, k_per_range);
      return;
    }
  }
  gemm_rows_kernel<R, MG, EPI, NW, U, false><<<grid, 64 * NW, 0, stream>>>(p, k_per_range);
}

template <int R, int MG, int NW, int U>
void launch_rows_of(const RowsProduct& p, int k_per_range, dim3 grid, hipStream_t stream) {
  if constexpr (NW > 4) {  // ranges side by side: the residual products'
    launch_rows_as<R, MG, NW, U, EPI_RESIDUAL>(p, k_per_range, grid, stream);
  } else {
    switch (p.epilogue) {
      case EPI_BF16: launch_rows_as<R, MG, NW, U, EPI_BF16>(p, k_per_range, grid, stream); break;
      case EPI_F32: launch_rows_as<R, MG, NW, U, EPI_F32>(p, k_per_range, grid, stream); break;
      case EPI_SWIGLU: launch_rows_as<R, MG, NW, U, EPI_SWIGLU>(p, k_per_range, grid, stream); break;
      case EPI_ROPE: launch_rows_as<R, MG, NW, U, EPI_ROPE>(p, k_per_range, grid, stream); break;
      default: launch_rows_as<R, MG, NW, U, EPI_RESIDUAL>(p, k_per_range, grid, stream); break;
    }
  }
}
