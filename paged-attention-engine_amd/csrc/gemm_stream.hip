// C[M, N] = A[M, K] W[N, K]^T for 17 to 64 rows: both streamed through LDS by loads that pass no registers.
//
// One workgroup of eight wavefronts per (16 NT weight rows, range of k).  A stage is 64 of k: the rows of A and of W, 128 bytes
// each, laid out as in wide_gemm.h; STAGES - 1 stages are on their way while one is multiplied, and the wavefronts meet once a stage.
// A wavefront takes 32 of the 64 and 16 rows of A (with two column tiles half of the weight rows as well): every row of the stage
// is read from LDS once or twice, and the two halves of k are added through LDS at the end.
//
// What bounds it: the weights' way from memory, and what a compute unit takes in beside them, as every workgroup reads the rows of A of
// its range.  Fitted over 63 products by 17 shapes at 20 to 64 rows (15 % root mean square): 3.9 us, the weights at 6.5 TB/s, what a
// unit's workgroups take in at 88 KB a microsecond, and 0.7 + 0.5 us a range for ranges whose sums are added up by ticket.  The
// kernels before it (gemm_skinny.hip) load weights to registers, move them to the instruction's order through LDS, and read A
// again for every 32 weight rows, or hold the whole range of k in a wavefront.  Measured with weights from memory, in us, at 64 / 32 rows,
// before and now: 17,920 x 1,536 with the gate 21.5 -> 19.0 / as before, 37,888 x 3,584 79 -> 56 / 63 -> 52, 9,728 x 896 14.7 -> 9.5 /
// 12.0 -> 8.7; 1,536 x 8,960 into the residual 18.3 -> 14.9 / 16.2 -> 11.4, 3,584 x 18,944 49 -> 36 / 37 -> 31, 3,584 x 3,584 17.5 ->
// 14.0 / 15.0 -> 11.1; 4,608 x 3,584 18.9 -> 12.8 / 15.4 -> 11.4; heads of 151,936 x 1,536 125 -> 111 / 99 -> 93 (20 rows).
// Twice the stages on their way changes nothing (18.0 and 18.5 us), nor do twice the workgroups.
#include "common.h"
#include "api.h"
#include "gemm_stream.h"
#include "wide_gemm.h"

namespace {

using wide_gemm::load_to_lds;
using wide_gemm::meet;
typedef ::f32x4 f32x4;

constexpr int KEPT = 256;  // bytes for the rows' scales
constexpr int HALF_LDS = 163840 / 2, ALL_LDS = 163840;

template <int MT_, int NT_>
struct Shape {
  static constexpr int MT = MT_, NT = NT_;
  static constexpr int STAGE = 16 * (MT + NT) * 128, LOADS = STAGE / 1024, EACH = LOADS / 8, MORE = LOADS % 8;
  static constexpr int FIT = (HALF_LDS - KEPT) / STAGE, STAGES = FIT > 8 ? 8 : FIT >= 3 ? FIT : (ALL_LDS - KEPT) / STAGE;
  static constexpr int SIDES = MT == 2 ? 2 : 1, TILES = NT / SIDES, MINE = (TILES + 1) / 2;  // tiles of a wavefront: in the loop, and at the end
  static constexpr int SUMS = 8 * TILES * 1024, LDS = (STAGES * STAGE > SUMS ? STAGES * STAGE : SUMS) + KEPT;
  static_assert(NT % SIDES == 0 && STAGES >= 3, "whole tiles, and loads ahead");
};

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(N) : "memory");
}

template <int MT, int NT, int EPI>
__global__ __launch_bounds__(512, 4) void gemm_stream_kernel(StreamProduct p) {
  using S = Shape<MT, NT>;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  float* s_scale = reinterpret_cast<float*>(lds + S::LDS - KEPT);
  const int lane = threadIdx.x % PAE_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  const int col = lane % 16, g4 = lane / 16;
  const int half = wave / 4, c = wave % 4, mt = MT == 2 ? c % 2 : c, side = MT == 2 ? c / 2 : 0;
  const int n0 = blockIdx.x * 16 * NT;
  const int k_lo = blockIdx.y * p.k_per_split, stages = (min(p.K, k_lo + p.k_per_split) - k_lo) / 64;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);

  // load i of this wavefront brings the LDS rows 8 (wave + 8 i) .. of a stage: rows of A, then of W
  constexpr int MOST = S::EACH + (S::MORE ? 1 : 0);
  const bool more = S::MORE == 0 || wave < S::MORE;
  const char* base[MOST];
  uint32_t offset[MOST];
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const int row = 8 * min(wave + 8 * i, S::LOADS - 1) + lane / 8;
    if (wave + 8 * i < 2 * MT) {
      base[i] = reinterpret_cast<const char*>(p.a + k_lo);
      offset[i] = min(row, p.M - 1) * (uint32_t)(p.lda * 2);
    } else {
      int n = n0 + row - 16 * MT;
      if (EPI == EPI_ROPE) {
        const int per_head = p.rope.hd / 16;
        n = n / 16 / per_head * p.rope.hd + rope_feature(n / 16 % per_head, n % 16, p.rope.rot);
      }
      const int first = EPI == EPI_ROPE ? n0 / p.rope.hd * p.rope.hd : n0;  // (the rotation's order stays within a head)
      base[i] = reinterpret_cast<const char*>(p.w + (int64_t)first * p.K + k_lo);
      offset[i] = (uint32_t)(min(n, p.N - 1) - first) * (uint32_t)(p.K * 2);  // rows past N: the last one's, never stored
    }
    offset[i] += wide_gemm::piece_of(lane, row);
  }
  auto load = [&](int slot) {
#pragma unroll
    for (int i = 0; i < MOST; ++i) {
      if (i < S::EACH || more) load_to_lds(lds0 + slot * S::STAGE + (wave + 8 * i) * 1024, offset[i], base[i]);
      base[i] += 128;
    }
  };
  f32x4 acc[S::TILES];
#pragma unroll
  for (int x = 0; x < S::TILES; ++x) acc[x] = (f32x4){0.f, 0.f, 0.f, 0.f};
  row_scales_to_lds<MT>(s_scale, p.norm, p.M, p.K, threadIdx.x, [&] {
    for (int s = 0; s < min(S::STAGES - 1, stages); ++s) load(s);
  });
  const uint32_t piece = ((half * 4 + g4) ^ ((col >> 1) & 7)) * 16;
  const uint32_t a_at = (16 * mt + col) * 128 + piece, w_at = (16 * (MT + side * S::TILES) + col) * 128 + piece;
  int slot = 0;
  auto stage = [&](bool ahead) {
    meet();
    if (ahead) load(slot == 0 ? S::STAGES - 1 : slot - 1);
    const char* at = lds + slot * S::STAGE;
    if (mt < MT) {
      const bf16x8 a = *reinterpret_cast<const bf16x8*>(at + a_at);
      bf16x8 w[S::TILES];
#pragma unroll
      for (int x = 0; x < S::TILES; ++x) w[x] = *reinterpret_cast<const bf16x8*>(at + w_at + x * 2048);
#pragma unroll
      for (int x = 0; x < S::TILES; ++x) acc[x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[x], a, acc[x], 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // read whole before the next barrier, behind which it is written again
    slot = slot == S::STAGES - 1 ? 0 : slot + 1;
  };
  int left = stages;
  for (; left >= S::STAGES; --left) {  // the loads of the STAGES - 2 stages behind this one may be on their way
    if (more) wait_loads<(S::STAGES - 2) * MOST>();
    else wait_loads<(S::STAGES - 2) * S::EACH>();
    stage(true);
  }
  for (; left > 0; --left) {
    wait_loads<0>();
    stage(false);
  }
  __syncthreads();

  // the two halves of k: each wavefront adds its partner's sums to its own for its part of the tiles
  f32x4* sums = reinterpret_cast<f32x4*>(lds);
#pragma unroll
  for (int x = 0; x < S::TILES; ++x)
    if ((x < S::MINE) != (half == 0)) sums[(wave * S::TILES + x) * 64 + lane] = acc[x];
  __syncthreads();
  f32x4 mine[S::MINE];
#pragma unroll
  for (int x = 0; x < S::MINE; ++x) {
    const int y = x + S::MINE < S::TILES ? x + S::MINE : x;
    const f32x4 first = half == 0 ? acc[x] : sums[((wave ^ 4) * S::TILES + y) * 64 + lane];
    const f32x4 second = half == 0 ? sums[((wave ^ 4) * S::TILES + x) * 64 + lane] : acc[y];
    mine[x] = first + second;
  }
  if (mt >= MT || (half == 1 && S::TILES == 1)) return;
  if (EPI != EPI_F32 && p.tickets.counters &&
      !add_up_k_ranges<S::MINE>(mine, (blockIdx.x * 4 + c) * 2 + half, blockIdx.y, gridDim.y, p.tickets))
    return;

  const int m0 = 16 * mt, tile = blockIdx.x * NT + side * S::TILES + (half ? S::MINE : 0);
  void* out = (EPI == EPI_F32 || EPI == EPI_RESIDUAL) ? (void*)((float*)p.out + m0 * p.ldc) : (void*)((bf16_t*)p.out + m0 * p.ldc);
  if (EPI == EPI_RESIDUAL) {
    p.norm.next_rows += m0 * p.norm.ld_next;
    p.norm.next_stats += (int64_t)m0 * p.norm.next_stat_tiles;
  }
  if (EPI == EPI_ROPE) {
    p.rope.positions += m0;
    if (p.rope.tok_seq) p.rope.tok_seq += m0;
    if (p.rope.cos_sin) p.rope.cos_sin += (int64_t)m0 * p.rope.rot;
  }
  const float scale[1] = {s_scale[m0 + col]};
  auto finish = [&](auto count) {
    constexpr int COUNT = decltype(count)::value;
    if constexpr (COUNT > 0) {
      f32x4 done[COUNT][1];
#pragma unroll
      for (int x = 0; x < COUNT; ++x) done[x][0] = mine[x];
      skinny_epilogue<1, COUNT, EPI>(done, tile, -1, out, p.ldc, p.bias, p.b_is_f32, p.M - m0, p.N, blockIdx.y, p.part_stride, p.rope,
                                     p.norm, scale);
    }
  };
  if (S::MINE == S::TILES - S::MINE || half == 0) finish(wide_gemm::Number<S::MINE>());
  else finish(wide_gemm::Number<S::TILES - S::MINE>());
}

template <int MT, int NT, int EPI>
int launch(const StreamProduct& p, int splits, hipStream_t stream) {
  using S = Shape<MT, NT>;
  const hipError_t err = hipFuncSetAttribute((const void*)gemm_stream_kernel<MT, NT, EPI>, hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
  PAE_REQUIRE(err == hipSuccess, "gemm_stream: %d bytes of LDS refused: %s", S::LDS, hipGetErrorString(err));
  gemm_stream_kernel<MT, NT, EPI><<<dim3((p.N + 16 * NT - 1) / (16 * NT), splits), 512, S::LDS, stream>>>(p);
  return pae_check_launch("gemm_stream");
}

template <int MT, int NT>
int launch_epilogue(const StreamProduct& p, int splits, hipStream_t stream) {
  switch (p.epilogue) {
    case EPI_BF16: return launch<MT, NT, EPI_BF16>(p, splits, stream);
    case EPI_F32: return launch<MT, NT, EPI_F32>(p, splits, stream);
    case EPI_SWIGLU: return launch<MT, NT, EPI_SWIGLU>(p, splits, stream);
    case EPI_ROPE: return launch<MT, NT, EPI_ROPE>(p, splits, stream);
    case EPI_RESIDUAL: return launch<MT, NT, EPI_RESIDUAL>(p, splits, stream);
    default: return pae_fail("gemm_stream: unknown epilogue %d", p.epilogue);
  }
}

}  // namespace

// Microseconds, by the fit above, of workgroups of `nt` tiles.  (A unit holds two workgroups, of 10 tiles one: those only where one
// round of the chip takes them all; and ranges by ticket only where all workgroups are there at once.)
constexpr double TICKETS = 0.7, EACH_TICKET = 0.5;

static double stream_time(int M, int N, int K, int nt, int splits) {
  const int mt = (M + 15) / 16, range = ((K + splits - 1) / splits + 127) / 128 * 128;
  const int64_t groups = (int64_t)((N + 16 * nt - 1) / (16 * nt)) * splits;
  if ((mt == 2 && nt % 2) || (nt == 10 && groups > 256) || (splits > 1 && groups > 512)) return 1e30;
  const double rounds = groups <= 512 ? (groups + 255) / 256 : groups / 256.0;
  return 3.9 + rounds * (mt + nt) * 32.0 * range / 88e3 + (double)N * K * 2 / 6.5e6 + (splits > 1 ? TICKETS + EACH_TICKET * splits : 0.0);
}

static const int TILES[] = {2, 3, 4, 5, 6, 8, 10};

static int best_tiles(int M, int N, int K, int splits, double& least) {
  int best = 0;
  least = 1e29;
  for (int nt : TILES) {
    const double t = stream_time(M, N, K, nt, splits);
    if (t < least) least = t, best = nt;
  }
  return best;
}

// Which products go here.  Few weight rows in one range stay with the kernel that shares out the rows of A (2,048 x 1,536 at 64 rows
// 5.7 us, here 7.4; 896 x 4,864 9.1 and 10.1; 2,048 x 2,048 8.3 and 8.9), and some of many weight rows with that launcher's one workgroup a
// unit (`pae_one_workgroup_a_unit`).  Neither come here few and short weight rows, for which the start alone, about 4 us, is more than the other kernels take
// (with the norm that adds the ranges, at 20 / 48 rows: 640 x 3,072 7.6 / 7.7 us in two ranges there, 8.6 / 9.9 in three here, 1,024 x 4,096 8.8 / 10.7 and
// 9.5 / 11.0, 896 x 4,864 9.8 / 11.6 and 10.2 / 11.9; but 1,280 x 4,096 0.95 / 0.99 of it here, 1,024 x 6,144 0.95 / 0.97, 1,536 x 3,072 level).
static bool few_and_short(int N, int K) { return N <= 1280 && (int64_t)N * K < 4500000; }

int stream_tiles(int epilogue, const void* a, const void* w, int M, int N, int K, int64_t lda, int splits) {
  if (((uintptr_t)a | (uintptr_t)w) % 16 || M <= 16 || M > 64 || K % 64 || K > 1 << 20 || lda >= 1 << 24 || (splits > 1 && epilogue != EPI_F32 && N > 131072)) return 0;
  if ((splits == 1 && N <= 3072) || few_and_short(N, K)) return 0;
  if (splits == 1 && (epilogue == EPI_BF16 || epilogue == EPI_SWIGLU) && pae_one_workgroup_a_unit(M, N, K)) return 0;
  double least;
  return best_tiles(M, N, K, splits, least);
}

// k ranges for a product of 17 to 64 rows that this kernel takes, 0 for one that it does not.
extern "C" int pae_stream_ranges(int M, int N, int K) {
  if (M <= 16 || M > 64 || K % 64 || K > 1 << 20 || few_and_short(N, K)) return 0;
  int best = 0;
  double least = 1e29;
  for (int splits = N <= 3072 ? 2 : 1; splits <= 8 && (splits == 1 || K / splits >= 384); ++splits) {
    const int range = ((K + splits - 1) / splits + 127) / 128 * 128;
    if ((int64_t)range * (splits - 1) >= K) continue;
    double t;
    if (best_tiles(M, N, K, splits, t) && t < least) least = t, best = splits;
  }
  return best;
}

// The same for partial sums that the kernel behind adds, where one range would be taken: a range costs less there, 0.2 us and its sums' way to memory
// and back at 4.5 TB/s (with the norm, one range and these: 32 rows, 8,192 x 4,096 26.2 and 21.8 us, 4,096 x 2,048 12.6 and 10.8; of 416 sizes 25 change,
// 0.93 of the time on average, 1.09 at worst: 20 rows, 6,144 x 3,072 17.6 and 19.1).  Several ranges by ticket stay as they are: counted anew they would be
// 0.99 of the time on average and 1.10 at worst.
extern "C" int pae_stream_part_ranges(int M, int N, int K) {
  const int ticketed = pae_stream_ranges(M, N, K);
  if (ticketed != 1 || N > 10240 || K < 1536) return ticketed;  // (as far as was measured)
  int best = 1;
  double least = 1e30;
  for (int splits = 1; splits <= 8 && (splits == 1 || K / splits >= 384); ++splits) {
    const int range = ((K + splits - 1) / splits + 127) / 128 * 128;
    double t;
    if ((int64_t)range * (splits - 1) >= K || !best_tiles(M, N, K, splits, t)) continue;
    if (splits > 1) t += splits * (0.2 + 8.0 * M * N / 4.5e6) - TICKETS - EACH_TICKET * splits;
    if (t < least) least = t, best = splits;
  }
  return best;
}

// Whether a product of 17 to 64 rows, with whole sums, takes one range of k in workgroups of 5 to 8 wavefronts of 16 weight rows, one a compute unit and
// nearly all units busy (gemm_skinny.hip), although it could be streamed.  Over 12 counts of weight rows (17,408 to 32,768) by 7 of k (1,024 to
// 8,192) at 33 to 64 rows the choice is 0.965 of that kernel's time and 1.08 at worst, streaming all of them 0.985 and 1.18.
//   * up to 32 rows always: level (17,920 x 1,536 at 32 and 20 rows 16.1 and 15.8 us, streamed 16.6 and 16.0; 22,016 x 2,048 24.4 and 22.7, 24.3 and 23.0);
//   * up to 48 with seven wavefronts and more (48 rows, 27,648 x 5,120 52.8, streamed 56.4; 28,672 x 4,096 51.2 and 55.4; but 24,576 x 3,072, six, 28.7 and
//     27.2), or where streaming would cut k in three ranges, or in two from 8,192 on (48 rows, 21,504 x 5,120 44.1 and 47.1, 17,920 x 8,192 64.9 and
//     70.8; but 17,920 x 4,096 32.2 and 31.6);
//   * beyond that with seven and more and k from 4,096 on (64 rows, 28,672 x 4,096 52.9 and 56.2; 28,672 x 2,048 0.99 of it streamed).
extern "C" int pae_one_workgroup_a_unit(int M, int N, int K) {
  const int tiles = (N + 15) / 16, waves = (tiles + 255) / 256;
  if (M <= 16 || M > 64 || waves < 5 || waves > 8 || (tiles + waves - 1) / waves < 216) return 0;
  if (M <= 32) return 1;
  return waves >= 7 ? M <= 48 || K >= 4096 : M <= 48 && pae_stream_ranges(M, N, K) > (K >= 8192 ? 1 : 2);
}

int stream_ticket_slots(int M, int N) { return M > 16 && N <= 131072 ? (N + 31) / 32 * 8 : 0; }
int64_t stream_ticket_floats(int M, int N, int splits) {
  int64_t most = 0;
  if (M <= 16 || N > 131072) return 0;
  for (int nt : TILES) {
    const int mine = (M > 32 ? nt : nt / 2) / 2 + (M > 32 ? nt : nt / 2) % 2;  // tiles a wavefront ends with (two column tiles: half the tiles each)
    const int64_t floats = (int64_t)((N + 16 * nt - 1) / (16 * nt)) * 8 * mine * splits * 4 * PAE_WAVE;
    if (floats > most) most = floats;
  }
  return most;
}

int launch_stream(const StreamProduct& p, int tiles, int splits, hipStream_t stream) {
  const int mt = (p.M + 15) / 16;
#define CASE(MT, NT) \
  if (mt == MT && tiles == NT) return launch_epilogue<MT, NT>(p, splits, stream);
  CASE(2, 2) CASE(2, 4) CASE(2, 6) CASE(2, 8) CASE(2, 10)
  CASE(3, 2) CASE(3, 3) CASE(3, 4) CASE(3, 5) CASE(3, 6) CASE(3, 8) CASE(3, 10)
  CASE(4, 2) CASE(4, 3) CASE(4, 4) CASE(4, 5) CASE(4, 6) CASE(4, 8) CASE(4, 10)
#undef CASE
  return pae_fail("gemm_stream: %d rows by workgroups of %d tiles are not built", p.M, tiles);
}
