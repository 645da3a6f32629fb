// The inner loop of bfloat16 products with many rows on the matrix cores: a workgroup of four wavefronts holds 128 rows
// of A by 256 rows of W, 64 of k a stage, three stages in LDS (144 KB: one workgroup a compute unit).
//
// What bounds such a loop is the way into LDS.  A compute unit has about 40 lines of 128 bytes on their way at a time, 500
// clocks each on average (counters of the experts' products: 42 and 511), so it takes in about 11 bytes a clock whatever
// the loads look like, where 128 x 256 tiles at the matrix cores' full rate want 48; the matrix cores are
// busy a quarter of the time.  LDS itself gives a wavefront's 64 x 128 piece 12 KB for 32 matrix instructions, 96 of
// its 128 bytes a clock at the full rate.  Rows go from memory to LDS without passing registers (global_load_lds), a
// whole 128-byte line of a row at a time, two to three stages ahead, so that the lines' queue is never empty.  One barrier
// a stage: it stands between the two halves of a stage's products, behind the reads of the second half, so
// that the wavefronts meet while they have products left to issue, and the stage that the barrier frees is filled
// behind it.
//
// LDS layout: rows of 64 numbers, 128 bytes, no padding (the load writes 64 lanes x 16 bytes in a row).  The 16-byte
// pieces of row r lie at places piece ^ ((r / 2) % 8): 16 lanes that read the same piece of 16 rows meet all banks
// once.
#pragma once
#include "common.h"

namespace tile_gemm {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

constexpr int BM = 128, BN = 256, BK = 64, STAGES = 3;
constexpr int ROW_BYTES = BK * 2;
constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES;
constexpr int LDS_BYTES = STAGES * STAGE_BYTES;
constexpr int A_LOADS = BM / 8 / 4, W_LOADS = BN / 8 / 4;  // of 8 rows, that a wavefront makes a stage

// One load of 64 lanes x 16 bytes to LDS at `lds` (the same in every lane), lane by lane in a row.  It is not a load to the
// compiler: the waits for it are written below.  It sets m0, which cannot be named as changed (the compiler reserves it): kernels
// that use this must have nothing else that goes through m0, as the compiler's own loads to LDS, indexed register moves or messages do.
__device__ __forceinline__ void load_to_lds(uint32_t lds, uint32_t offset, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(offset), "s"(base) : "memory");
}

// What a lane brings: the byte offsets (from `a` and `w`, the same in every lane of a wavefront, which go forward with k)
// of its 16 bytes of each load.  Row of load j of wavefront v: (v * LOADS + j) * 8 + lane / 8.
struct Source {
  const char* a;
  const char* w;
  uint32_t a_off[A_LOADS], w_off[W_LOADS];
};

// The piece of 16 bytes that the lane brings of row `row`.
__device__ __forceinline__ uint32_t piece_of(int lane, int row) { return (uint32_t)((lane % 8) ^ ((row >> 1) & 7)) * 16; }

// Load `j` of a stage that this wavefront makes.
__device__ __forceinline__ void load_one(const Source& src, uint32_t stage, int wave, int j) {
  if (j < A_LOADS) load_to_lds(stage + (wave * A_LOADS + j) * 1024, src.a_off[j], src.a);
  else load_to_lds(stage + BM * ROW_BYTES + (wave * W_LOADS + j - A_LOADS) * 1024, src.w_off[j - A_LOADS], src.w);
}

template <int V>
struct Number {
  static constexpr int value = V;
};

// Keeps the sums where the matrix instructions add them: without it the compiler moves them between the register files.
__device__ __forceinline__ void pin(f32x4 (&acc)[4][8]) {
#pragma unroll
  for (int mt = 0; mt < 4; ++mt)
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) asm volatile("" : "+a"(acc[mt][nt]));
}

// acc[mt][nt] += W rows x A rows over `stages` * 64 of k: wavefront (wr, wc) holds A rows wr * 64 + 16 mt + lane % 16 (the
// columns of its results) by W rows w_row[nt] + 4 (lane / 16) + i.  `w_row`: first row in the tile of each of its eight
// groups of 16.  All four wavefronts call it together; `lds` is the workgroup's LDS_BYTES.
__device__ __forceinline__ void run(f32x4 (&acc)[4][8], char* lds, Source& src, int stages, const int (&w_row)[8]) {
  const int lane = threadIdx.x % PAE_WAVE, col = lane % 16, kg = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  const int wr = wave / 2;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  uint32_t a_at[2], w_at[2];  // of the lane's piece of both halves of a stage, within a group of 16 rows
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    a_at[h] = (wr * 64 + col) * ROW_BYTES + (((h * 4 + kg) ^ ((col >> 1) & 7)) * 16);
    w_at[h] = BM * ROW_BYTES + col * ROW_BYTES + (((h * 4 + kg) ^ ((col >> 1) & 7)) * 16);
  }
  bf16x8 a[2][4], w[2][8];
  auto read_a = [&](int h, const char* stage, int mt) { a[h][mt] = *reinterpret_cast<const bf16x8*>(stage + a_at[h] + mt * 16 * ROW_BYTES); };
  auto read_w = [&](int h, const char* stage, int nt) { w[h][nt] = *reinterpret_cast<const bf16x8*>(stage + w_at[h] + w_row[nt] * ROW_BYTES); };
  constexpr int LOADS = A_LOADS + W_LOADS;
  static_assert(LOADS == 12, "the waits below count a stage's loads");
  // Half h's products in eight groups of four; between them, two reads a group, the operands of the other half (READ)
  // from `from`, and one a group, six loads of a stage to come (PART 0: the first six, 1: the others, 2: none).  A
  // wavefront issues in order: twelve loads in a row, all four wavefronts', kept it from its products for 700 clocks.
  auto half = [&](auto h_, auto read_, auto part_, const char* from, uint32_t to) {
    constexpr int h = h_.value, READ = read_.value, PART = part_.value;
#pragma unroll
    for (int nt = 0; nt < 8; ++nt) {
      if (READ && nt < 2) {
        read_a(1 - h, from, 2 * nt);
        read_a(1 - h, from, 2 * nt + 1);
      }
      if (READ && nt >= 2 && nt < 6) {
        read_w(1 - h, from, 2 * nt - 4);
        read_w(1 - h, from, 2 * nt - 3);
      }
      if (PART < 2 && nt >= 1 && nt < 7) load_one(src, to, wave, PART * 6 + nt - 1);
#pragma unroll
      for (int mt = 0; mt < 4; ++mt)
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[h][nt], a[h][mt], acc[mt][nt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (PART == 1) {
      src.a += ROW_BYTES;
      src.w += ROW_BYTES;
    }
  };
  for (int s = 0; s < STAGES && s < stages; ++s) {
    for (int j = 0; j < LOADS; ++j) load_one(src, lds0 + s * STAGE_BYTES, wave, j);
    src.a += ROW_BYTES;
    src.w += ROW_BYTES;
  }
  // the first stage has arrived when at most the others' loads are on their way
  if (stages >= 3) asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
  else if (stages == 2) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 4; ++i) read_a(0, lds, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) read_w(0, lds, i);
  int at = 0, before = 0;  // the places of the stage and of the one before it
  // FIRST: behind the barrier begin to fill the stage's place again (stage s + 3); SECOND: go on with the place of the stage
  // before (stage s + 2, begun a stage ago).  IN_FLIGHT: loads that may still be on their way when the next stage is read.
  auto stage = [&](auto first, auto second, auto in_flight, auto next) {
    half(Number<0>(), Number<1>(), Number<second.value ? 1 : 2>(), lds + at * STAGE_BYTES, lds0 + before * STAGE_BYTES);
    const int other = at == STAGES - 1 ? 0 : at + 1;
    if (next.value) {
      // this wavefront has read the stage whole, and its loads of the next one have arrived
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(in_flight.value) : "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    half(Number<1>(), Number<next.value>(), Number<first.value ? 0 : 2>(), lds + other * STAGE_BYTES, lds0 + at * STAGE_BYTES);
    before = at;
    at = other;
  };
  const Number<0> no;
  const Number<1> yes;
  int left = stages;  // stages to come, this one included
  if (left > STAGES) {
    pin(acc);
    stage(yes, no, Number<12>(), yes);
    --left;
    for (; left > STAGES; --left) {
      pin(acc);
      stage(yes, yes, Number<12>(), yes);
    }
    stage(no, yes, Number<12>(), yes);
    --left;
  }
  for (; left > 2; --left) stage(no, no, Number<12>(), yes);
  if (left == 2) stage(no, no, Number<0>(), yes);
  stage(no, no, Number<0>(), no);
}

}  // namespace tile_gemm
