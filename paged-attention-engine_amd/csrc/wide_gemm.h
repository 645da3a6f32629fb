// The inner loops of bfloat16 products with more rows than the few-row kernels take: tiles of A rows by W rows, 64 of k a
// stage, rows brought from memory to LDS without passing registers (global_load_lds), products by 16 x 16 x 32 matrix
// instructions.  k ascends in steps of 32 for every sum in every tile shape, so a result is the same bits whichever
// shape a launch takes and whatever rows are beside it.
//
// What bounds such a loop on this chip is LDS.  It passes 128 bytes a clock, and per stage a tile of BM x BN writes BM + BN rows
// of 128 bytes and reads (PM + PN) rows in each of its wavefronts, which hold PM x PN; the matrix cores need BM * BN / 32 clocks:
//
//     tile, wavefronts, each one's part     LDS     matrix cores   measured, a compute unit alone / all of them
//     256 x 256, 8 of 128 x 64             2,048       2,048          2,290 / 2,600 clocks
//     128 x 256, 8 of  64 x 64             1,408       1,024
//     128 x 128, 4 of  64 x 64               768         512            920 / 1,100
//     128 x  96, 4 of  64 x 48               672         384            790 / 1,000
//      64 x  64, 4 of  32 x 32               384         128            480
//
// Lines come in at up to 100 KB a microsecond and compute unit where the die's L2 has them, twice what any of these takes.
// With one wavefront a SIMD the loads to LDS, which a wavefront issues in order, hold up its products, and from 128 x 64 on
// a wavefront's part needs the accumulation registers, between which and the others the compiler then moves the sums; a
// 256 x 256 tile of four wavefronts took 4,800 clocks a stage.  So the large tile has two wavefronts a SIMD that take turns: while
// one multiplies, the other reads its next operands and issues its loads.  What the whole chip takes on top of one compute
// unit's time is its clock (1.9 GHz under these loads).
//
// LDS layout: rows of 64 numbers, 128 bytes, no padding (a load writes 64 lanes x 16 bytes in a row).  The 16-byte pieces
// of row r lie at places piece ^ ((r / 2) % 8): 16 lanes that read the same piece of 16 rows meet all banks once.
//
// Which row of W a row of LDS holds is free, as every row is brought by its own address.  The rows of a wavefront's
// part are dealt so that its results leave in stores of 16 bytes a lane, 64 bytes in a row of the result: a lane ends with 8
// neighbours of 32 in two groups (X: groups of 16 W rows; a single group left over: 4 of 16), with 4 of 16 where the sums leave as
// float32, and for gated products, whose rows alternate in blocks of 8 of the gate and 8 of the other factor, with 2 X
// neighbouring gates and the same features' other factors.  Heads whose pairs of features are rotated are dealt likewise, 8 features
// and the 8 they are rotated with.
#pragma once
#include "common.h"

namespace wide_gemm {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int BK = 64, ROW_BYTES = BK * 2;

// One load of 64 lanes x 16 bytes to LDS at `lds` (the same in every lane), lane by lane in a row.  It is not a load to the
// compiler: the waits for it are written below.  It sets m0, which cannot be named as changed (the compiler reserves it): kernels
// that use this must have nothing else that goes through m0, as the compiler's own loads to LDS, indexed register moves or messages do.
__device__ __forceinline__ void load_to_lds(uint32_t lds, uint32_t offset, const void* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds), "v"(offset), "s"(base) : "memory");
}

template <int V>
struct Number {
  static constexpr int value = V;
};

// The piece of 16 bytes that a lane brings of the LDS row `row` of its tile.
__device__ __forceinline__ uint32_t piece_of(int lane, int row) { return (uint32_t)((lane % 8) ^ ((row >> 1) & 7)) * 16; }

enum { PLAIN, GATED, SUMS, ROTATED };  // what leaves: bfloat16, act(gate) * other in bfloat16, float32, heads with pairs of features rotated

// The W row, among the PN of a wavefront's part, that row `r` of its group `x` of 16 (of X) holds.
template <int MODE, int X>
__device__ __forceinline__ int dealt_row(int x, int r) {
  if (MODE == GATED || MODE == ROTATED) {
    const int feature = (r / 4) * (2 * X) + (x / 2) * 4 + r % 4;
    return (feature / 8) * 16 + feature % 8 + 8 * (x % 2);
  }
  if (MODE == SUMS || (X % 2 && x == X - 1)) return x * 16 + r;
  return (x / 2) * 32 + (r / 4) * 8 + (x % 2) * 4 + r % 4;
}

// The barrier alone, with nothing moved across it: unlike __syncthreads() it waits for no load on its way.
__device__ __forceinline__ void meet() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// A tile of BM x BN by WM x WN wavefronts, STAGES stages in LDS.  The wavefronts meet once a stage, between its two halves of
// 32 of k, behind the reads of the second half: the stage that is then free is filled again while they multiply.
template <int BM_, int BN_, int WM_, int WN_, int STAGES_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, STAGES = STAGES_;
  static constexpr int WAVES = WM * WN, PM = BM / WM, PN = BN / WN, MT = PM / 16, X = PN / 16;
  static constexpr int A_LOADS = BM / 8 / WAVES, W_LOADS = BN / 8 / WAVES, LOADS = A_LOADS + W_LOADS;
  static constexpr int STAGE_BYTES = (BM + BN) * ROW_BYTES, LDS_BYTES = STAGES * STAGE_BYTES;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0 && PM % 16 == 0 && PN % 16 == 0, "whole loads and groups");
  static_assert(STAGES >= 2 && STAGES <= 4, "the last stages' waits are written out");
  static_assert((STAGES - 1) * LOADS < 64, "loads on their way are counted in six bits");

  // What a lane brings: byte offsets from `a` and `w` (the same in every lane, they go forward with k) of its 16 bytes of
  // each load.  Load j of wavefront v is of the rows (v * A_LOADS + j) * 8 + lane / 8.
  struct Source {
    const char* a;
    const char* w;
    uint32_t a_off[A_LOADS], w_off[W_LOADS];
  };

  // acc[mt][x] += A rows wm * PM + 16 mt + lane % 16 by LDS rows wn * PN + 16 x + 4 (lane / 16) + i of W, over `stages` >= 1
  // stages.  All wavefronts call it together; `lds` has LDS_BYTES.
  static __device__ __forceinline__ void run(f32x4 (&acc)[MT][X], char* lds, Source& src, int stages) {
    const int lane = threadIdx.x % PAE_WAVE, col = lane % 16, kg = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
    const int wm = wave / WN, wn = wave % WN;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
    auto load_one = [&](uint32_t stage, int j) {
      if (j < A_LOADS) load_to_lds(lds0 + stage + (wave * A_LOADS + j) * 1024, src.a_off[j < A_LOADS ? j : 0], src.a);
      else load_to_lds(lds0 + stage + BM * ROW_BYTES + (wave * W_LOADS + j - A_LOADS) * 1024, src.w_off[j < A_LOADS ? 0 : j - A_LOADS], src.w);
    };
    uint32_t a_at[2], w_at[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t piece = ((s * 4 + kg) ^ ((col >> 1) & 7)) * 16;
      a_at[s] = (wm * PM + col) * ROW_BYTES + piece;
      w_at[s] = (BM + wn * PN + col) * ROW_BYTES + piece;
    }
    bf16x8 a[2][MT], w[2][X];
    auto read_a = [&](int s, uint32_t stage, int i) { a[s][i] = *reinterpret_cast<const bf16x8*>(lds + stage + a_at[s] + i * 16 * ROW_BYTES); };
    auto read_w = [&](int s, uint32_t stage, int x) { w[s][x] = *reinterpret_cast<const bf16x8*>(lds + stage + w_at[s] + x * 16 * ROW_BYTES); };
    // the products of half s; between them the other half's operands from `from` (READ) and a stage's loads to `to` (LOAD)
    auto half = [&](auto s_, auto read_, auto load_, uint32_t from, uint32_t to) {
      constexpr int s = s_.value, READ = read_.value, LOAD = load_.value;
#pragma unroll
      for (int x = 0; x < X; ++x) {
        if (READ) {
#pragma unroll
          for (int i = x * MT / X; i < (x + 1) * MT / X; ++i) read_a(1 - s, from, i);
          read_w(1 - s, from, x);
        }
        if (LOAD) {
#pragma unroll
          for (int j = x * LOADS / X; j < (x + 1) * LOADS / X; ++j) load_one(to, j);
        }
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i][x] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][x], a[s][i], acc[i][x], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (LOAD) {
        src.a += ROW_BYTES;
        src.w += ROW_BYTES;
      }
    };
    const int first = min(STAGES, stages);
    for (int s = 0; s < first; ++s) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j) load_one(s * STAGE_BYTES, j);
      src.a += ROW_BYTES;
      src.w += ROW_BYTES;
    }
    // the first stage has arrived when at most the others' loads are on their way
    if (stages >= STAGES) asm volatile("s_waitcnt vmcnt(%0)" : : "n"((STAGES - 1) * LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    meet();
#pragma unroll
    for (int i = 0; i < MT; ++i) read_a(0, 0, i);
#pragma unroll
    for (int x = 0; x < X; ++x) read_w(0, 0, x);
    uint32_t at = 0;
    // IN_FLIGHT: loads that may still be on their way when the next stage is read
    auto stage = [&](auto load, auto in_flight, auto next) {
      half(Number<0>(), Number<1>(), Number<0>(), at, 0);
      const uint32_t other = at == (STAGES - 1) * STAGE_BYTES ? 0 : at + STAGE_BYTES;
      if (next.value) {
        // this wavefront has read the stage whole, and its loads of the next one have arrived
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(in_flight.value) : "memory");
        meet();
      }
      half(Number<1>(), next, load, other, at);
      at = other;
    };
    const Number<0> no;
    const Number<1> yes;
    int left = stages;
    for (; left > STAGES; --left) stage(yes, Number<(STAGES - 2) * LOADS>(), yes);
    // what is left has been asked for: the loads on their way are those of the stages behind the next one
    if constexpr (STAGES >= 4) {
      if (left == 4) {
        stage(no, Number<2 * LOADS>(), yes);
        --left;
      }
    }
    if constexpr (STAGES >= 3) {
      if (left == 3) {
        stage(no, Number<LOADS>(), yes);
        --left;
      }
    }
    if (left == 2) stage(no, no, yes);
    stage(no, no, no);
  }
};

// The tile of 256 x 256 by eight wavefronts of 128 x 64, two stages in LDS.  Wavefronts 0 to 3 and 4 to 7 (one of each
// on every SIMD) take turns: a stage is four quarters of 64 x 32, and between barriers one half of the wavefronts multiplies
// a quarter while the other reads the operands of its next quarter and issues loads.
//
//   quarter (A half, W half)    read before it       loads issued before it (stage t being multiplied)
//     (0, 0)                    A half 0             A half 1 of t + 1
//     (0, 1)                    W half 1             W half 0 of t + 2
//     (1, 0)                    A half 1             A half 0 of t + 2
//     (1, 1)                    W half 0 of t + 1    W half 1 of t + 2
//
// A half of the stage's rows is written again only behind a barrier that all reads of it were answered before, in both halves of the
// wavefronts (the second runs one barrier behind the first).  The first quarter's products wait for the reads of A half 0, the second's
// for W half 1 and the third's for A half 1, each two barriers or more before the loads that write there.  W half 0 is read a quarter
// early, and the second half's first products come in the very interval in which the first half's loads overwrite it: the reads
// before the first quarter wait for it, which costs nothing (its four are older than A's eight, and LDS answers in order).
// What a quarter reads has arrived because every wavefront waited for its own loads of it before a barrier that lies in between.
struct Large {
  static constexpr int BM = 256, BN = 256, WM = 2, WN = 4, WAVES = 8, PM = 128, PN = 64, MT = 8, X = 4;
  static constexpr int HALF = 128 * ROW_BYTES, STAGE_BYTES = 4 * HALF, LDS_BYTES = 2 * STAGE_BYTES;

  // offsets [half][load]: load j of wavefront v is of LDS rows (v * 2 + j) * 8 + lane / 8 of the half
  struct Source {
    const char* a;
    const char* w;
    uint32_t a_off[2][2], w_off[2][2];
  };
  // the A row of the tile at LDS row q of half h, and the group of 16 and row in it of W's (of wavefront column q / 32)
  static __device__ __forceinline__ int a_row(int h, int q) { return (q / 64) * 128 + h * 64 + q % 64; }
  template <int MODE>
  static __device__ __forceinline__ int w_row(int h, int q) { return (q / 32) * PN + dealt_row<MODE, X>(h * 2 + (q / 16) % 2, q % 16); }

  static __device__ __forceinline__ uint32_t lds_at(const char* lds) {
    return __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)lds);
  }
  static __device__ __forceinline__ void load_a(uint32_t lds0, const Source& src, int h, uint32_t stage) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
#pragma unroll
    for (int j = 0; j < 2; ++j) load_to_lds(lds0 + stage + h * HALF + (wave * 2 + j) * 1024, src.a_off[h][j], src.a);
  }
  static __device__ __forceinline__ void load_w(uint32_t lds0, const Source& src, int h, uint32_t stage) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
#pragma unroll
    for (int j = 0; j < 2; ++j) load_to_lds(lds0 + stage + (2 + h) * HALF + (wave * 2 + j) * 1024, src.w_off[h][j], src.w);
  }
  // The first loads of a tile; no wavefront reads `lds` any more (as when `run` is through).
  static __device__ __forceinline__ void begin(char* lds, Source& src) {
    const uint32_t lds0 = lds_at(lds);
    load_w(lds0, src, 0, 0);
    load_a(lds0, src, 0, 0);
    load_w(lds0, src, 1, 0);
    load_a(lds0, src, 1, 0);
    src.a += ROW_BYTES;
    src.w += ROW_BYTES;
    load_w(lds0, src, 0, STAGE_BYTES);
    load_a(lds0, src, 0, STAGE_BYTES);
    load_w(lds0, src, 1, STAGE_BYTES);
  }

  // Behind `begin`; `stages` >= 2.  Loads and stores that came between are waited for with its loads, but for STORES if `stored`: that many were.
  template <int STORES>
  static __device__ __forceinline__ void run(f32x4 (&acc)[MT][X], char* lds, Source& src, int stages, bool stored) {
    const int lane = threadIdx.x % PAE_WAVE, col = lane % 16, kg = lane / 16;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
    const int wm = wave / WN, wn = wave % WN;
    const uint32_t lds0 = lds_at(lds);
    auto load_a = [&](int h, uint32_t stage) { Large::load_a(lds0, src, h, stage); };
    auto load_w = [&](int h, uint32_t stage) { Large::load_w(lds0, src, h, stage); };
    uint32_t a_at[2], w_at[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const uint32_t piece = ((s * 4 + kg) ^ ((col >> 1) & 7)) * 16;
      a_at[s] = (wm * 64 + col) * ROW_BYTES + piece;
      w_at[s] = 2 * HALF + (wn * 32 + col) * ROW_BYTES + piece;
    }
    bf16x8 a[4][2], w[2][2][2];  // [group][half of k], [W half][group][half of k]
    auto read_a = [&](int h, uint32_t stage) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) a[i][s] = *reinterpret_cast<const bf16x8*>(lds + stage + h * HALF + a_at[s] + i * 16 * ROW_BYTES);
    };
    auto read_w = [&](int h, uint32_t stage) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int x = 0; x < 2; ++x) w[h][x][s] = *reinterpret_cast<const bf16x8*>(lds + stage + h * HALF + w_at[s] + x * 16 * ROW_BYTES);
    };
    auto multiply = [&](int ha, int hw) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int x = 0; x < 2; ++x)
            acc[ha * 4 + i][hw * 2 + x] =
                __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[hw][x][s], a[i][s], acc[ha * 4 + i][hw * 2 + x], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    };
    auto forward = [&]() {
      src.a += ROW_BYTES;
      src.w += ROW_BYTES;
    };
    // the first stage: all but the last three halves, of two loads each
    if (STORES > 0 && stored) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(6 + STORES) : "memory");
    else asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
    meet();
    if (wm == 1) meet();
    // ONE, TWO: stages t + 1 and t + 2 there are
    auto stage = [&](auto one_, auto two_, uint32_t at) {
      constexpr int ONE = one_.value, TWO = two_.value;
      const uint32_t other = at ^ STAGE_BYTES;
      read_a(0, at);
      asm volatile("s_waitcnt lgkmcnt(8)" ::: "memory");  // W half 0, whose rows the other half's next loads write: all but A's eight reads
      if (ONE) {
        load_a(1, other);
        forward();
      }
      meet();
      multiply(0, 0);
      meet();
      read_w(1, at);
      if (TWO) load_w(0, at);
      meet();
      multiply(0, 1);
      meet();
      read_a(1, at);
      if (TWO) load_a(0, at);
      // W half 0 of t + 1: behind it A half 0, W half 1 and A half 1 of t + 1 and two halves of t + 2 were asked for
      if (TWO) asm volatile("s_waitcnt vmcnt(10)" ::: "memory");
      else if (ONE) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
      meet();
      multiply(1, 0);
      meet();
      if (ONE) read_w(0, other);
      if (TWO) load_w(1, at);
      // the whole of t + 1
      if (TWO) asm volatile("s_waitcnt vmcnt(6)" ::: "memory");
      else if (ONE) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      meet();
      multiply(1, 1);
      meet();
    };
    read_w(0, 0);
    asm volatile("" ::: "memory");  // before the reads of A half 0, as that wait counts them
    __builtin_amdgcn_sched_barrier(0);
    uint32_t at = 0;
    for (int left = stages; left > 2; --left) {
      stage(Number<1>(), Number<1>(), at);
      at ^= STAGE_BYTES;
    }
    stage(Number<1>(), Number<0>(), at);
    stage(Number<0>(), Number<0>(), at ^ STAGE_BYTES);
    if (wm == 0) meet();
  }
};

}  // namespace wide_gemm
