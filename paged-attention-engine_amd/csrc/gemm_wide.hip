// bfloat16 products with many rows, C = A W^T, on the matrix cores: the loops of wide_gemm.h, with what follows a product in the
// epilogue: a bias and an activation, a gated activation, or the sums of a range of k as they are.
//
// A launch is either the tiles of 256 x 256 as long as they fill rounds of the chip's 256 compute units, then what is left over
// of them whole, in halves or in quarters, where these still make one round; or, where that leaves too many units
// idle, smaller tiles throughout; and of either k may be cut into ranges that leave float32 sums of their own.  Which one is the
// least of what the shapes' measured times say (pae_gemm_wide_plan).
//
// An attention layer's projections are rotated and stored by the product as well (ROTATED), which then writes queries, keys and values once
// where a kernel behind it read and wrote them again: 2,048 x 2,048 x 1,536 18.3 and 11.2 us behind it, 22.9 in one; 6,030 x 4,608 x 3,584
// 160 and 45.6, 177 in one.  What the epilogue adds is the angles' and pages' way and the values' stores of 2 bytes.
//
// Measured beside the platform library's product (weights from memory, us; rows x features x k):
//     2,048 x 17,920 x  1,536   library 111 and 22 for the gate behind it    here with the gate 101
//     2,048 x  1,536 x  8,960           71                                   66
//     2,048 x  2,048 x  1,536           19                                   15
//     6,030 x 37,888 x  3,584        1,209 and 117 for the gate              1,175 with the gate
//     6,030 x  3,584 x 18,944        1,041                                   600
//       601 x  1,536 x  8,960           36                                   24 in ranges of k
//       200 x  1,536 x  1,536           20                                   8
// With the norm that adds the ranges' sums, without ranges in the tiles of 256 x 256 and with them: 2,048 x 1,536 x 8,960 77.7 and, in five
// ranges, 69.4; 2,500 x 2,048 x 11,008 134 and, in three, 107.
#include "wide_gemm.h"
#include "api.h"

#include <type_traits>

using wide_gemm::bf16x4;
using wide_gemm::bf16x8;
using wide_gemm::f32x4;
using wide_gemm::Large;
using wide_gemm::Tile;

namespace {

constexpr int UNITS = 256, DIES = 8, NO_ACT = -1;

// Where the rows of a projection to query, key and value heads go, and how they are rotated (ROTATED).
struct Heads {
  const float* cos_sin;     // [M][rot / 2][2]
  const int* positions;     // [M]
  const int* tok_seq;       // [M] row of block_tables
  const int* block_tables;  // [sequences][max_blocks]
  bf16_t* k_cache;          // [block][key/value head][bs][hd]
  bf16_t* v_cache;          // [block][key/value head][hd][bs]
  int nh, nkv, hd, rot, max_blocks, bs;
};

struct Product {
  void* out;  // bfloat16 [M][ldc], or float32 [split][M][ldc]
  int64_t ldc;
  const char* a;  // rows of lda bytes
  const char* w;  // rows of ldw bytes
  int64_t lda, ldw;
  const void* bias;
  int b_is_f32;
  int M, N, stages, splits;
  int row_tiles, col_tiles, strip;
  int whole;  // tiles of 256 x 256 that are run as such
  Heads heads;
};

// The row of W that a tile takes as its row n: of a rotated head's rows, in sixteens, 8 features and then the 8 they are rotated with.
template <int MODE>
__device__ __forceinline__ int w_row_of(const Product& p, int n) {
  if (MODE != wide_gemm::ROTATED) return n;
  const int head = n / p.heads.hd, f = n % p.heads.hd, half = p.heads.rot / 2;
  if (head >= p.heads.nh + p.heads.nkv || f >= p.heads.rot) return n;
  return head * p.heads.hd + (f % 16 < 8 ? f / 16 * 8 + f % 8 : half + f / 16 * 8 + f % 8);
}

// The first row of W that the tile from n0 on may take.
template <int MODE>
__device__ __forceinline__ int first_w_row(const Product& p, int n0) { return MODE == wide_gemm::ROTATED ? n0 / p.heads.hd * p.heads.hd : n0; }

// Workgroups i, i + 8, i + 16, ... run on one die: they take an eighth of `count` in a row, so that tiles that share
// rows of A or W find them in their die's L2.
__device__ __forceinline__ int in_row(int i, int count) {
  const int q = count / DIES, r = count % DIES, die = i % DIES;
  return die * q + min(die, r) + i / DIES;
}

// Tile `id` of row_tiles x col_tiles: strips of `strip` row tiles, column by column.
__device__ __forceinline__ void place_of(int id, int row_tiles, int col_tiles, int strip, int& tm, int& tn) {
  const int s = id / (strip * col_tiles), in = id - s * strip * col_tiles, rows = min(strip, row_tiles - s * strip);
  tm = s * strip + in % rows;
  tn = in / rows;
}

// What an activation reads: the sum as a product kept in bfloat16 holds it.  So a product with its activation is the same bits as the
// product and the activation's kernel behind it, which make it where there is no plan, and a near tie among a later
// layer's experts falls the same way whichever of the two ran.
__device__ __forceinline__ float rounded(float sum) { return (float)(__bf16)sum; }

// acc[i][x][e] of a wavefront: row row0 + 16 i + lane % 16 by W row n0 + dealt_row(x, 4 (lane / 16) + e).
// ACT: the activation's code (common.h), NO_ACT none; a template's argument, as code for all of them at every element is more than
// the instruction cache holds (2,048 rows by 17,920 features: 150 us instead of 115).
template <int MODE, int ACT, int MT, int X>
__device__ __forceinline__ void finish(const Product& p, const f32x4 (&acc)[MT][X], int row0, int n0, int split) {
  const int lane = threadIdx.x % PAE_WAVE, col = lane % 16, kg = lane / 16;
  if constexpr (MODE == wide_gemm::GATED) {
    static_assert(X == 2 || X == 4, "4 or 8 neighbouring features a lane");
    const int f = n0 / 2 + kg * (2 * X);
    if (f >= p.N / 2) return;  // N / 2 is a multiple of 8
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = row0 + 16 * i + col;
      if (row >= p.M) continue;
      bf16_t* o = (bf16_t*)p.out + row * p.ldc + f;
      __bf16 v[2 * X];
#pragma unroll
      for (int x = 0; x < X; x += 2)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[2 * x + e] = (__bf16)(act_to<bf16_t>(rounded(acc[i][x][e]), ACT) * rounded(acc[i][x + 1][e]));
      if constexpr (X == 4) *reinterpret_cast<bf16x8*>(o) = *reinterpret_cast<const bf16x8*>(v);
      else *reinterpret_cast<bf16x4*>(o) = *reinterpret_cast<const bf16x4*>(v);
    }
  } else if constexpr (MODE == wide_gemm::ROTATED) {
    static_assert(X == 2 || X == 4, "4 or 8 neighbouring features a lane");
    // a lane's 2 X features of a row and, 8 rows of the tile behind them, those they are rotated with (or simply the next ones)
    const Heads& h = p.heads;
    const int at = kg * (2 * X), n = n0 + at / 8 * 16 + at % 8;  // tile row of the first
    if (n >= p.N) return;
    // (the same head in the whole part, and wholly turned or not: heads and what is rotated of them are multiples of 64 wide)
    const int head = n0 / h.hd, f0 = n - head * h.hd, half = h.rot / 2;
    const bool turned = head < h.nh + h.nkv && n0 - head * h.hd < h.rot, cached = head >= h.nh, value = head >= h.nh + h.nkv;
    const int lo = turned ? f0 / 16 * 8 + f0 % 8 : f0, hi = turned ? lo + half : f0 + 8;
    f32x4 bias[X];
#pragma unroll
    for (int x = 0; x < X; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) bias[x][e] = p.bias ? load_param(p.bias, p.b_is_f32, head * h.hd + (x % 2 ? hi : lo) + x / 2 * 4 + e) : 0.f;
    constexpr int AT_ONCE = MT < 4 ? MT : 4;  // rows whose angles and pages are asked for together
#pragma unroll
    for (int i0 = 0; i0 < MT; i0 += AT_ONCE) {
      f32x4 angles[AT_ONCE][X];  // (cosine, sine) of 2 X pairs
      int64_t place[AT_ONCE];
      if (turned) {
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) {
          const float* from = h.cos_sin + ((int64_t)min(row0 + 16 * (i0 + i) + col, p.M - 1) * half + lo) * 2;
#pragma unroll
          for (int x = 0; x < X; ++x) angles[i][x] = *reinterpret_cast<const f32x4*>(from + 4 * x);
        }
      }
      if (cached) {
        int pos[AT_ONCE], seq[AT_ONCE];
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i) {
          const int row = min(row0 + 16 * (i0 + i) + col, p.M - 1);
          pos[i] = h.positions[row];
          seq[i] = h.tok_seq[row];
        }
#pragma unroll
        for (int i = 0; i < AT_ONCE; ++i)
          place[i] = ((int64_t)h.block_tables[(int64_t)seq[i] * h.max_blocks + pos[i] / h.bs] * h.nkv + (head - h.nh) % h.nkv) * ((int64_t)h.bs * h.hd) +
                     (int64_t)(pos[i] % h.bs) * (value ? 1 : h.hd);
      }
#pragma unroll
      for (int i = 0; i < AT_ONCE; ++i) {
        const int row = row0 + 16 * (i0 + i) + col;
        if (row >= p.M) continue;
        // the projection is rounded to bfloat16 before the rotation, as where the two are separate kernels
        __bf16 v[2][2 * X];
#pragma unroll
        for (int x = 0; x < X; ++x)
#pragma unroll
          for (int e = 0; e < 4; ++e) v[x % 2][x / 2 * 4 + e] = (__bf16)(acc[i0 + i][x][e] + bias[x][e]);
        if (turned) {
#pragma unroll
          for (int e = 0; e < 2 * X; ++e) {
            const float a = (float)v[0][e], b = (float)v[1][e], c = angles[i][e / 2][2 * (e % 2)], s = angles[i][e / 2][2 * (e % 2) + 1];
            v[0][e] = (__bf16)(a * c - b * s);
            v[1][e] = (__bf16)(b * c + a * s);
          }
        }
        if (value) {  // values lie the other way round
          __bf16* values = (__bf16*)h.v_cache + place[i];
#pragma unroll
          for (int part = 0; part < 2; ++part)
#pragma unroll
            for (int e = 0; e < 2 * X; ++e) values[(int64_t)((part ? hi : lo) + e) * h.bs] = v[part][e];
          continue;
        }
        bf16_t* o = cached ? h.k_cache + place[i] : (bf16_t*)p.out + row * p.ldc + (int64_t)head * h.hd;
        if constexpr (X == 4) {
          *reinterpret_cast<bf16x8*>(o + lo) = *reinterpret_cast<const bf16x8*>(v[0]);
          *reinterpret_cast<bf16x8*>(o + hi) = *reinterpret_cast<const bf16x8*>(v[1]);
        } else {
          *reinterpret_cast<bf16x4*>(o + lo) = *reinterpret_cast<const bf16x4*>(v[0]);
          *reinterpret_cast<bf16x4*>(o + hi) = *reinterpret_cast<const bf16x4*>(v[1]);
        }
      }
    }
  } else if constexpr (MODE == wide_gemm::SUMS) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = row0 + 16 * i + col;
      if (row >= p.M) continue;
      float* o = (float*)p.out + ((int64_t)split * p.M + row) * p.ldc;
#pragma unroll
      for (int x = 0; x < X; ++x) {
        const int n = n0 + 16 * x + 4 * kg;
        if (n < p.N) *reinterpret_cast<f32x4*>(o + n) = acc[i][x];
      }
    }
  } else {
    f32x4 bias[X];
    if (p.bias) {
#pragma unroll
      for (int x = 0; x < X; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          bias[x][e] = load_param(p.bias, p.b_is_f32, min(n0 + wide_gemm::dealt_row<MODE, X>(x, 4 * kg + e), p.N - 1));
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = row0 + 16 * i + col;
      if (row >= p.M) continue;
      bf16_t* o = (bf16_t*)p.out + row * p.ldc;
      f32x4 z[X];
#pragma unroll
      for (int x = 0; x < X; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) z[x][e] = ACT == NO_ACT ? acc[i][x][e] : rounded(acc[i][x][e]);
      if (p.bias) {
#pragma unroll
        for (int x = 0; x < X; ++x) z[x] += bias[x];
      }
      __bf16 v[4 * X];
#pragma unroll
      for (int x = 0; x < X; ++x)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * x + e] = (__bf16)(ACT == NO_ACT ? z[x][e] : act_to<bf16_t>(z[x][e], ACT));
#pragma unroll
      for (int x = 0; x < X; x += 2) {
        const int n = n0 + 16 * x + (x + 1 < X ? 8 : 4) * kg;
        if (n >= p.N) continue;  // N is a multiple of 8
        if (x + 1 < X) *reinterpret_cast<bf16x8*>(o + n) = *reinterpret_cast<const bf16x8*>(v + 4 * x);
        else *reinterpret_cast<bf16x4*>(o + n) = *reinterpret_cast<const bf16x4*>(v + 4 * x);
      }
    }
  }
}

// The tile of T at rows m0.. and W rows n0..; stages [first, first + stages) of k.
template <int MODE, int ACT, typename T>
__device__ __forceinline__ void small_tile(const Product& p, char* lds, int m0, int n0, int first, int stages, int split) {
  const int lane = threadIdx.x % PAE_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  typename T::Source src;
  src.a = p.a + m0 * p.lda + (int64_t)first * wide_gemm::ROW_BYTES;
  const int w0 = first_w_row<MODE>(p, n0);
  src.w = p.w + w0 * p.ldw + (int64_t)first * wide_gemm::ROW_BYTES;
#pragma unroll
  for (int j = 0; j < T::A_LOADS; ++j) {
    const int q = (wave * T::A_LOADS + j) * 8 + lane / 8;
    src.a_off[j] = (uint32_t)min(q, p.M - 1 - m0) * (uint32_t)p.lda + wide_gemm::piece_of(lane, q);
  }
#pragma unroll
  for (int j = 0; j < T::W_LOADS; ++j) {
    const int q = (wave * T::W_LOADS + j) * 8 + lane / 8;
    const int n = q / T::PN * T::PN + wide_gemm::dealt_row<MODE, T::X>(q % T::PN / 16, q % 16);
    src.w_off[j] = (uint32_t)(w_row_of<MODE>(p, min(n0 + n, p.N - 1)) - w0) * (uint32_t)p.ldw + wide_gemm::piece_of(lane, q);
  }
  f32x4 acc[T::MT][T::X];
#pragma unroll
  for (int i = 0; i < T::MT; ++i)
#pragma unroll
    for (int x = 0; x < T::X; ++x) acc[i][x] = f32x4{0.f, 0.f, 0.f, 0.f};
  T::run(acc, lds, src, stages);
  finish<MODE, ACT>(p, acc, m0 + wave / T::WN * T::PM, n0 + wave % T::WN * T::PN, split);
}

using Half = Tile<128, 256, 2, 4, 3>;     // of a tile of 256 x 256, by the same eight wavefronts
using Quarter = Tile<128, 128, 2, 4, 4>;

// Whether a workgroup takes one tile of 256 x 256 after another (see below): where an activation makes the epilogue long.  Without one a workgroup a tile
// is ahead (us, in turns and not: sums of ranges 6,030 x 1,536 x 8,960 in three 146.7 and 141.7, 2,500 x 2,048 x 11,008 in five 114.0 and 111.9; 2,048 x 37,888 x
// 3,584 410.8 and 405.4), and the epilogue of rotated heads has no registers left for it, 28 bytes a lane went to memory and back (6,030 x 4,608 x 3,584 165.6
// and 165.2).  With one: by erf 8,192 x 8,960 x 1,536 211.6 and 217.6.
template <int MODE, int ACT>
constexpr bool in_turns() { return ACT != NO_ACT; }

// parts: into how many each tile behind the whole ones is cut (1, 2 or 4)
template <int MODE, int ACT, int PARTS>
__global__ __launch_bounds__(512, 2) void wide_large_kernel(Product p) {
  extern __shared__ __attribute__((aligned(16))) char wide_lds[];
  const int lane = threadIdx.x % PAE_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  int tm, tn;
  const int ranges = MODE == wide_gemm::SUMS ? p.whole * p.splits : p.whole, together = in_turns<MODE, ACT>() ? min(ranges, UNITS) : ranges;
  if (PARTS > 1 && (int)blockIdx.x >= together) {
    const int rest = (p.row_tiles * p.col_tiles - p.whole) * PARTS, at = in_row(blockIdx.x - together, rest);
    place_of(p.whole + at / PARTS, p.row_tiles, p.col_tiles, p.strip, tm, tn);
    const int m0 = tm * 256 + at % PARTS / (PARTS / 2) * 128, n0 = tn * 256 + (PARTS == 4 ? at % 2 * 128 : 0);
    if (m0 >= p.M || n0 >= p.N) return;
    small_tile<MODE, ACT, typename std::conditional<PARTS == 4, Quarter, Half>::type>(p, wide_lds, m0, n0, 0, p.stages, 0);
    return;
  }
  // A unit's workgroup takes one tile after another (the ones that it would be given one by one), and asks for the next one's first stages
  // before it leaves a tile's results: what a tile needs beside its stages, some 11 of 39 us at k 1,536, is the way of its first stage, its epilogue and
  // a workgroup's start (gated, us, a workgroup a tile and this: 8,192 x 17,920 x 1,536 356 and 349, 6,030 271 and 263, 2,048 102.2 and 100.7, 8,192 x 22,016 x
  // 2,048 552 and 539, 8,192 x 9,728 x 896 132 and 127; 6,030 x 37,888 x 3,584 1,178 and 1,175).
  Large::Source src;
  int m0, n0, split, stages;
  auto begin = [&](int i) {
    int id = in_row(i, ranges), first = 0;
    split = 0;
    stages = p.stages;
    if (MODE == wide_gemm::SUMS) {  // the ranges of k lie one after another
      split = id / p.whole;
      id -= split * p.whole;
      first = (int)((int64_t)p.stages * split / p.splits);
      stages = (int)((int64_t)p.stages * (split + 1) / p.splits) - first;
    }
    place_of(id, p.row_tiles, p.col_tiles, p.strip, tm, tn);
    m0 = tm * 256;
    n0 = tn * 256;
    src.a = p.a + m0 * p.lda + (int64_t)first * wide_gemm::ROW_BYTES;
    const int w0 = first_w_row<MODE>(p, n0);
    src.w = p.w + w0 * p.ldw + (int64_t)first * wide_gemm::ROW_BYTES;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int q = (wave * 2 + j) * 8 + lane / 8;
        src.a_off[h][j] = (uint32_t)min(Large::a_row(h, q), p.M - 1 - m0) * (uint32_t)p.lda + wide_gemm::piece_of(lane, q);
        src.w_off[h][j] = (uint32_t)(w_row_of<MODE>(p, min(n0 + Large::w_row<MODE>(h, q), p.N - 1)) - w0) * (uint32_t)p.ldw + wide_gemm::piece_of(lane, q);
      }
    Large::begin(wide_lds, src);
  };
  begin(blockIdx.x);
  // Stores of a whole tile's results by a wavefront, 16 bytes a lane each and none under a condition then: the next tile's first stage is
  // waited for and they are not (gated, us, waited for and not, with a SiLU of half the instructions: 8,192 x 17,920 x 1,536 338 and 334, 2,048 96.4 and 95.5, 8,192 x 9,728 x 896 117 and 113).
  constexpr int STORES = !in_turns<MODE, ACT>() ? 0 : MODE == wide_gemm::GATED ? Large::MT : Large::MT * Large::X / 2;
  bool stored = false;
  for (int i = blockIdx.x; i < ranges; i += together) {
    f32x4 acc[Large::MT][Large::X];
#pragma unroll
    for (int j = 0; j < Large::MT; ++j)
#pragma unroll
      for (int x = 0; x < Large::X; ++x) acc[j][x] = f32x4{0.f, 0.f, 0.f, 0.f};
    Large::run<STORES>(acc, wide_lds, src, stages, stored);
    stored = m0 + 256 <= p.M && n0 + 256 <= p.N;
    const int row0 = m0 + wave / Large::WN * Large::PM, col0 = n0 + wave % Large::WN * Large::PN, of = split;
    if (in_turns<MODE, ACT>() && i + together < ranges) begin(i + together);
    finish<MODE, ACT>(p, acc, row0, col0, of);
    if (!in_turns<MODE, ACT>()) return;
  }
}

// One shape of smaller tiles throughout; the ranges of k lie one after another.  (Never all 512 registers for a wavefront: the
// compiler would put part of the sums into the accumulation file and move them to and fro.)
template <int MODE, int ACT, typename T>
__global__ __launch_bounds__(T::WAVES * 64, 2) void wide_small_kernel(Product p) {
  extern __shared__ __attribute__((aligned(16))) char wide_lds[];
  const int tiles = p.row_tiles * p.col_tiles;
  int id = in_row(blockIdx.x, tiles * p.splits), tm, tn;
  const int split = id / tiles;
  id -= split * tiles;
  place_of(id, p.row_tiles, p.col_tiles, p.strip, tm, tn);
  const int first = (int)((int64_t)p.stages * split / p.splits), last = (int)((int64_t)p.stages * (split + 1) / p.splits);
  small_tile<MODE, ACT, T>(p, wide_lds, tm * T::BM, tn * T::BN, first, last - first, split);
}

template <typename K>
int launch(K kernel, const Product& p, int64_t blocks, int threads, int lds, hipStream_t stream) {
  const hipError_t err = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  PAE_REQUIRE(err == hipSuccess, "wide product: %d bytes of LDS refused: %s", lds, hipGetErrorString(err));
  kernel<<<(unsigned)blocks, threads, lds, stream>>>(p);
  return pae_check_launch("gemm_wide");
}

int64_t tiles_of(int M, int N, int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); }

template <int MODE, int ACT, typename T>
int launch_small(Product p, hipStream_t stream) {
  p.row_tiles = (p.M + T::BM - 1) / T::BM;
  p.col_tiles = (p.N + T::BN - 1) / T::BN;
  p.strip = 8;
  PAE_REQUIRE((int64_t)p.row_tiles * p.col_tiles * p.splits < (1ll << 30), "wide product: too many tiles");
  return launch(wide_small_kernel<MODE, ACT, T>, p, (int64_t)p.row_tiles * p.col_tiles * p.splits, T::WAVES * 64, T::LDS_BYTES, stream);
}

// Workgroups of tiles of 256 x 256.
template <int MODE, int ACT>
int64_t together(int64_t tiles) { return in_turns<MODE, ACT>() && tiles > UNITS ? UNITS : tiles; }

template <int MODE, int ACT>
int launch_large(Product p, hipStream_t stream) {
  p.row_tiles = (p.M + 255) / 256;
  p.col_tiles = (p.N + 255) / 256;
  p.strip = 8;
  const int64_t tiles = (int64_t)p.row_tiles * p.col_tiles;
  PAE_REQUIRE(tiles < (1ll << 28), "wide product: too many tiles");
  if constexpr (MODE == wide_gemm::SUMS) {
    p.whole = (int)tiles;
    PAE_REQUIRE(tiles * p.splits < (1ll << 30), "wide product: too many tiles");
    return launch(wide_large_kernel<MODE, ACT, 1>, p, together<MODE, ACT>(tiles * p.splits), 512, Large::LDS_BYTES, stream);
  }
  const int rest = (int)(tiles % UNITS), parts = rest == 0 || rest > UNITS / 2 ? 1 : rest > UNITS / 4 ? 2 : 4;
  p.whole = (int)(parts == 1 ? tiles : tiles - rest);
  constexpr int LDS = Large::LDS_BYTES > Half::LDS_BYTES ? Large::LDS_BYTES : Half::LDS_BYTES;
  static_assert(Quarter::LDS_BYTES <= LDS, "room for every part");
  if (parts == 1) return launch(wide_large_kernel<MODE, ACT, 1>, p, together<MODE, ACT>(tiles), 512, Large::LDS_BYTES, stream);
  if (parts == 2) return launch(wide_large_kernel<MODE, ACT, 2>, p, together<MODE, ACT>(p.whole) + 2 * rest, 512, LDS, stream);
  return launch(wide_large_kernel<MODE, ACT, 4>, p, together<MODE, ACT>(p.whole) + 4 * rest, 512, LDS, stream);
}

enum { SHAPE_LARGE, SHAPE_128_256, SHAPE_128_128, SHAPE_128_96, SHAPE_64_128, SHAPE_64_64, SHAPES };

// Microseconds of a product in a shape, from times of all shapes at 14 sizes of weights (896 to 18,944 of k) by 24 row counts
// from 72 to 8,192, which this meets within 11 to 13 % (root mean square): a round of tiles costs its start and end and so much a
// stage.  The shapes of two workgroups a unit take a quarter longer a stage from 2,048 of k on, with weights from memory (64 x 64 at up
// to one a unit: 0.16 to 0.20 up to k 1,536, 0.24 to 0.26 from 2,048 to 18,944; 64 x 128 0.32 and 0.40 to 0.43).  The least of all is on
// average 1 % behind the fastest shape (300 x 4,608 x 3,584 24.8 us; without that quarter 64 x 128 was taken, 28.1).
// Ranges of k in tiles of 256 x 256: 1.15 us a stage where all tiles are one round and 1.45 behind that, where the chip's clock has gone down; with
// the norm that adds the ranges' sums, at 7 widths by 15 row counts, the choice is 1.1 % behind the fastest (in us, without such tiles and with them:
// 2,048 x 1,536 x 8,960 77.7 and 69.4 in five ranges, 3,000 x 1,536 x 8,960 111 and 90, 4,096 x 1,536 x 8,960 139 and 114, 2,500 x 2,048 x 11,008 134
// and 107, 1,000 x 3,584 x 18,944 147 and 131, 2,048 x 3,584 x 18,944 269 and 234; but 6,000 x 3,584 x 18,944 681 whole and 702).
double shape_time(int shape, int M, int N, int K, int splits) {
  const double stages = K / 64.0 / splits;
  struct Cost { int bm, bn, blocks; double launch, round, stage, part; };  // part: a stage of a last round that half the units' places or fewer take
  static const Cost cost[SHAPES] = {{256, 256, 1, 0.0, 3.5, 1.35, 0.0},  {128, 256, 1, 0.0, 2.9, 0.73, 0.73}, {128, 128, 1, 0.0, 2.4, 0.46, 0.46},
                                    {128, 96, 1, 0.3, 2.4, 0.39, 0.39}, {64, 128, 2, 2.5, 0.0, 0.62, 0.33},  {64, 64, 2, 2.9, 0.0, 0.38, 0.21}};
  const Cost& c = cost[shape];
  const double far = c.blocks == 2 && K >= 2048 * splits ? 1.25 : 1.0;
  const int64_t tiles = tiles_of(M, N, c.bm, c.bn) * splits, places = (int64_t)UNITS * c.blocks;
  const int64_t rest = tiles % places;
  double last = 0.0;
  if (shape == SHAPE_LARGE && splits > 1) return (tiles + UNITS - 1) / UNITS * (c.round + stages * (tiles <= UNITS ? 1.15 : 1.45));
  if (rest) last = c.round + stages * (shape == SHAPE_LARGE ? (rest > UNITS / 2 ? c.stage : rest > UNITS / 4 ? 0.77 : 0.40) : far * (rest > places / 2 ? c.stage : c.part));
  return c.launch + tiles / places * (c.round + stages * far * c.stage) + last;
}

template <int MODE, int ACT>
int run_shape(int shape, const Product& p, hipStream_t stream) {
  constexpr bool PAIRS = MODE == wide_gemm::GATED || MODE == wide_gemm::ROTATED;
  switch (shape) {
    case SHAPE_LARGE: return launch_large<MODE, ACT>(p, stream);
    case SHAPE_128_256: return launch_small<MODE, ACT, Tile<128, 256, 2, 4, 3>>(p, stream);
    case SHAPE_128_128: return launch_small<MODE, ACT, Tile<128, 128, 2, 2, 4>>(p, stream);
    case SHAPE_128_96:
      if constexpr (!PAIRS) return launch_small<MODE, ACT, Tile<128, 96, 2, 2, 4>>(p, stream);
      break;
    case SHAPE_64_128: return launch_small<MODE, ACT, Tile<64, 128, 2, 2, 3>>(p, stream);
    case SHAPE_64_64: return launch_small<MODE, ACT, Tile<64, 64, 2, 2, 4>>(p, stream);
  }
  return pae_fail("wide product: shape %d does not take mode %d", shape, MODE);
}

}  // namespace

// Microseconds of a projection by the platform's library and the kernel that rotates and stores behind it, where the rule below leaves the
// product to the library: met within 11 % (root mean square) over 187 such products of 12 widths of heads (768 to 12,288 rows of W, k 2,048 to
// 8,192) by 65 to 6,030 rows.
static double library_and_rotation_time(int M, int N, int K) {
  return 12.8 + 0.80e-9 * M * N * K + 0.72e-6 * N * K + 2.3e-6 * M * N + 1.8e-6 * M * K;
}

// The shape for a product, in the low byte, and its ranges of k behind that.  `mode` as for pae_gemm_wide; `ranges` != 0: the
// product may leave float32 sums of ranges of k for a caller that reads them again (counted at 3.6 TB/s against one bfloat16
// result).  -1: the platform library, which shares a product out over k, for one without an activation that no shape here fills
// the chip with.  That is from 30 us on and below 0.95 PFLOP/s by the times above, where the library was ahead of
// these shapes two times in three (6,030 x 1,536 x 8,960 141 against 160 us, 2,048 x 4,608 x 3,584 59 against 68); and from 48 stages of k
// on where even tiles of 64 x 64 leave half the units idle, whose one chain of stages is then longer than the library's shares: up
// to 64 tiles 0.84 to 1.83 times its time, 1.30 on average, and up to 128 0.85 to 1.26, 1.04 on average (128 x 896 x 4,864 23.9 against 13.1
// us, 300 x 256 x 4,096 18.6 against 11.2, 65 x 16 x 8,192 22.4 against 8.3).  Up to 35 stages as few tiles are ahead (65 x 1,536 x 2,240 8.8
// against 11.4), and so are 128 to 256 of them (0.84 on average).
// Heads that are rotated (mode 3) leave the library its products only where that and a rotation behind it are ahead by their times: over
// those 187 products the tiles with the rotation in them take 0.94 of its time with this rule and 1.01 without, 1.09 at worst and
// 1.71 (us, tiles and library: 65 x 1,536 x 8,192 35.2 and 20.9, 127 x 768 x 4,096 22.6 and 15.6, 993 x 1,536 x 8,192 67.6 and 52.5, 240 x
// 5,120 x 6,144 64.0 and 51.3, which go to the library; 993 x 4,608 x 3,584 56.8 and 63.6, 385 x 7,168 x 5,120 44.4 and 65.6, 127 x 10,240 x 8,192
// 80.9 and 74.3, which do not).
extern "C" int pae_gemm_wide_plan(int mode, int act, int M, int N, int K, int ranges) {
  static const int CUTS[] = {2, 3, 4, 5, 6, 8};
  int best = SHAPE_LARGE, cuts = 1;
  double least = 1e30;
  for (int shape = 0; shape < SHAPES; ++shape) {
    if ((shape == SHAPE_128_96 && (mode == wide_gemm::GATED || mode == wide_gemm::ROTATED)) || (shape == SHAPE_LARGE && K < 128)) continue;
    const double t = shape_time(shape, M, N, K, 1);
    if (t < least) least = t, best = shape;
  }
  for (int shape = SHAPE_LARGE; ranges && shape < SHAPES; ++shape)
    for (int n : CUTS) {
      if (K < 1024 * n) break;  // (k of 1,536 in two ranges: 8.2 -> 7.8 us at best, and slower from 900 rows on)
      const double t = shape_time(shape, M, N, K, n) + (4.0 * n - 2.0) * M * N / 3.6e6;
      if (t < least) least = t, best = shape, cuts = n;
    }
  if (mode == wide_gemm::PLAIN && act == NO_ACT &&
      ((least > 30.0 && 2.0 * M * N * K / least < 0.95e9) || (K >= 48 * 64 && tiles_of(M, N, 64, 64) <= UNITS / 2)))
    return -1;
  if (mode == wide_gemm::ROTATED && pae_gemm_wide_plan(wide_gemm::PLAIN, NO_ACT, M, N, K, 0) < 0 &&
      1.05 * least + 1.3 + 0.9e-6 * M * N > 0.95 * library_and_rotation_time(M, N, K))
    return -1;
  return best | cuts << 8;
}

static int wide_product(int mode, int act, int plan, void* out, int64_t ldc, const void* a, int64_t lda, const void* w, const void* bias,
                        int b_is_f32, int M, int N, int K, const Heads& heads, hipStream_t stream);

// C = A W^T for A [M, K] (rows of lda numbers), W [N, K]; K a multiple of 64, N of 16.  mode 0: bfloat16 [M, N] of act(A W^T + bias), act
// -1 (none), 0 or 3; 1: bfloat16 [M, N / 2] of act(gate) * other, W's rows in blocks of 8 of the one and of the
// other, act 1 or 2; 2: float32 [ranges, M, N] of the sums over ranges of k.  Operands begin at multiples of 16 bytes.
extern "C" int pae_gemm_wide(int mode, int act, int plan, void* out, int64_t ldc, const void* a, int64_t lda, const void* w, const void* bias,
                             int b_is_f32, int M, int N, int K, hipStream_t stream) {
  PAE_REQUIRE(mode != wide_gemm::ROTATED, "wide product: heads that are rotated have an entry point of their own");
  return wide_product(mode, act, plan, out, ldc, a, lda, w, bias, b_is_f32, M, N, K, Heads{}, stream);
}

static int wide_product(int mode, int act, int plan, void* out, int64_t ldc, const void* a, int64_t lda, const void* w, const void* bias,
                        int b_is_f32, int M, int N, int K, const Heads& heads, hipStream_t stream) {
  const int shape = plan & 255, ranges = plan >> 8;
  PAE_REQUIRE(M > 0 && N > 0 && N % 16 == 0 && K > 0 && K % 64 == 0, "wide product: bad sizes M=%d N=%d K=%d", M, N, K);
  PAE_REQUIRE(plan >= 0 && shape < SHAPES && ranges >= 1 && ranges <= K / 64 && (mode == wide_gemm::SUMS || ranges == 1) && (shape != SHAPE_LARGE || K >= 128 * ranges),
              "wide product: plan %d for mode %d and K=%d", plan, mode, K);
  PAE_REQUIRE(lda >= 0 && lda % 8 == 0 && lda < (1 << 22) && K < (1 << 22), "wide product: rows of %lld numbers", (long long)lda);  // 256 rows in 32 bits
  PAE_REQUIRE(ldc % (mode == wide_gemm::SUMS ? 4 : 8) == 0 && ((uintptr_t)out | (uintptr_t)a | (uintptr_t)w) % 16 == 0, "wide product: operands must lie at multiples of 16 bytes");
  Product p;
  p.out = out;
  p.ldc = ldc;
  p.a = (const char*)a;
  p.lda = lda * 2;
  p.w = (const char*)w;
  p.ldw = (int64_t)K * 2;
  p.bias = bias;
  p.b_is_f32 = b_is_f32;
  p.M = M;
  p.N = N;
  p.stages = K / 64;
  p.splits = ranges;
  p.row_tiles = p.col_tiles = p.strip = p.whole = 0;
  p.heads = heads;
  if (mode == wide_gemm::ROTATED) {
    PAE_REQUIRE(heads.hd > 0, "wide projection: heads of no width");
    return run_shape<wide_gemm::ROTATED, NO_ACT>(shape, p, stream);
  }
  if (mode == wide_gemm::SUMS) return run_shape<wide_gemm::SUMS, NO_ACT>(shape, p, stream);
  if (mode == wide_gemm::PLAIN && act == NO_ACT) return run_shape<wide_gemm::PLAIN, NO_ACT>(shape, p, stream);
  if (mode == wide_gemm::PLAIN && act == 0) return run_shape<wide_gemm::PLAIN, 0>(shape, p, stream);
  if (mode == wide_gemm::PLAIN && act == 3) return run_shape<wide_gemm::PLAIN, 3>(shape, p, stream);
  if (mode == wide_gemm::GATED && act == 1) return run_shape<wide_gemm::GATED, 1>(shape, p, stream);
  if (mode == wide_gemm::GATED && act == 2) return run_shape<wide_gemm::GATED, 2>(shape, p, stream);
  return pae_fail("wide product: mode %d with activation %d", mode, act);
}

// A W^T + bias, W [(nh + 2 nkv) hd, K] the projections to query, key and value heads: query heads, their first `rot` features rotated in pairs
// (i, i + rot / 2), to out [M, nh hd], key heads rotated likewise and value heads to their places in the pages, as pae_rope_kv_write
// puts them.  `plan` as pae_gemm_wide_plan gives it for mode 3.  nkv may be 0: only queries.
extern "C" int pae_gemm_wide_rope(int plan, void* out, int64_t ldc, const void* a, int64_t lda, const void* w, const void* bias, int b_is_f32,
                                  int M, int K, int nh, int nkv, int hd, int rot, const float* cos_sin, const int* positions, const int* tok_seq,
                                  const int* block_tables, int max_blocks, int bs, void* k_cache, void* v_cache, hipStream_t stream) {
  PAE_REQUIRE(nh > 0 && nkv >= 0 && hd > 0 && hd % 64 == 0 && rot >= 0 && rot <= hd && rot % 64 == 0 && (rot == 0 || cos_sin),
              "wide projection: heads of %d with %d features rotated", hd, rot);
  PAE_REQUIRE(nkv == 0 || (bs > 0 && max_blocks > 0 && k_cache && v_cache && block_tables && tok_seq && positions),
              "wide projection: the cache write needs tables and pools");
  PAE_REQUIRE(ldc >= (int64_t)nh * hd && (uintptr_t)k_cache % 16 == 0 && (uintptr_t)cos_sin % 16 == 0 && (int64_t)(256 + hd) * K < (1ll << 31),
              "wide projection: rows of %lld numbers, or operands between multiples of 16 bytes", (long long)ldc);
  return wide_product(wide_gemm::ROTATED, NO_ACT, plan, out, ldc, a, lda, w, bias, b_is_f32, M, (nh + 2 * nkv) * hd, K,
                      Heads{cos_sin, positions, tok_seq, block_tables, (bf16_t*)k_cache, (bf16_t*)v_cache, nh, nkv, hd, rot, max_blocks, bs}, stream);
}
