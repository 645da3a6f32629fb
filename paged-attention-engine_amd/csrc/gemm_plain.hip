// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]): the plain matrix product of the
// float32 path, also available for bfloat16 operands with float32 accumulation.
//
// W is stored (out_features, in_features) row-major as in the checkpoint, the
// layout F.linear takes in the reference (engine/model.py:303-305,315,318-320).
//
// Products run on the float32 matrix cores (v_mfma_f32_16x16x4_f32: products and sums in full
// 32-bit).  k is cut into slabs of 16, of which one instruction takes the j-th number of every
// four (j = 0..3 in turn: a lane reads four neighbouring k at once), and into blocks of 512 whose
// sums are then added up in order (with rows of 30,000 terms one running sum loses a digit more
// than the block sums do).  Every kernel here adds in this order, so that the value of an output
// element does not depend on M, on the tile it falls in, on how the blocks are shared out
// or on which other rows share the launch.
//
// Why three kernels.  Up to 64 rows the weights' way from memory is the time: `few` gives 16 weight
// rows to a workgroup whose wavefronts take a block of k each, nothing staged (a wavefront reads 16
// rows x 64 bytes an instruction).  With more rows the matrix cores are: `tiles` stages 32 of k of 64
// rows of either side through LDS, two buffers that take turns.  Where a launch has too
// few tiles for the chip the blocks of k are shared out over workgroups as well (`splits`): the
// block sums go to scratch memory and `sum` adds them in order.
// Measured, weights from HBM, 2,048 / 1,536 / 17,920 x 1,536 and 1,536 x 8,960 (the kernel before this one, 64 x 64 tiles of
// multiply-adds on the vector ALU, took 240 ms of a pass of three requests of 601 tokens in all and four steps behind
// them at the 1.5B sizes; these take 25):
//   3 rows     6.6, 6.6, 25.1 (4.4 TB/s), 21.9 us
//   601 rows   50, 37, 311 (106 TFLOP/s), 184 us
//   2,048      115, 87, 970 (116 TFLOP/s), 478 us (118 of the 154 that the chip gives)
// Tried: tiles of 128 x 128, 128 x 64 (the accumulators and block totals of a wavefront then leave one or two of
// them a SIMD: 377 and 326 us for the third product at 601 rows), 16 and 64 of k a stage (329, 322 us).  In `few`
// the compiler moves the loads of a batch down to where they are used unless it is told not to (sched_barrier): 18.8
// against 15.3 us a launch in the step.
#include "common.h"
#include "api.h"

#define GP_BLOCK 512  // k of a block whose sum is formed before it joins the total
#define GP_SLAB 16    // k of four instructions
#define GP_FEW_ROWS 64
#define GP_FEW_WAVES 8
#define GP_TILE 64    // rows of either side of a tile
#define GP_UNITS 256  // compute units

typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 load4(const float* p) { return *(const f32x4*)p; }
__device__ __forceinline__ f32x4 load4(const bf16_t* p) {
  const uint2 v = *(const uint2*)p;
  return f32x4{__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
               __uint_as_float(v.y & 0xffff0000u)};
}
// Four numbers of a row from k on, zeros from `end` on; number by number.
template <typename T>
__device__ __forceinline__ f32x4 load4_to(const T* row, int k, int end) {
  f32x4 v;
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = k + u < end ? to_f32(row[k + u]) : 0.f;
  return v;
}

// One slab: four instructions, the j-th numbers of the lanes' fours.
__device__ __forceinline__ f32x4 slab(f32x4 acc, f32x4 a, f32x4 b) {
#pragma unroll
  for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[j], acc, 0, 0, 0);
  return acc;
}

// Up to 16 * MT rows: blockIdx.x 16 weight rows, blockIdx.y the product of the batch, blockIdx.z a share of
// the blocks of k, one block a wavefront at a time.  VEC: rows may be read four numbers at a time.
template <typename TA, typename TC, int MT, bool VEC>
__global__ __launch_bounds__(64 * GP_FEW_WAVES) void gemm_plain_few_kernel(
    TC* __restrict__ C, int64_t ldc, const TA* __restrict__ A, int64_t lda, const TA* __restrict__ W,
    const void* __restrict__ bias, int b_is_f32, int M, int N, int K, int64_t batch_c, int64_t batch_a,
    int64_t batch_w, float* __restrict__ scratch) {
  C += blockIdx.y * batch_c;
  A += blockIdx.y * batch_a;
  W += blockIdx.y * batch_w;
  extern __shared__ float part[];  // [wavefront][16 * MT][16]
  const int waves = blockDim.x / PAE_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  const int lane = threadIdx.x % PAE_WAVE, r = lane % 16, kq = lane / 16;
  const int n0 = blockIdx.x * 16;
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  const int step = waves * gridDim.z;
  // rows past the end are read as the last one and dropped
  const TA* w_row = W + (int64_t)min(n0 + r, N - 1) * K;
  const TA* a_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) a_row[i] = A + (int64_t)min(i * 16 + r, M - 1) * lda;
  constexpr int U = MT == 1 ? 4 : 2;  // slabs whose loads are on their way together, twice
  constexpr int TOTALS = (16 * MT * 16) / PAE_WAVE;
  float total[TOTALS];  // thread t: outputs t, t + threads, ...
#pragma unroll
  for (int i = 0; i < TOTALS; ++i) total[i] = 0.f;

  for (int first = 0; first < blocks; first += step) {  // the same trips for every wavefront
    const int block = first + blockIdx.z * waves + wave;
    f32x4 acc[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (block < blocks) {
      int k = block * GP_BLOCK;
      const int end = min(K, k + GP_BLOCK);
      const int steady = VEC ? (end - k) / (GP_SLAB * U) : 0;
      if (steady) {
        // two batches take turns; no load stands under a condition of its own
        struct Batch {
          f32x4 w[U], a[U][MT];
        } b0, b1;
        auto fetch = [&](Batch& b, int at) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            b.w[u] = load4(w_row + at + u * GP_SLAB + kq * 4);
#pragma unroll
            for (int i = 0; i < MT; ++i) b.a[u][i] = load4(a_row[i] + at + u * GP_SLAB + kq * 4);
          }
          __builtin_amdgcn_sched_barrier(0);
        };
        auto multiply = [&](const Batch& b) {
#pragma unroll
          for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < MT; ++i) acc[i] = slab(acc[i], b.a[u][i], b.w[u]);
          __builtin_amdgcn_sched_barrier(0);
        };
        constexpr int STEP = GP_SLAB * U;
        int batches = steady;
        fetch(b0, k);
        while (batches >= 3) {
          fetch(b1, k + STEP);
          multiply(b0);
          fetch(b0, k + 2 * STEP);
          multiply(b1);
          k += 2 * STEP;
          batches -= 2;
        }
        if (batches == 2) {
          fetch(b1, k + STEP);
          multiply(b0);
          multiply(b1);
        } else {
          multiply(b0);
        }
        k += batches * STEP;
      }
      for (; k < end; k += GP_SLAB) {
        const f32x4 w = load4_to(w_row, k + kq * 4, end);
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i] = slab(acc[i], load4_to(a_row[i], k + kq * 4, end), w);
      }
    }
    if (scratch) {  // this block's sums to memory; another kernel adds them up
      if (block < blocks && n0 + r < N) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int m = i * 16 + kq * 4 + e;
            if (m < M) scratch[((int64_t)block * M + m) * N + n0 + r] = acc[i][e];
          }
      }
      continue;
    }
    float* mine = part + wave * (MT * 256);
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) mine[(i * 16 + kq * 4 + e) * 16 + r] = acc[i][e];
    __syncthreads();
    const int here = min(waves, blocks - first);
#pragma unroll
    for (int i = 0; i < TOTALS; ++i) {
      const int o = threadIdx.x + i * blockDim.x;
      if (o < MT * 256)
        for (int v = 0; v < here; ++v) total[i] += part[v * (MT * 256) + o];
    }
    __syncthreads();
  }
  if (scratch) return;
#pragma unroll
  for (int i = 0; i < TOTALS; ++i) {
    const int o = threadIdx.x + i * blockDim.x, m = o / 16, n = n0 + o % 16;
    if (o < MT * 256 && m < M && n < N) {
      float v = total[i];
      if (bias) v += load_param(bias, b_is_f32, n);
      C[(int64_t)m * ldc + n] = from_f32<TC>(v);
    }
  }
}

// Tiles of BM x BN, four wavefronts of BM/2 x BN/2.  blockIdx.x: the tiles, those of one column of tiles (the same weights)
// next to each other on one die; blockIdx.y: the product of the batch; blockIdx.z: a share of the blocks of k.
// A row's 16 numbers of a slab lie in LDS as four fours, at places turned by the row so that the 16 rows
// a wavefront reads a four of fall into different banks.
template <typename TA, typename TC, int BM, int BN, int SLABS, bool VEC>
__global__ __launch_bounds__(256) void gemm_plain_tiles_kernel(
    TC* __restrict__ C, int64_t ldc, const TA* __restrict__ A, int64_t lda, const TA* __restrict__ W,
    const void* __restrict__ bias, int b_is_f32, int M, int N, int K, int64_t batch_c, int64_t batch_a,
    int64_t batch_w, float* __restrict__ scratch) {
  C += blockIdx.y * batch_c;
  A += blockIdx.y * batch_a;
  W += blockIdx.y * batch_w;
  __shared__ f32x4 a_lds[2][SLABS][BM * 4], w_lds[2][SLABS][BN * 4];
  const int tid = threadIdx.x, lane = tid % PAE_WAVE, r = lane % 16, kq = lane / 16;
  const int wave = __builtin_amdgcn_readfirstlane(tid / PAE_WAVE);
  const int tiles_m = (M + BM - 1) / BM;
  const int tiles = gridDim.x;
  // workgroups i, i + 8, i + 16, ... run on one die: they take neighbouring tiles
  const int per = tiles / 8, rest = tiles % 8, die = blockIdx.x % 8;
  const int tile = die * per + min(die, rest) + blockIdx.x / 8;
  const int m0 = (tile % tiles_m) * BM, n0 = (tile / tiles_m) * BN;
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  const int share = (blocks + gridDim.z - 1) / gridDim.z;
  const int block0 = blockIdx.z * share, block1 = min(blocks, block0 + share);
  if (block0 >= block1) return;

  constexpr int CA = BM * 4 / 256, CW = BN * 4 / 256;  // fours that a thread brings of either side
  const TA* a_src[CA];
  const TA* w_src[CW];
  int a_dst[CA], w_dst[CW];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const int c = tid + i * 256, row = c / 4;
    a_src[i] = A + (int64_t)min(m0 + row, M - 1) * lda;
    a_dst[i] = row * 4 + ((c % 4) ^ ((row >> 2) & 3));
  }
#pragma unroll
  for (int i = 0; i < CW; ++i) {
    const int c = tid + i * 256, row = c / 4;
    w_src[i] = W + (int64_t)min(n0 + row, N - 1) * K;
    w_dst[i] = row * 4 + ((c % 4) ^ ((row >> 2) & 3));
  }
  const int kc = (tid % 4) * 4;
  constexpr int TM = BM / 32, TN = BN / 32;  // matrix tiles of a wavefront
  const int wm = (wave / 2) * (BM / 2), wn = (wave % 2) * (BN / 2);
  const int at = r * 4 + (kq ^ ((r >> 2) & 3));  // of the lane's four within a matrix tile's 16 rows

  f32x4 acc[TM][TN], total[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  f32x4 a_reg[SLABS][CA], w_reg[SLABS][CW];
  auto fetch = [&](int k) {
    if (VEC && k + GP_SLAB * SLABS <= K) {
#pragma unroll
      for (int u = 0; u < SLABS; ++u) {
#pragma unroll
        for (int i = 0; i < CA; ++i) a_reg[u][i] = load4(a_src[i] + k + u * GP_SLAB + kc);
#pragma unroll
        for (int i = 0; i < CW; ++i) w_reg[u][i] = load4(w_src[i] + k + u * GP_SLAB + kc);
      }
    } else {  // zeros past the end add nothing
#pragma unroll
      for (int u = 0; u < SLABS; ++u) {
#pragma unroll
        for (int i = 0; i < CA; ++i) a_reg[u][i] = load4_to(a_src[i], k + u * GP_SLAB + kc, K);
#pragma unroll
        for (int i = 0; i < CW; ++i) w_reg[u][i] = load4_to(w_src[i], k + u * GP_SLAB + kc, K);
      }
    }
  };
  auto put = [&](int buf) {
#pragma unroll
    for (int u = 0; u < SLABS; ++u) {
#pragma unroll
      for (int i = 0; i < CA; ++i) a_lds[buf][u][a_dst[i]] = a_reg[u][i];
#pragma unroll
      for (int i = 0; i < CW; ++i) w_lds[buf][u][w_dst[i]] = w_reg[u][i];
    }
  };
  const int k_begin = block0 * GP_BLOCK, k_end = min(K, block1 * GP_BLOCK);
  fetch(k_begin);
  put(0);
  __syncthreads();
  int buf = 0;
  for (int block = block0; block < block1; ++block) {
    const int end = min(K, (block + 1) * GP_BLOCK);
    for (int k = block * GP_BLOCK; k < end; k += GP_SLAB * SLABS) {
      const bool more = k + GP_SLAB * SLABS < k_end;
      if (more) fetch(k + GP_SLAB * SLABS);
#pragma unroll
      for (int u = 0; u < SLABS; ++u) {
        f32x4 a[TM], w[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = a_lds[buf][u][(wm + i * 16) * 4 + at];
#pragma unroll
        for (int j = 0; j < TN; ++j) w[j] = w_lds[buf][u][(wn + j * 16) * 4 + at];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i][q], w[j][q], acc[i][j], 0, 0, 0);
      }
      if (more) {
        put(buf ^ 1);
        __syncthreads();
        buf ^= 1;
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        if (scratch) {
          const int n = n0 + wn + j * 16 + r;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int m = m0 + wm + i * 16 + kq * 4 + e;
            if (m < M && n < N) scratch[((int64_t)block * M + m) * N + n] = acc[i][j][e];
          }
        } else {
          total[i][j] += acc[i][j];
        }
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  if (scratch) return;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + wn + j * 16 + r;
    if (n >= N) continue;
    const float b = bias ? load_param(bias, b_is_f32, n) : 0.f;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int m = m0 + wm + i * 16 + kq * 4 + e;
        if (m >= M) continue;
        float v = total[i][j][e];
        if (bias) v += b;
        C[(int64_t)m * ldc + n] = from_f32<TC>(v);
      }
  }
}

// The block sums [blocks][M][N] added up in order.
template <typename TC>
__global__ __launch_bounds__(256) void gemm_plain_sum_kernel(TC* __restrict__ C, int64_t ldc,
                                                             const float* __restrict__ scratch,
                                                             const void* __restrict__ bias, int b_is_f32, int M,
                                                             int N, int blocks) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  const int m = blockIdx.y;
  if (n >= N) return;
  const int64_t stride = (int64_t)M * N;
  const float* p = scratch + (int64_t)m * N + n;
  float total = 0.f;
  int b = 0;
  for (; b + 8 <= blocks; b += 8) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = p[(b + u) * stride];
#pragma unroll
    for (int u = 0; u < 8; ++u) total += v[u];
  }
  for (; b < blocks; ++b) total += p[b * stride];
  if (bias) total += load_param(bias, b_is_f32, n);
  C[(int64_t)m * ldc + n] = from_f32<TC>(total);
}

// Over how many workgroups the blocks of k of one tile are shared: 1 where the tiles fill the chip by themselves or
// there is one block only.  A share costs its sums a way to memory and back and the launch that adds them (about
// 4 us), so that up to 64 rows a workgroup's wavefronts take up to GP_FEW_WAVES blocks side by side first.
// Up to 64 rows a compute unit works through its workgroups in rounds, and shares pay where they leave fewer rounds of the whole
// k; with more rows, up to one and a half tiles a compute unit.  Measured without shares / with them: 3 rows of 11,008 by 128 sixteens of
// weight rows (2 rounds of a third) 36.1 / 30.1 us, of 16,384 by 192 (3 of a quarter) 50.0 / 44.3, of 8,192 by 192 (2 of a half)
// 27.0 / 28.6, of 11,008 by 256 (3 of a third) 44.8 / 49.3; 320 tiles 392 / 299 (601 x 2,048 x 11,008), 376 669 / 632 (3,000 x 512 x
// 18,944), 416 397 / 433 (800 x 2,048 x 11,008), 658 258 / 288 (3,000 x 896 x 4,864), 728 992 / 1,121 (800 x 3,584 x 18,944).
static int splits_of(int M, int N, int K) {
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  if (M <= 0 || blocks == 1) return 1;
  if (M <= GP_FEW_ROWS) {
    if (blocks <= GP_FEW_WAVES) return 1;
    const int64_t sixteens = (N + 15) / 16, shares = (blocks + GP_FEW_WAVES - 1) / GP_FEW_WAVES;
    const int64_t rounds = (sixteens + GP_UNITS - 1) / GP_UNITS, rounds_of_shares = (sixteens * shares + GP_UNITS - 1) / GP_UNITS;
    return rounds_of_shares < rounds * shares && shares <= 65535 ? (int)shares : 1;
  }
  const int64_t tiles = (int64_t)((M + GP_TILE - 1) / GP_TILE) * ((N + GP_TILE - 1) / GP_TILE);
  if (2 * tiles >= 3 * GP_UNITS) return 1;
  const int want = (int)((3 * GP_UNITS + tiles - 1) / tiles);  // three workgroups a compute unit
  return want < blocks ? want : blocks;
}

// Rows and columns of C that one pass of launches makes.  A product with shared blocks of k keeps their sums, whatever the
// number of shares: up to GP_SCRATCH floats (128 MiB) at once, more rows or columns than that one after the other, the longer side of C
// cut into equal parts (all at once, a product of 2,000 x 512 x 18,944 would keep 152 MB; cut it takes 428 us instead of 380; one of
// 200 x 3,584 x 18,944 keeps 106 MB).  And a grid's threads along x are counted in 32 bits.
#define GP_SCRATCH (32 << 20)
struct GpPart {
  int rows, cols;
};
static GpPart part_of(int M, int N, int K, bool shared) {
  const int64_t blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
  auto cut = [](int whole, int64_t most) {  // equal parts of at most `most`, in multiples of a tile
    const int64_t tiles = (whole + GP_TILE - 1) / GP_TILE, fit = most / GP_TILE > 0 ? most / GP_TILE : 1, parts = (tiles + fit - 1) / fit;
    return parts == 1 ? whole : (int)((tiles + parts - 1) / parts * GP_TILE);
  };
  GpPart part = {M, cut(N, 1 << 26)};
  if (shared && splits_of(M, N, K) > 1 && blocks * M * N > GP_SCRATCH) {
    if (N >= M) part.cols = cut(N, GP_SCRATCH / (blocks * M));
    else part.rows = cut(M, GP_SCRATCH / (blocks * N));
  }
  part.rows = cut(part.rows, (int64_t)0xffffff / ((part.cols + GP_TILE - 1) / GP_TILE) * GP_TILE);
  return part;
}

// part_of, for who wants to look: part[0] rows by part[1] columns.
extern "C" void pae_gemm_plain_part(int M, int N, int K, int shared, int* part) {
  const GpPart p = part_of(M, N, K, shared != 0);
  part[0] = p.rows;
  part[1] = p.cols;
}

// Floats of scratch memory that pae_gemm_plain_shared is best called with (0: none).
extern "C" int64_t pae_gemm_plain_scratch(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || splits_of(M, N, K) == 1) return 0;
  const GpPart part = part_of(M, N, K, true);
  return (int64_t)((K + GP_BLOCK - 1) / GP_BLOCK) * part.rows * part.cols;
}

template <typename TA, typename TC, bool VEC>
static int launch_plain(void* C, int64_t ldc, int64_t batch_c, const void* A, int64_t lda, int64_t batch_a,
                        const void* W, int64_t batch_w, const void* bias, int b_is_f32, int M, int N, int K, int batch,
                        float* scratch, int splits, hipStream_t stream) {
  const int blocks = (K + GP_BLOCK - 1) / GP_BLOCK;
#define GP_ARGS                                                                                                  \
  (TC*)C, ldc, (const TA*)A, lda, (const TA*)W, bias, b_is_f32, M, N, K, batch_c, batch_a, batch_w, scratch
  // (over 32 rows read number by number by one wavefront a workgroup: the tiles are faster, 64 x 130 x 511 67 -> 44 us; over
  // five blocks of k they are not, 64 x 1,537 x 2,049 74 against 171)
  if (M <= (VEC || blocks > 1 ? GP_FEW_ROWS : GP_FEW_ROWS / 2)) {
    const int each = (blocks + splits - 1) / splits;
    const int waves = each < GP_FEW_WAVES ? each : GP_FEW_WAVES;
    const dim3 grid((N + 15) / 16, batch, splits);
#define GP_FEW(MT)                                                                                               \
  gemm_plain_few_kernel<TA, TC, MT, VEC><<<grid, waves * PAE_WAVE, scratch ? 0 : waves * MT * 1024, stream>>>(GP_ARGS)
    if (M <= 16) GP_FEW(1);
    else if (M <= 32) GP_FEW(2);
    else GP_FEW(4);
#undef GP_FEW
  } else {
    const dim3 grid((unsigned)(((M + GP_TILE - 1) / GP_TILE) * (int64_t)((N + GP_TILE - 1) / GP_TILE)), batch, splits);
    gemm_plain_tiles_kernel<TA, TC, GP_TILE, GP_TILE, 2, VEC><<<grid, 256, 0, stream>>>(GP_ARGS);
  }
#undef GP_ARGS
  if (scratch) {
    const int bad = pae_check_launch("gemm_plain");
    if (bad) return bad;
    gemm_plain_sum_kernel<TC><<<dim3((N + 255) / 256, M), 256, 0, stream>>>((TC*)C, ldc, scratch, bias, b_is_f32, M, N, blocks);
  }
  return pae_check_launch("gemm_plain");
}

// in_dtype: operands; out_dtype: C.  Supported: f32->f32, bf16->bf16, bf16->f32.
// `batch` products at once (one per head, say): product b reads A + b batch_a and W + b batch_w and
// writes C + b batch_c, with the same leading dimensions; no bias then.  `scratch`: pae_gemm_plain_scratch floats for one product,
// whose k may then be shared over workgroups, or null.
extern "C" int pae_gemm_plain_shared(int in_dtype, int out_dtype, void* C, int64_t ldc, int64_t batch_c, const void* A,
                                     int64_t lda, int64_t batch_a, const void* W, int64_t batch_w, const void* bias,
                                     int b_is_f32, int M, int N, int K, int batch, float* scratch, hipStream_t stream) {
  PAE_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  PAE_REQUIRE(batch >= 1 && batch <= 65535 && (batch == 1 || !bias), "gemm: %d products at once (1..65535, no bias)", batch);
  PAE_REQUIRE(lda >= K && ldc >= N, "gemm: leading dimensions lda=%lld ldc=%lld too small for K=%d N=%d",
              (long long)lda, (long long)ldc, K, N);
  PAE_REQUIRE(batch == 1 || !scratch, "gemm: shares of k go with one product at a time, not with %d", batch);
  if (M == 0) return 0;
  PAE_REQUIRE(M <= 65535 * 64, "gemm: M=%d exceeds the grid", M);
  PAE_REQUIRE((in_dtype == PAE_F32 && out_dtype == PAE_F32) || (in_dtype == PAE_BF16 && (out_dtype == PAE_BF16 || out_dtype == PAE_F32)),
              "gemm: unsupported dtype pair in=%d out=%d", in_dtype, out_dtype);
  // four numbers at a time: 16 bytes in float32, 8 in bfloat16
  const int elem = in_dtype == PAE_F32 ? 4 : 2, out_elem = out_dtype == PAE_F32 ? 4 : 2;
  const bool vec = K % 4 == 0 && lda % 4 == 0 && (batch == 1 || (batch_a % 4 == 0 && batch_w % 4 == 0)) &&
                   (uintptr_t)A % (4 * elem) == 0 && (uintptr_t)W % (4 * elem) == 0;
  const GpPart part = part_of(M, N, K, scratch != nullptr);
  for (int64_t n0 = 0; n0 < N; n0 += part.cols)
    for (int64_t m0 = 0; m0 < M; m0 += part.rows) {
      const int rows = (int)(M - m0 < part.rows ? M - m0 : part.rows), cols = (int)(N - n0 < part.cols ? N - n0 : part.cols);
      char* c = (char*)C + (m0 * ldc + n0) * out_elem;
      const char* a = (const char*)A + m0 * lda * elem;
      const char* w = (const char*)W + n0 * K * elem;
      const char* b = bias ? (const char*)bias + n0 * (b_is_f32 ? 4 : 2) : nullptr;
      const int splits = scratch ? splits_of(rows, cols, K) : 1;
      float* sums = splits > 1 ? scratch : nullptr;
#define GP_GO(TA, TC)                                                                                                    \
  (vec ? launch_plain<TA, TC, true>(c, ldc, batch_c, a, lda, batch_a, w, batch_w, b, b_is_f32, rows, cols, K, batch, sums, \
                                    splits, stream)                                                                      \
       : launch_plain<TA, TC, false>(c, ldc, batch_c, a, lda, batch_a, w, batch_w, b, b_is_f32, rows, cols, K, batch,    \
                                     sums, splits, stream))
      const int rc = in_dtype == PAE_F32 ? GP_GO(float, float) : out_dtype == PAE_BF16 ? GP_GO(bf16_t, bf16_t) : GP_GO(bf16_t, float);
#undef GP_GO
      if (rc) return rc;
    }
  return 0;
}

extern "C" int pae_gemm_plain_batched(int in_dtype, int out_dtype, void* C, int64_t ldc, int64_t batch_c, const void* A,
                                      int64_t lda, int64_t batch_a, const void* W, int64_t batch_w, const void* bias,
                                      int b_is_f32, int M, int N, int K, int batch, hipStream_t stream) {
  return pae_gemm_plain_shared(in_dtype, out_dtype, C, ldc, batch_c, A, lda, batch_a, W, batch_w, bias, b_is_f32, M, N, K,
                               batch, nullptr, stream);
}
