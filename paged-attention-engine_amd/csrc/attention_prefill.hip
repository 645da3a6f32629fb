// Causal attention of runs of tokens over the paged cache (bfloat16, pages of 16), keys and values shared through LDS.
//
// One workgroup of eight wavefronts per (32 QG consecutive tokens of a sequence, query head): QG groups of 32 tokens by
// KG = 8 / QG groups of keys.  A key group takes every KG-th tile of 16 QG keys; each of its QG wavefronts holds 32 tokens'
// queries in registers, brings one page of the tile's keys and values to LDS and multiplies all of the tile's with its queries:
//   S^T[32 keys x 32 tokens] = K Q^T,   O^T[features x 32 tokens] += V^T P^T     (MFMA 32x32x16)
// At the end the key groups' sums (reference, sum of weights, unnormalised output) are added through LDS, in their order.
//
// What bounds it: the matrix cores need 32 clocks a product and 1,024 a tile of 64 keys, a wavefront's exponentials,
// maxima, sums and roundings 650 to 1,150, and LDS 1,280 for a tile that four wavefronts read (128 KB) and fill (32 KB).
// So the wavefronts 0 to 3 and 4 to 7 (one of each on every SIMD) take turns: between two barriers one half multiplies (1,420
// clocks measured: the next tile's scores, then this tile's values, eight operands read ahead, the loads of the tile
// after that in between), the other weighs its scores (1,160).  A tile is 2,750 clocks for both, three quarters of the
// matrix rate, at the clock the chip holds under it (1.6 to 1.9 GHz); a workgroup's start, last tile and end are 10 us more.
// Measured, 12 heads of 128 over 2 key/value heads: one prompt of 2,048 tokens 37.8 -> 27.0 us, 8,192 tokens 326 -> 213
// (0.97 PFLOP/s), with a bias by distance and a gate 405 -> 231; 28 heads over 4, 6,000 tokens 452 -> 276; heads of 192 with
// values of 128, 6 prompts of 833 tokens 79 -> 37; before: the kernel of attention_mfma.hip, whose wavefronts each read their
// own keys from the cache.  Of the parts, left out one at a time in a copy (8,192 tokens, 231 us then): the weighing 199, the
// loads 192 (they stood beside the weighing then), three quarters of the second product 243.
//
// A score's place: the matrix instruction leaves lane (h = lane / 32, column = lane % 32), register i the row
// 8 (i / 4) + 4 h + i % 4 of S^T.  Which key is which row is free, as each lane reads its own row's key from LDS; it is dealt so
// that registers 8 m .. 8 m + 7 are the keys 16 m + 8 h .. of the tile in order.  That is the order in which the second
// product takes P^T against 16 bytes of a value row in its page ([feature][16 keys]): nothing moves between lanes.
//
// LDS: pages as they lie in the cache, rows of keys [HD] and of values [16]; the 16-byte pieces of a key row r are
// at places piece ^ (r % 16) (HD a multiple of 128) or piece ^ (r / 2 % 8), the two of a value row d at half ^ (d / 8 % 2): 16
// lanes that read at once meet all banks once (no conflicts counted).
//
// Two buffers a key group for keys and two for values.  Between the barriers in which a half multiplies tile n + 1's scores and
// tile n's values (both read from LDS), it asks for tile n + 2's keys and tile n + 1's values, to where tile n's keys and
// tile n - 1's values were, which every wavefront of the half had read before the barrier two back; every wavefront waits for its
// own loads before the barrier in front of the products that read them.
//
// The softmax's reference is as in attention_mfma.hip.  With QG = 2 keys are dealt to four key groups of 32 as there, and a
// result differs in the order of adding alone.  With QG = 4 there are two key groups of 64, and the sum of weights is that of the
// rounded ones, by which the values are multiplied: errors against 64 bits, relative, of 2,048 normal tokens 0.00201,
// by the unrounded weights 0.00204 (fewer keys then weigh exactly one), with QG = 2 and by the kernel before 0.00202.
#include "attention_device.h"
#include "attention_prefill.h"
#include "wide_gemm.h"

namespace {

using wide_gemm::load_to_lds;
using wide_gemm::meet;

typedef __attribute__((ext_vector_type(16))) float f32x16;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;

template <int HD, int VD, int QG>
struct Shape {
  static constexpr int KG = 8 / QG, TOK = 32 * QG, KEYS = 16 * QG, ST = QG / 2;
  static constexpr int K_PAGE = 16 * HD * 2, V_PAGE = 16 * VD * 2, K_TILE = QG * K_PAGE, V_TILE = QG * V_PAGE;
  static constexpr int K_LOADS = K_PAGE / 1024, V_LOADS = V_PAGE / 1024, GROUP = 2 * (K_TILE + V_TILE);
  static constexpr int SUMS = 8 * 64 * (VD / 2) * 4, MERGE = SUMS + 8 * 64 * 8;  // bytes: every wavefront's sums, references and shares
  static constexpr int LDS = KG * GROUP > MERGE ? KG * GROUP : MERGE;
};

template <int V>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" : : "n"(V) : "memory");
}

template <int HD, int VD, int QG, bool CAPPED, bool BIASED>
__global__ __launch_bounds__(512, 2) void attn_prefill_shared_kernel(PrefillArgs p) {
  using S = Shape<HD, VD, QG>;
  constexpr int KG = S::KG, ST = S::ST, QS = HD / 16, DT = VD / 32, PARTS = PREFILL_RUN / S::TOK;
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE), lane = threadIdx.x % PAE_WAVE;
  const int col = lane % 32, h = lane / 32, qg = wave % QG, kg = wave / QG;
  const int head = blockIdx.x % p.nh, kvh = head / (p.nh / p.nkv);
  const int tile = blockIdx.y, part = PARTS - 1 - blockIdx.x / p.nh;
  const int seq_row = p.tiles[tile * 3];
  const int tok0 = p.tiles[tile * 3 + 1] + part * S::TOK;
  const int ntok = min(S::TOK, p.tiles[tile * 3 + 2] - part * S::TOK);
  if (ntok <= 0) return;  // the whole workgroup
  // read by scalar loads (the constant address space: no store of this kernel goes there)
  const auto table = (const __attribute__((address_space(4))) int*)(p.block_tables + (int64_t)seq_row * p.max_blocks);
  const int pos0 = p.positions[tok0];
  const int hi = pos0 + ntok - 1;
  auto first_of = [&](int pos) { return BIASED ? first_visible(pos, p.window, p.chunked) : (p.window > 0 && pos - p.window + 1 > 0) ? pos - p.window + 1 : 0; };
  const int first = first_of(pos0), lo = first / 16 * 16;
  const int rounds = (hi - lo) / (S::KEYS * KG) + 1;

  const int c = 32 * qg + col;
  const bool live = c < ntok;
  const int pos = live ? pos0 + c : -1, start = live ? first_of(pos) : 0;
  const int wave_first = pos0 + 32 * qg, wave_start = first_of(min(hi, wave_first + 31));  // the wavefront's first position, its last one's first key
  bf16x8 qf[QS];
  {
    const bf16_t* qrow = p.q + (int64_t)(tok0 + (live ? c : 0)) * p.q_stride + (int64_t)head * HD + 8 * h;
#pragma unroll
    for (int j = 0; j < QS; ++j) qf[j] = *reinterpret_cast<const bf16x8*>(qrow + 16 * j);
  }

  // places in LDS
  auto fold = [](int row) { return HD % 128 == 0 ? row % 16 : (row >> 1) & 7; };
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds);
  const uint32_t group0 = kg * S::GROUP;
  uint32_t k_off[S::K_LOADS];
#pragma unroll
  for (int j = 0; j < S::K_LOADS; ++j) {
    const int piece = 64 * j + lane, row = piece / (HD / 8), place = piece % (HD / 8);
    k_off[j] = row * HD * 2 + (place ^ fold(row)) * 16;
  }
  const uint32_t v_off = (lane / 2) * 32 + ((lane % 2) ^ ((lane / 16) & 1)) * 16;
  const int key_row = 16 * (col / 16) + 8 * ((col / 4) % 2) + 4 * ((col / 8) % 2) + col % 4;  // see above
  const uint32_t k_at = group0 + (key_row / 16) * S::K_PAGE + (key_row % 16) * HD * 2;
  const uint32_t k_fold = (h ^ fold(key_row % 16)) * 16;
  const uint32_t v_at = group0 + 2 * S::K_TILE + col * 32 + (h ^ ((col / 8) & 1)) * 16;

  auto first_key = [&](int n) { return lo + ((BIASED ? rounds - 1 - n : n) * KG + kg) * S::KEYS; };
  auto page_of = [&](int n) {  // the page of this wavefront's sixteen keys of tile n; keys past the last one seen: the last one's page
    const int key = first_key(min(n, rounds - 1)) + 16 * qg;
    return max((int)table[min(key, hi) / 16], 0);
  };
  auto load_k = [&](const bf16_t* base, int buf, int j) { load_to_lds(lds0 + group0 + buf * S::K_TILE + qg * S::K_PAGE + j * 1024, k_off[j], base); };
  auto load_v = [&](const char* base, int buf, int j) {
    load_to_lds(lds0 + group0 + 2 * S::K_TILE + buf * S::V_TILE + qg * S::V_PAGE + j * 1024, v_off, base + j * 1024);
  };
  auto keys_of = [&](int page) { return p.k + ((int64_t)page * p.nkv + kvh) * (16 * HD); };
  auto values_of = [&](int page) { return reinterpret_cast<const char*>(p.v + ((int64_t)page * p.nkv + kvh) * (16 * VD)); };

  f32x16 acc[DT], s[ST];
  float ref = NEG_BIG, l = 0.f;
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
  bf16x8 pb[QG];

  const float slope = (BIASED && p.slopes) ? p.slopes[head] * p.inv_scale : 0.f;
  // The products of tile n's scores (SCORE) and of tile n - 1's weights with its values (ADD), and, between them, the loads
  // of the keys of tile n + 1 and the values of tile n (LOAD)
  auto products = [&](auto score_, auto add_, auto load_, int n, int page_k, int page_v) {
    constexpr bool SCORE = score_.value, ADD = add_.value, LOAD = load_.value;
    constexpr int FIRST = SCORE ? QS * ST : 0, N = FIRST + (ADD ? QG * DT : 0), AHEAD = 8;
    constexpr int LOADS = LOAD ? S::K_LOADS + S::V_LOADS : 0;
    if (SCORE) {
      const float from = BIASED ? (float)(first_key(n) + 8 * h - pos0) : 0.f;
#pragma unroll
      for (int st = 0; st < ST; ++st)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[st][i] = BIASED ? slope * (from + (float)(32 * st + 16 * (i / 8) + i % 8)) : 0.f;
    }
    const uint32_t kb = k_at + (n & 1) * S::K_TILE, vb = v_at + ((n & 1) ^ 1) * S::V_TILE;
    const bf16_t* next_k = LOAD ? keys_of(page_k) : nullptr;
    const char* next_v = LOAD ? values_of(page_v) : nullptr;
    bf16x8 a[AHEAD];
    auto read = [&](int i) {
      if (i < FIRST) a[i % AHEAD] = *reinterpret_cast<const bf16x8*>(lds + kb + (i % ST) * 2 * S::K_PAGE + (k_fold ^ (32 * (i / ST))));
      else a[i % AHEAD] = *reinterpret_cast<const bf16x8*>(lds + vb + ((i - FIRST) / DT) * S::V_PAGE + ((i - FIRST) % DT) * 1024);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) read(i);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (i < FIRST) s[i % ST] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i % AHEAD], qf[i / ST], s[i % ST], 0, 0, 0);
      else acc[(i - FIRST) % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i % AHEAD], pb[(i - FIRST) / DT], acc[(i - FIRST) % DT], 0, 0, 0);
      if (i + AHEAD < N) read(i + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      if (LOADS && i % (N / LOADS) == 0 && i / (N / LOADS) < LOADS) {
        const int j = i / (N / LOADS);
        if (j < S::V_LOADS) load_v(next_v, n & 1, j);
        else load_k(next_k, (n + 1) & 1, j - S::V_LOADS);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // what the other wavefronts may overwrite has been read
  };
  auto weights = [&](int n) {
    const int key0 = first_key(n);
    if (CAPPED) {  // s <- (cap / scale) tanh(s scale / cap): what follows multiplies by the scale as before
#pragma unroll
      for (int st = 0; st < ST; ++st)
#pragma unroll
        for (int i = 0; i < 16; ++i) s[st][i] = p.cap_over_scale * tanh_fast(s[st][i] * p.scale_over_cap);
    }
    if (!(key0 + S::KEYS - 1 <= wave_first && key0 >= wave_start)) {  // some key is hidden from some token of the wavefront
#pragma unroll
      for (int st = 0; st < ST; ++st)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = key0 + 32 * st + 16 * (i / 8) + 8 * h + i % 8;
          if (!(key <= pos && key >= start)) s[st][i] = -INFINITY;
        }
    }
    float mx = s[0][0];
#pragma unroll
    for (int st = 0; st < ST; ++st)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[st][i]);
    mx *= p.scale_log2;
    if (__builtin_amdgcn_ballot_w64(mx > ref + RESCALE_STEP) != 0) {  // the same in every lane; rare after the first tiles
      float m = fmaxf(mx, NEG_BIG);
      m = fmaxf(m, __shfl_xor(m, 32, PAE_WAVE));
      const float to = m > ref + RESCALE_STEP ? m : ref;
      const float alpha = __builtin_amdgcn_exp2f(ref - to);
      ref = to;
      l *= alpha;
#pragma unroll
      for (int t = 0; t < DT; ++t) acc[t] *= alpha;
    }
#pragma unroll
    for (int g = 0; g < QG; ++g) {
      float w[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) w[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[g / 2][8 * (g % 2) + i], p.scale_log2, -ref));
      bf16x2* pairs = reinterpret_cast<bf16x2*>(&pb[g]);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        pairs[i] = __builtin_convertvector((f32x2){w[2 * i], w[2 * i + 1]}, bf16x2);
        if (QG == 4) {  // what the values are multiplied by adds up to one
          const unsigned both = reinterpret_cast<unsigned*>(&pb[g])[i];
          w[2 * i] = __uint_as_float(both << 16);
          w[2 * i + 1] = __uint_as_float(both & 0xffff0000u);
        }
      }
      l += ((w[0] + w[1]) + (w[2] + w[3])) + ((w[4] + w[5]) + (w[6] + w[7]));
    }
  };

  const wide_gemm::Number<0> no;
  const wide_gemm::Number<1> yes;
  int page = page_of(0), next = page_of(1);
#pragma unroll
  for (int j = 0; j < S::K_LOADS; ++j) load_k(keys_of(page), 0, j);
  wait_loads<0>();
#pragma unroll
  for (int j = 0; j < QS; ++j) asm volatile("" : "+v"(qf[j]));  // the queries are there as well
  meet();
  if (wave >= 4) meet();
  products(yes, no, yes, 0, next, page);
  meet();
  for (int n = 0; n + 1 < rounds; ++n) {
    page = next;
    next = page_of(n + 2);
    weights(n);
    wait_loads<0>();
    asm volatile("" : "+s"(next));  // the table entry is there: the reads of LDS below are counted without it
    meet();
    __builtin_amdgcn_s_setprio(1);
    products(yes, yes, yes, n + 1, next, page);
    __builtin_amdgcn_s_setprio(0);
    meet();
  }
  weights(rounds - 1);
  wait_loads<0>();
  meet();
  products(no, yes, no, rounds, 0, 0);
  if (wave < 4) meet();

  // the groups' sums, references and shares through LDS; every group's wavefront adds up its part of the features
  l += __shfl_xor(l, 32, PAE_WAVE);
  __syncthreads();
  f32x4* sums = reinterpret_cast<f32x4*>(lds);
  float* shares = reinterpret_cast<float*>(lds + S::SUMS);
#pragma unroll
  for (int t = 0; t < DT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i)
      sums[((wave * DT + t) * 4 + i) * 64 + lane] = (f32x4){acc[t][4 * i], acc[t][4 * i + 1], acc[t][4 * i + 2], acc[t][4 * i + 3]};
  shares[wave * 128 + lane] = ref;
  shares[wave * 128 + 64 + lane] = l;
  __syncthreads();
  if (!live) return;
  float m = NEG_BIG;
#pragma unroll
  for (int g = 0; g < KG; ++g) m = fmaxf(m, shares[(g * QG + qg) * 128 + lane]);
  const float sink = p.sinks ? p.sinks[head] * LOG2E : 0.f;
  if (p.sinks) m = fmaxf(m, sink);
  float factor[KG], sum = p.sinks ? exp2f(sink - m) : 0.f;  // the head's sink joins the denominator without a value
#pragma unroll
  for (int g = 0; g < KG; ++g) {
    factor[g] = exp2f(shares[(g * QG + qg) * 128 + lane] - m);
    sum += shares[(g * QG + qg) * 128 + 64 + lane] * factor[g];
  }
  float inv = 1.0f / sum;
  if (!BIASED && p.head_gate)
    inv *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-__bfloat162float(p.head_gate[(int64_t)(tok0 + c) * p.head_gate_stride + head]) * LOG2E));
  bf16_t* o = p.out + (int64_t)(tok0 + c) * p.out_stride + (int64_t)head * VD + 4 * h;
  const bf16_t* gt = (BIASED && p.gate) ? p.gate + (int64_t)(tok0 + c) * p.gate_stride + (int64_t)head * VD + 4 * h : nullptr;
#pragma unroll
  for (int e = 0; e < DT * 4 / KG; ++e) {
    const int t = (kg * DT * 4 / KG + e) / 4, i = (kg * DT * 4 / KG + e) % 4;  // features 32 t + 8 i + 4 h ..
    f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < KG; ++g) a += sums[(((g * QG + qg) * DT + t) * 4 + i) * 64 + lane] * factor[g];
    a *= inv;
    if (BIASED && gt) {  // sigmoid by the hardware's exponential and reciprocal (about a unit in the last place each)
      const s16x4 gates = *reinterpret_cast<const s16x4*>(gt + 32 * t + 8 * i);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float g = __uint_as_float((unsigned)(unsigned short)gates[k] << 16);
        a[k] *= __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-g * LOG2E));
      }
    }
    s16x4 w4;
#pragma unroll
    for (int k = 0; k < 4; ++k) w4[k] = bf16_bits(a[k]);
    *reinterpret_cast<s16x4*>(o + 32 * t + 8 * i) = w4;
  }
}

template <int HD, int VD, int QG, bool CAPPED, bool BIASED>
int launch(const PrefillArgs& p, hipStream_t stream) {
  using S = Shape<HD, VD, QG>;
  const hipError_t err = hipFuncSetAttribute((const void*)attn_prefill_shared_kernel<HD, VD, QG, CAPPED, BIASED>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, S::LDS);
  PAE_REQUIRE(err == hipSuccess, "attn_prefill: %d bytes of LDS refused: %s", S::LDS, hipGetErrorString(err));
  attn_prefill_shared_kernel<HD, VD, QG, CAPPED, BIASED><<<dim3(p.nh * (PREFILL_RUN / S::TOK), p.num_tiles), 512, S::LDS, stream>>>(p);
  return pae_check_launch("attn_prefill");
}

template <int HD, int VD, int QG>
int launch_kind(const PrefillArgs& p, bool biased, hipStream_t stream) {
  if constexpr (HD == VD) {
    if (biased) return launch<HD, VD, QG, false, true>(p, stream);
    if (p.cap_over_scale > 0.f) return launch<HD, VD, QG, true, false>(p, stream);
  }
  return launch<HD, VD, QG, false, false>(p, stream);
}

}  // namespace

bool attn_prefill_shared_takes(int hd, int vd, int page_size) {
  return page_size == 16 && ((hd == 128 && vd == 128) || (hd == 64 && vd == 64) || (hd == 192 && vd == 128));
}

int attn_prefill_shared(const PrefillArgs& p, int hd, int vd, bool biased, int groups, hipStream_t stream) {
  if (hd == 128 && vd == 128) return groups == 4 ? launch_kind<128, 128, 4>(p, biased, stream) : launch_kind<128, 128, 2>(p, biased, stream);
  if (hd == 192 && vd == 128) return groups == 4 ? launch_kind<192, 128, 4>(p, biased, stream) : launch_kind<192, 128, 2>(p, biased, stream);
  if (hd == 64 && vd == 64 && groups == 2) return launch_kind<64, 64, 2>(p, biased, stream);
  return pae_fail("attn_prefill: %d query groups with keys of %d and values of %d are not built", groups, hd, vd);
}
