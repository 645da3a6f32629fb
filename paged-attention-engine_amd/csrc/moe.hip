// A feed-forward of many small gated experts, of which every token uses a few.
//
//   project_f32     float32 sums of a few output features (router logits, gate logits) from rows of either
//                   type: one wavefront an output, k shared out over its lanes in a fixed order
//   moe_route       per token: scores = softmax(logits) over all experts; the experts form `groups`
//                   equal groups of neighbours, a group's score is its largest score, only experts of the
//                   `keep` best groups can be chosen; the `top` largest scores among those are chosen,
//                   and their weights are the scores times `scale` (not renormalised).  Of equal
//                   scores the lower index wins.  With a `choice_bias` [E], experts and groups are compared
//                   by score + bias, while the weights stay the scores themselves.  With `among_chosen`
//                   instead, experts are compared by their logits and the weights are the softmax over
//                   the chosen logits alone, times `scale`.  Experts that every token uses are `shared_pieces`
//                   more entries behind the chosen ones, experts E, E + 1, ..., each weighted by the sigmoid
//                   of the logit behind the experts' own.  One wavefront a token.
//   moe_gate_up     for every (token, chosen expert): act(W_gate x) * (W_up x), rounded to the activation type
//   moe_down        for every token: sum over its chosen experts of weight * W_down act, float32
//
// A token's routing and its experts' sums depend on that token alone, so its result does not depend on
// the batch.  The two expert kernels stream every chosen expert's weights once per (token, expert) pair;
// they are the kernels for steps of a few rows.
#include "common.h"
#include "api.h"
#include "wide_gemm.h"

template <typename T>
__global__ __launch_bounds__(256) void project_f32_kernel(float* __restrict__ out, int64_t ldo, const T* __restrict__ A,
                                                          int64_t lda, const T* __restrict__ W,
                                                          const void* __restrict__ bias, int b_is_f32, int N, int K) {
  const int64_t t = blockIdx.x;
  const int n = blockIdx.y * 4 + threadIdx.x / PAE_WAVE, lane = threadIdx.x % PAE_WAVE;
  if (n >= N) return;
  const T* a = A + t * lda;
  const T* w = W + (int64_t)n * K;
  float sum = 0.f;
  for (int k = lane; k < K; k += PAE_WAVE) sum = fmaf(to_f32(a[k]), to_f32(w[k]), sum);
  sum = wave_sum(sum);
  if (lane == 0) out[t * ldo + n] = sum + (bias ? load_param(bias, b_is_f32, n) : 0.f);
}

// The same sums with 16-byte loads, for rows and widths that allow them: a workgroup takes one row and `per_wave`
// outputs for each of its four wavefronts (all of a row's outputs in steps of many rows, one each in steps of
// few); a lane adds its 8 (or 4) consecutive k of every 64-lane stretch, then the lanes meet.
template <typename T>
__global__ __launch_bounds__(256) void project_f32_wide_kernel(float* __restrict__ out, int64_t ldo, const T* __restrict__ A,
                                                               int64_t lda, const T* __restrict__ W,
                                                               const void* __restrict__ bias, int b_is_f32, int N, int K,
                                                               int per_wave) {
  constexpr int VEC = 16 / sizeof(T);
  struct alignas(16) Chunk { T v[VEC]; };
  const int64_t t = blockIdx.x;
  const int wave = threadIdx.x / PAE_WAVE, lane = threadIdx.x % PAE_WAVE;
  const T* a = A + t * lda;
  const int first = blockIdx.y * 4 * per_wave + wave;
  for (int n = first; n < N && n < first + 4 * per_wave; n += 4) {
    const T* w = W + (int64_t)n * K;
    float sum = 0.f;
    for (int k = lane * VEC; k < K; k += PAE_WAVE * VEC) {
      const Chunk x = *reinterpret_cast<const Chunk*>(a + k);
      const Chunk y = *reinterpret_cast<const Chunk*>(w + k);
#pragma unroll
      for (int i = 0; i < VEC; ++i) sum = fmaf(to_f32(x.v[i]), to_f32(y.v[i]), sum);
    }
    sum = wave_sum(sum);
    if (lane == 0) out[t * ldo + n] = sum + (bias ? load_param(bias, b_is_f32, n) : 0.f);
  }
}

// The same sums, to the bit, in steps of many bfloat16 rows of up to STEPS stretches: a workgroup takes ROWS of them, which its wavefronts hold in
// registers, so that an output's weights are fetched once for all (what bounds the kernel above there: 98 KB of weights through a unit's first
// cache for every row), the next output's on their way beside an output's sums.
template <int STEPS, int ROWS>
__global__ __launch_bounds__(256) void project_f32_rows_kernel(float* __restrict__ out, int64_t ldo, const bf16_t* __restrict__ A, int64_t lda,
                                                               const bf16_t* __restrict__ W, const void* __restrict__ bias, int b_is_f32, int M,
                                                               int N, int K) {
  struct alignas(16) Chunk { bf16_t v[8]; };
  const int t0 = blockIdx.x * ROWS, wave = threadIdx.x / PAE_WAVE, lane = threadIdx.x % PAE_WAVE;
  auto place = [&](int i) { return min(lane * 8 + i * 512, K - 8); };  // (what lies behind a row's end is read at its end and not added)
  Chunk a[ROWS][STEPS], next[STEPS];
#pragma unroll
  for (int i = 0; i < STEPS; ++i) {
    next[i] = *reinterpret_cast<const Chunk*>(W + (int64_t)min(wave, N - 1) * K + place(i));
#pragma unroll
    for (int r = 0; r < ROWS; ++r) a[r][i] = *reinterpret_cast<const Chunk*>(A + (int64_t)min(t0 + r, M - 1) * lda + place(i));
  }
  for (int n = wave; n < N; n += 4) {
    Chunk w[STEPS];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      w[i] = next[i];
      next[i] = *reinterpret_cast<const Chunk*>(W + (int64_t)min(n + 4, N - 1) * K + place(i));
    }
    float sum[ROWS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r) sum[r] = 0.f;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const bool in = lane * 8 + i * 512 < K;  // K is a multiple of 8
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float y = to_f32(w[i].v[e]);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          const float more = fmaf(to_f32(a[r][i].v[e]), y, sum[r]);
          sum[r] = in ? more : sum[r];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r) sum[r] = wave_sum(sum[r]);
    const float b = bias ? load_param(bias, b_is_f32, n) : 0.f;
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      if (lane == r && t0 + r < M) out[(int64_t)(t0 + r) * ldo + n] = sum[r] + b;
  }
}

extern "C" int pae_project_f32(int dtype, float* out, int64_t ldo, const void* A, int64_t lda, const void* W,
                               const void* bias, int b_is_f32, int M, int N, int K, hipStream_t stream) {
  PAE_REQUIRE(N > 0 && K > 0 && N <= 4 * 65535, "float32 projection: bad sizes N=%d K=%d", N, K);
  PAE_REQUIRE(ldo >= N && lda >= K, "float32 projection: row strides too small");
  PAE_REQUIRE(dtype == PAE_F32 || dtype == PAE_BF16, "float32 projection: unknown dtype code %d", dtype);
  if (M <= 0) return 0;
  const int vec = dtype == PAE_F32 ? 4 : 8;
  const bool wide = K % vec == 0 && lda % vec == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
  // (from where its workgroups are two a unit, and there are outputs enough for the held rows: 3,001 x 32 x 1,536 20.4 -> 16.0 us, 8,192 49.1 -> 35.0, 2,000 x
  // 16 x 896 6.5 -> 6.4, x 2,048 10.7 -> 9.1; but 3,001 x 2 x 2,048 3.8 and 5.9, 2,000 x 32 x 256 7.5 and 8.3, 1,500 x 33 x 1,536 13.7 and 14.4)
  if (wide && dtype == PAE_BF16 && M >= 2000 && N >= 16 && K > 512 && K <= 4 * 512) {
    constexpr int rows = 4;
    const int groups = (M + rows - 1) / rows;
#define PROJECT_ROWS(STEPS) \
  project_f32_rows_kernel<STEPS, rows><<<groups, 256, 0, stream>>>(out, ldo, (const bf16_t*)A, lda, (const bf16_t*)W, bias, b_is_f32, M, N, K)
    if (K <= 1024) PROJECT_ROWS(2);
    else if (K <= 1536) PROJECT_ROWS(3);
    else PROJECT_ROWS(4);
#undef PROJECT_ROWS
    return pae_check_launch("project_f32 (many rows)");
  }
  dim3 grid(M, (N + 3) / 4);
  const int per_wave = M >= 512 ? (N + 3) / 4 : 1;
  dim3 wide_grid(M, (N + 4 * per_wave - 1) / (4 * per_wave));
  if (dtype == PAE_F32) {
    if (wide)
      project_f32_wide_kernel<float><<<wide_grid, 256, 0, stream>>>(out, ldo, (const float*)A, lda, (const float*)W, bias, b_is_f32, N, K, per_wave);
    else
      project_f32_kernel<float><<<grid, 256, 0, stream>>>(out, ldo, (const float*)A, lda, (const float*)W, bias, b_is_f32, N, K);
  } else {
    if (wide)
      project_f32_wide_kernel<bf16_t><<<wide_grid, 256, 0, stream>>>(out, ldo, (const bf16_t*)A, lda, (const bf16_t*)W, bias, b_is_f32, N, K, per_wave);
    else
      project_f32_kernel<bf16_t><<<grid, 256, 0, stream>>>(out, ldo, (const bf16_t*)A, lda, (const bf16_t*)W, bias, b_is_f32, N, K);
  }
  return pae_check_launch("project_f32");
}

#define MOE_MAX_PER_LANE 16  // experts a lane holds: up to 1,024 experts

// The larger of two (number, place), the lower place of equal numbers, over a wavefront: in every lane.
__device__ __forceinline__ void wave_best(float& best, int& at) {
  auto meet = [&](float other, int other_at) {
    if (other > best || (other == best && other_at < at)) {
      best = other;
      at = other_at;
    }
  };
  {
    const auto v = __builtin_amdgcn_permlane32_swap(__float_as_uint(best), __float_as_uint(best), false, false);
    const auto p = __builtin_amdgcn_permlane32_swap((unsigned)at, (unsigned)at, false, false);
    best = __uint_as_float(v[0]);
    at = (int)p[0];
    meet(__uint_as_float(v[1]), (int)p[1]);
  }
  {
    const auto v = __builtin_amdgcn_permlane16_swap(__float_as_uint(best), __float_as_uint(best), false, false);
    const auto p = __builtin_amdgcn_permlane16_swap((unsigned)at, (unsigned)at, false, false);
    best = __uint_as_float(v[0]);
    at = (int)p[0];
    meet(__uint_as_float(v[1]), (int)p[1]);
  }
  meet(row_rotated<8>(best), __float_as_int(row_rotated<8>(__int_as_float(at))));
  meet(row_rotated<4>(best), __float_as_int(row_rotated<4>(__int_as_float(at))));
  meet(row_rotated<2>(best), __float_as_int(row_rotated<2>(__int_as_float(at))));
  meet(row_rotated<1>(best), __float_as_int(row_rotated<1>(__int_as_float(at))));
}

// One token's routing by one wavefront: `z` its logits (memory or LDS), `lds` [E] scores, [groups] group scores, and with
// a bias [E] what experts are compared by; `chosen` and `weights` its [top + shared_pieces] results.
template <int PER_LANE>
__device__ __forceinline__ void route_token(const float* z, float* lds, int E, int groups, int keep, int top, float scale,
                                            const float* __restrict__ choice_bias, int among_chosen, int shared_pieces,
                                            int* __restrict__ chosen, float* __restrict__ weights) {
  float* score = lds;
  float* group_score = lds + E;
  float* rank = choice_bias ? group_score + groups : score;
  const int lane = threadIdx.x % PAE_WAVE;
  float top_z = -INFINITY;
  for (int e = lane; e < E; e += PAE_WAVE) top_z = fmaxf(top_z, z[e]);
  top_z = wave_max(top_z);
  float sum = 0.f;
  for (int e = lane; e < E; e += PAE_WAVE) {
    const float p = among_chosen ? z[e] : expf(z[e] - top_z);
    score[e] = p;
    sum += p;
  }
  sum = wave_sum(sum);
  if (choice_bias)
    for (int e = lane; e < E; e += PAE_WAVE) rank[e] = score[e] / sum + choice_bias[e];
  __syncthreads();
  const int per_group = E / groups;
  for (int g = lane; g < groups; g += PAE_WAVE) {
    float best = -INFINITY;
    for (int j = 0; j < per_group; ++j) best = fmaxf(best, rank[g * per_group + j]);
    group_score[g] = best;
  }
  __syncthreads();
  // an expert may be chosen if fewer than `keep` groups come before its own (a larger score, or an equal one
  // at a lower index)
  float mine[PER_LANE];
#pragma unroll
  for (int j = 0; j < PER_LANE; ++j) {
    const int e = lane + PAE_WAVE * j;
    mine[j] = -INFINITY;
    if (e < E) {
      const int g = e / per_group;
      const float gs = group_score[g];
      int before = 0;
      for (int o = 0; o < groups; ++o) before += (group_score[o] > gs || (group_score[o] == gs && o < g)) ? 1 : 0;
      if (before < keep) mine[j] = rank[e];
    }
  }
  float kept = 0.f;
  int kept_at = 0;
  float first = 0.f, total = 0.f;  // among_chosen: the largest chosen logit, and the sum of exponentials against it
  for (int r = 0; r < top; ++r) {
    float best = -INFINITY;
    int at = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j)
      if (mine[j] > best) {  // a lane's experts ascend with j: the first of equals stays
        best = mine[j];
        at = lane + PAE_WAVE * j;
      }
    wave_best(best, at);
    if (at >= E) at = 0;  // no logit compares (not a number): an index that exists
    if (r == 0) first = best;
    const float e = among_chosen ? expf(best - first) : 0.f;
    total += e;
    if (lane == r % PAE_WAVE) {  // held until the sum is known; more than 64 choices are written as they come
      kept_at = at;
      kept = among_chosen ? e : score[at] / sum * scale;
      if (top > PAE_WAVE) {
        chosen[r] = kept_at;
        weights[r] = kept;
      }
    }
#pragma unroll
    for (int j = 0; j < PER_LANE; ++j)
      if (lane + PAE_WAVE * j == at) mine[j] = -INFINITY;
  }
  if (top <= PAE_WAVE && lane < top) {
    chosen[lane] = kept_at;
    weights[lane] = among_chosen ? kept / total * scale : kept;
  }
  if (top > PAE_WAVE && among_chosen)  // each lane its own numbers of the loop above
    for (int r = lane; r < top; r += PAE_WAVE) weights[r] = weights[r] / total * scale;
  if (lane != 0) return;
  for (int p = 0; p < shared_pieces; ++p) {
    chosen[top + p] = E + p;
    weights[top + p] = 1.0f / (1.0f + expf(-z[E]));
  }
}

template <int PER_LANE>
__global__ __launch_bounds__(PAE_WAVE) void moe_route_kernel(const float* __restrict__ logits, int E, int groups, int keep,
                                                             int top, float scale, const float* __restrict__ choice_bias,
                                                             int64_t ldz, int among_chosen, int shared_pieces,
                                                             int* __restrict__ chosen, float* __restrict__ weights) {
  extern __shared__ float lds[];
  const int64_t t = blockIdx.x, places = top + shared_pieces;
  route_token<PER_LANE>(logits + t * ldz, lds, E, groups, keep, top, scale, choice_bias, among_chosen, shared_pieces,
                        chosen + t * places, weights + t * places);
}

// Logits and routing of a token in one workgroup, for steps of a few tokens (two launches of a few microseconds' work
// before): the sums of project_f32_wide_kernel, five outputs of a wavefront on their way together, to LDS, then the
// first wavefront routes.  7 rows, 32 experts, 1,536 wide: 7.0 + 5.8 -> 7.9 us.
template <typename T, int PER_LANE>
__global__ __launch_bounds__(512) void moe_choose_kernel(const T* __restrict__ A, int64_t lda, const T* __restrict__ W,
                                                         const void* __restrict__ bias, int b_is_f32, int N, int K, int E,
                                                         int groups, int keep, int top, float scale,
                                                         const float* __restrict__ choice_bias, int among_chosen,
                                                         int shared_pieces, int* __restrict__ chosen,
                                                         float* __restrict__ weights) {
  constexpr int VEC = 16 / sizeof(T), OUTS = 5;  // (eight wavefronts: up to 40 outputs side by side)
  struct alignas(16) Chunk { T v[VEC]; };
  extern __shared__ float lds[];  // [N] logits, then route_token's
  const int64_t t = blockIdx.x, places = top + shared_pieces;
  const int wave = threadIdx.x / PAE_WAVE, lane = threadIdx.x % PAE_WAVE;
  const T* a = A + t * lda;
  for (int first = wave * OUTS; first < N; first += 8 * OUTS) {
    float sum[OUTS];
#pragma unroll
    for (int o = 0; o < OUTS; ++o) sum[o] = 0.f;
    for (int k = lane * VEC; k < K; k += PAE_WAVE * VEC) {
      const Chunk x = *reinterpret_cast<const Chunk*>(a + k);
      Chunk y[OUTS];
#pragma unroll
      for (int o = 0; o < OUTS; ++o) y[o] = *reinterpret_cast<const Chunk*>(W + (int64_t)min(first + o, N - 1) * K + k);
#pragma unroll
      for (int o = 0; o < OUTS; ++o)
#pragma unroll
        for (int i = 0; i < VEC; ++i) sum[o] = fmaf(to_f32(x.v[i]), to_f32(y[o].v[i]), sum[o]);
    }
#pragma unroll
    for (int o = 0; o < OUTS; ++o) {
      sum[o] = wave_sum(sum[o]);
      if (lane == 0 && first + o < N) lds[first + o] = sum[o] + (bias ? load_param(bias, b_is_f32, first + o) : 0.f);
    }
  }
  __syncthreads();
  if (wave > 0) return;  // (a barrier counts the wavefronts that are left)
  route_token<PER_LANE>(lds, lds + N, E, groups, keep, top, scale, choice_bias, among_chosen, shared_pieces,
                        chosen + t * places, weights + t * places);
}

static int check_route(int experts, int groups, int keep, int top, const float* choice_bias, int among_chosen, int shared_pieces) {
  PAE_REQUIRE(shared_pieces >= 0, "routing: %d shared pieces", shared_pieces);
  PAE_REQUIRE(!among_chosen || (groups == 1 && !choice_bias), "routing: a softmax over the chosen logits goes with one group and no choice bias");
  PAE_REQUIRE(experts > 0 && experts <= PAE_WAVE * MOE_MAX_PER_LANE, "routing: %d experts (1..%d)", experts,
              PAE_WAVE * MOE_MAX_PER_LANE);
  PAE_REQUIRE(groups > 0 && experts % groups == 0 && keep > 0 && keep <= groups, "routing: %d groups of %d experts, %d kept",
              groups, experts, keep);
  PAE_REQUIRE(top > 0 && top <= keep * (experts / groups), "routing: %d experts chosen of %d that can be", top,
              keep * (experts / groups));
  return 0;
}

// Whether pae_moe_choose takes rows of A: a few (above, the two kernels by themselves have workgroups enough), read 16 bytes
// at a time.
extern "C" int pae_moe_choose_takes(int dtype, const void* A, int64_t lda, const void* W, int M, int K) {
  const int vec = dtype == PAE_F32 ? 4 : 8;
  return M <= 256 && K % vec == 0 && lda % vec == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
}

// Whether it is ahead of the two launches for a router of N rows of K: all of them pass one workgroup, which has up to 40 outputs
// on their way side by side, where the projection by itself spreads them over N / 4 workgroups.  One launch / two, 12 rows: 32 x 1,536 in
// bfloat16 8.6 / 9.1 us, 40 x 1,536 8.9 / 9.4, 32 x 2,560 9.2 / 9.5, 41 x 1,536 9.9 / 9.6, 64 x 1,024 10.6 / 10.0, 8 x 7,168 10.6 / 10.3, 128 x
// 2,048 19.3 / 14.2, 256 x 7,168 66 / 25.
extern "C" int pae_moe_choose_pays(int dtype, int N, int K) { return N <= 40 && (int64_t)K * (dtype == PAE_F32 ? 4 : 2) <= 5120; }

// pae_project_f32 and pae_moe_route in one launch: W [experts (+ 1 with shared pieces)][K], bias or null.
extern "C" int pae_moe_choose(int dtype, const void* A, int64_t lda, const void* W, const void* bias, int b_is_f32, int M,
                              int K, int experts, int groups, int keep, int top, float scale, const float* choice_bias,
                              int among_chosen, int shared_pieces, int* chosen, float* weights, hipStream_t stream) {
  if (int rc = check_route(experts, groups, keep, top, choice_bias, among_chosen, shared_pieces)) return rc;
  PAE_REQUIRE(dtype == PAE_F32 || dtype == PAE_BF16, "routing: unknown dtype code %d", dtype);
  PAE_REQUIRE(K > 0 && lda >= K && pae_moe_choose_takes(dtype, A, lda, W, M, K), "routing: %d rows of %d, %lld apart", M, K, (long long)lda);
  if (M <= 0) return 0;
  const int N = experts + (shared_pieces > 0 ? 1 : 0);
  const size_t lds = (size_t)(N + experts + groups + (choice_bias ? experts : 0)) * sizeof(float);
#define MOE_CHOOSE(T, PER_LANE)                                                                                       \
  moe_choose_kernel<T, PER_LANE><<<M, 512, lds, stream>>>((const T*)A, lda, (const T*)W, bias, b_is_f32, N, K, experts, \
                                                          groups, keep, top, scale, choice_bias, among_chosen,        \
                                                          shared_pieces, chosen, weights)
#define MOE_CHOOSE_ANY(T)                               \
  if (experts <= PAE_WAVE) MOE_CHOOSE(T, 1);            \
  else if (experts <= 4 * PAE_WAVE) MOE_CHOOSE(T, 4);   \
  else MOE_CHOOSE(T, MOE_MAX_PER_LANE);
  if (dtype == PAE_F32) {
    MOE_CHOOSE_ANY(float)
  } else {
    MOE_CHOOSE_ANY(bf16_t)
  }
#undef MOE_CHOOSE_ANY
#undef MOE_CHOOSE
  return pae_check_launch("moe_choose");
}

extern "C" int pae_moe_route(const float* logits, int num_tokens, int experts, int groups, int keep, int top, float scale,
                             const float* choice_bias, int64_t ldz, int among_chosen, int shared_pieces, int* chosen,
                             float* weights, hipStream_t stream) {
  PAE_REQUIRE(ldz >= experts + (shared_pieces > 0 ? 1 : 0) && shared_pieces >= 0, "routing: rows of %lld logits for %d experts and %d shared pieces",
              (long long)ldz, experts, shared_pieces);
  if (int rc = check_route(experts, groups, keep, top, choice_bias, among_chosen, shared_pieces)) return rc;
  if (num_tokens <= 0) return 0;
  const size_t lds = (size_t)(experts + groups + (choice_bias ? experts : 0)) * sizeof(float);
#define MOE_ROUTE(PER_LANE)                                                                                            \
  moe_route_kernel<PER_LANE><<<num_tokens, PAE_WAVE, lds, stream>>>(logits, experts, groups, keep, top, scale, choice_bias, ldz, \
                                                                    among_chosen, shared_pieces, chosen, weights)
  if (experts <= PAE_WAVE) MOE_ROUTE(1);
  else if (experts <= 4 * PAE_WAVE) MOE_ROUTE(4);
  else MOE_ROUTE(MOE_MAX_PER_LANE);
#undef MOE_ROUTE
  return pae_check_launch("moe_route");
}

// One workgroup of four wavefronts per (pair, 16 features of the expert's width): a wavefront takes four
// features in turn, its lanes share out the hidden width.
template <typename T>
__global__ __launch_bounds__(256) void moe_gate_up_kernel(T* __restrict__ act, const T* __restrict__ x, int64_t ldx,
                                                          const T* __restrict__ gate_w, const T* __restrict__ up_w,
                                                          const int* __restrict__ chosen, int top, int hidden, int inter,
                                                          int act_kind) {
  const int64_t pair = blockIdx.x;
  const int e = chosen[pair];
  const T* row = x + (pair / top) * ldx;
  const int wave = threadIdx.x / PAE_WAVE, lane = threadIdx.x % PAE_WAVE;
  for (int j = 0; j < 4; ++j) {
    const int f = blockIdx.y * 16 + wave * 4 + j;
    if (f >= inter) return;
    const T* g = gate_w + ((int64_t)e * inter + f) * hidden;
    const T* u = up_w + ((int64_t)e * inter + f) * hidden;
    float gs = 0.f, us = 0.f;
    for (int k = lane; k < hidden; k += PAE_WAVE) {
      const float xv = to_f32(row[k]);
      gs = fmaf(xv, to_f32(g[k]), gs);
      us = fmaf(xv, to_f32(u[k]), us);
    }
    gs = wave_sum(gs);
    us = wave_sum(us);
    // the gate is applied to the float32 sums and the product rounded once
    if (lane == 0) act[pair * inter + f] = from_f32<T>(act_of(gs, act_kind) * us);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void moe_down_kernel(float* __restrict__ out, const T* __restrict__ act,
                                                       const T* __restrict__ down_w, const int* __restrict__ chosen,
                                                       const float* __restrict__ weights, int top, int hidden, int inter) {
  const int64_t t = blockIdx.x;
  const int wave = threadIdx.x / PAE_WAVE, lane = threadIdx.x % PAE_WAVE;
  for (int j = 0; j < 4; ++j) {
    const int n = blockIdx.y * 16 + wave * 4 + j;
    if (n >= hidden) return;
    float total = 0.f;
    for (int r = 0; r < top; ++r) {
      const int e = chosen[t * top + r];
      const T* w = down_w + ((int64_t)e * hidden + n) * inter;
      const T* a = act + (t * top + r) * inter;
      float sum = 0.f;
      for (int k = lane; k < inter; k += PAE_WAVE) sum = fmaf(to_f32(a[k]), to_f32(w[k]), sum);
      total = fmaf(weights[t * top + r], wave_sum(sum), total);
    }
    if (lane == 0) out[t * hidden + n] = total;
  }
}

extern "C" int pae_moe_gate_up(int dtype, void* act, const void* x, int64_t ldx, const void* gate_w, const void* up_w,
                               const int* chosen, int num_tokens, int top, int hidden, int inter, int act_kind,
                               hipStream_t stream) {
  PAE_REQUIRE(top > 0 && hidden > 0 && inter > 0 && ldx >= hidden, "experts: bad sizes top=%d H=%d F=%d", top, hidden, inter);
  PAE_REQUIRE((inter + 15) / 16 <= 65535, "experts: width %d exceeds the grid", inter);
  if (num_tokens <= 0) return 0;
  dim3 grid(num_tokens * top, (inter + 15) / 16);
  if (dtype == PAE_F32)
    moe_gate_up_kernel<float><<<grid, 256, 0, stream>>>((float*)act, (const float*)x, ldx, (const float*)gate_w,
                                                        (const float*)up_w, chosen, top, hidden, inter, act_kind);
  else if (dtype == PAE_BF16)
    moe_gate_up_kernel<bf16_t><<<grid, 256, 0, stream>>>((bf16_t*)act, (const bf16_t*)x, ldx, (const bf16_t*)gate_w,
                                                         (const bf16_t*)up_w, chosen, top, hidden, inter, act_kind);
  else
    return pae_fail("experts: unknown dtype code %d", dtype);
  return pae_check_launch("moe_gate_up");
}

extern "C" int pae_moe_down(int dtype, float* out, const void* act, const void* down_w, const int* chosen,
                            const float* weights, int num_tokens, int top, int hidden, int inter, hipStream_t stream) {
  PAE_REQUIRE(top > 0 && hidden > 0 && inter > 0, "experts: bad sizes top=%d H=%d F=%d", top, hidden, inter);
  PAE_REQUIRE((hidden + 15) / 16 <= 65535, "experts: width %d exceeds the grid", hidden);
  if (num_tokens <= 0) return 0;
  dim3 grid(num_tokens, (hidden + 15) / 16);
  if (dtype == PAE_F32)
    moe_down_kernel<float><<<grid, 256, 0, stream>>>(out, (const float*)act, (const float*)down_w, chosen, weights, top,
                                                     hidden, inter);
  else if (dtype == PAE_BF16)
    moe_down_kernel<bf16_t><<<grid, 256, 0, stream>>>(out, (const bf16_t*)act, (const bf16_t*)down_w, chosen, weights, top,
                                                      hidden, inter);
  else
    return pae_fail("experts: unknown dtype code %d", dtype);
  return pae_check_launch("moe_down");
}

// ---------------------------------------------------------------------------------------------------------------
// The experts on the matrix cores (bfloat16, widths in multiples of 32).  The (token, expert) pairs of a step are
// sorted by expert on the device, and every expert's pairs are cut into tiles of up to 16 MT rows; a workgroup takes one
// tile and 64 or more output features, its four wavefronts a quarter each, so an expert's weights are streamed once per
// tile: once in all for a step of a few tokens, and once per 16 MT of an expert's tokens in a prompt.  Which tile a
// pair falls into changes nothing of its sums (k ascends in steps of 32 for every row by itself), so a token's
// result does not depend on the batch.
//
//   moe_sort            counts, offsets and tiles by expert (one workgroup; the order of an expert's pairs among
//                       themselves is whatever the counters' turn gives, and does not matter)
//   gate/up             act(W_gate x) * (W_up x) for a tile's rows, rounded, to rows in sorted order
//   down                weight * W_down act for a tile's rows, float32, to y[chosen place][token]: the `top` places
//                       of a token are float32 partial sums that the stream's next norm adds in order
// each in three kernels by the step's size: moe_few_tiles (up to 512 pairs), moe_tiles_gate_up / moe_tiles_down (up to
// 4,096), moe_big_tiles (above).
using wide_gemm::bf16x8;
using wide_gemm::f32x4;

__global__ __launch_bounds__(1024) void moe_sort_kernel(const int* __restrict__ chosen, int pairs, int experts, int tile_rows,
                                                        int* __restrict__ order, int4* __restrict__ tiles, int max_tiles) {
  extern __shared__ int sorted_lds[];  // [experts] counts, starts, cursors, first tiles; [1] tiles in all
  int* count = sorted_lds;
  int* start = count + experts;
  int* cursor = start + experts;
  int* first_tile = cursor + experts;
  int* total = first_tile + experts;
  for (int e = threadIdx.x; e < experts; e += 1024) count[e] = cursor[e] = 0;
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += 1024) atomicAdd(&count[chosen[p]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int rows = 0, tile = 0;
    for (int e = 0; e < experts; ++e) {
      start[e] = rows;
      first_tile[e] = tile;
      rows += count[e];
      tile += (count[e] + tile_rows - 1) / tile_rows;
    }
    *total = tile;
  }
  __syncthreads();
  for (int p = threadIdx.x; p < pairs; p += 1024) {
    const int e = chosen[p];
    order[start[e] + atomicAdd(&cursor[e], 1)] = p;
  }
  for (int e = threadIdx.x; e < experts; e += 1024)
    for (int j = 0; j * tile_rows < count[e]; ++j)
      tiles[first_tile[e] + j] = make_int4(e, start[e] + j * tile_rows, min(tile_rows, count[e] - j * tile_rows),
                                           j << 16 | ((count[e] + tile_rows - 1) / tile_rows & 0xffff));
  for (int i = *total + threadIdx.x; i < max_tiles; i += 1024) tiles[i] = make_int4(0, 0, 0, 0);
  if (threadIdx.x == 0) tiles[max_tiles] = make_int4(*total, 0, 0, 0);
}

// A wavefront holds MT tiles of 16 rows by NT tiles of 16 features: MT + NT (2 NT with gate and up) operand loads
// feed MT NT (2 MT NT) matrix instructions in every step of 32 of k.
template <int MT, int NT>
__global__ __launch_bounds__(256) void moe_tiles_gate_up_kernel(bf16_t* __restrict__ act, const bf16_t* __restrict__ x,
                                                                int64_t ldx, const bf16_t* __restrict__ gate_w,
                                                                const bf16_t* __restrict__ up_w, const int* __restrict__ order,
                                                                const int4* __restrict__ tiles, int top, int hidden, int inter,
                                                                int act_kind) {
  const int4 tile = tiles[blockIdx.x];  // (expert, first sorted row, rows, unused)
  const int lane = threadIdx.x % PAE_WAVE, wave = threadIdx.x / PAE_WAVE;
  const int col = lane % 16, kg = lane / 16;
  const int f0 = (blockIdx.y * 4 + wave) * 16 * NT;
  if (tile.z <= 0 || f0 >= inter) return;
  const bf16_t* gw[NT];
  const bf16_t* uw[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int64_t w_row = (int64_t)tile.x * inter + min(f0 + 16 * nt + col, inter - 1);
    gw[nt] = gate_w + w_row * hidden + 8 * kg;
    uw[nt] = up_w + w_row * hidden + 8 * kg;
  }
  const bf16_t* rows[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + col;
    rows[mt] = x + (int64_t)(order[tile.y + (r < tile.z ? r : 0)] / top) * ldx + 8 * kg;
  }
  f32x4 gs[MT][NT], us[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) gs[mt][nt] = us[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // operands of the step after are on their way while a step's matrix instructions run; the loop's loads are
  // unconditional and the last step stands by itself
  bf16x8 g[2][NT], u[2][NT], a[2][MT];
  auto load = [&](int set, int k) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      g[set][nt] = *reinterpret_cast<const bf16x8*>(gw[nt] + k);
      u[set][nt] = *reinterpret_cast<const bf16x8*>(uw[nt] + k);
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) a[set][mt] = *reinterpret_cast<const bf16x8*>(rows[mt] + k);
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        gs[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g[set][nt], a[set][mt], gs[mt][nt], 0, 0, 0);
        us[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(u[set][nt], a[set][mt], us[mt][nt], 0, 0, 0);
      }
  };
  load(0, 0);
  int k = 0;
  for (; k + 64 < hidden; k += 64) {
    load(1, k + 32);
    multiply(0);
    load(0, k + 64);
    multiply(1);
  }
  if (k + 32 < hidden) {
    load(1, k + 32);
    multiply(0);
    multiply(1);
  } else {
    multiply(0);
  }
  // a lane holds features f0 + 16 nt + 4 kg .. + 3 of the row mt * 16 + col
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + col;
    if (r >= tile.z) continue;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int f = f0 + 16 * nt + 4 * kg;
      bf16_t* o = act + (int64_t)(tile.y + r) * inter + f;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (f + i < inter) o[i] = __float2bfloat16(act_to<bf16_t>(gs[mt][nt][i], act_kind) * us[mt][nt][i]);
    }
  }
}

template <int MT, int NT>
__global__ __launch_bounds__(256) void moe_tiles_down_kernel(float* __restrict__ y, const bf16_t* __restrict__ act,
                                                             const bf16_t* __restrict__ down_w, const int* __restrict__ order,
                                                             const float* __restrict__ weights, const int4* __restrict__ tiles,
                                                             int top, int num_tokens, int hidden, int inter) {
  const int4 tile = tiles[blockIdx.x];
  const int lane = threadIdx.x % PAE_WAVE, wave = threadIdx.x / PAE_WAVE;
  const int col = lane % 16, kg = lane / 16;
  const int n0 = (blockIdx.y * 4 + wave) * 16 * NT;
  if (tile.z <= 0 || n0 >= hidden) return;
  const bf16_t* w[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    w[nt] = down_w + ((int64_t)tile.x * hidden + min(n0 + 16 * nt + col, hidden - 1)) * inter + 8 * kg;
  const bf16_t* rows[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + col;
    rows[mt] = act + (int64_t)(tile.y + (r < tile.z ? r : 0)) * inter + 8 * kg;
  }
  f32x4 sums[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) sums[mt][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 wk[2][NT], a[2][MT];
  auto load = [&](int set, int k) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) wk[set][nt] = *reinterpret_cast<const bf16x8*>(w[nt] + k);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) a[set][mt] = *reinterpret_cast<const bf16x8*>(rows[mt] + k);
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        sums[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wk[set][nt], a[set][mt], sums[mt][nt], 0, 0, 0);
  };
  load(0, 0);
  int k = 0;
  for (; k + 64 < inter; k += 64) {
    load(1, k + 32);
    multiply(0);
    load(0, k + 64);
    multiply(1);
  }
  if (k + 32 < inter) {
    load(1, k + 32);
    multiply(0);
    multiply(1);
  } else {
    multiply(0);
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = mt * 16 + col;
    if (r >= tile.z) continue;
    const int pair = order[tile.y + r];
    const float weight = weights[pair];
    float* row = y + ((int64_t)(pair % top) * num_tokens + pair / top) * hidden;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const int n = n0 + 16 * nt + 4 * kg;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (n + i < hidden) row[n + i] = weight * sums[mt][nt][i];
    }
  }
}

// The two products for steps of up to 512 pairs (decode steps, small portions), where an expert sees at most a few
// tokens and its weights are streamed exactly once: a tile is up to 16 rows, and the four wavefronts of a workgroup share
// one tile of 16 features and take a quarter of k each, leave their sums in LDS, and the first adds them in wavefront
// order (a wavefront per 16 features and the whole of k was measured against it: 35 + 22 us against 25 + 14 at one
// token, 85 + 57 against 67 + 39 at eight).  The order of adding is a function of the sizes alone.  A wavefront asks for
// two steps of 32 at once and works on the two before: a row's lines are whole in one batch (a step has half of
// each), and five wavefronts a SIMD or more are resident.  Four steps at once take 128 registers where two take 80, and the chip then
// has too few wavefronts: 8 tokens by four of 32 experts, 1,536 x 2,240, both products, one step 112, two 94, four 101 us; 16 by
// eight of 128, 2,048 x 768, 179, 158 and 186; 24 by eight of 256, 2,048 x 512, 196, 181 and 216.  The weights' stream bounds it.
//
// In steps of up to 32 tokens and 256 pairs no sorting comes first: a workgroup looks its expert's pairs up itself, in their
// order (two barriers, against a launch of 6 us, 30 with 256 experts, and the same trip to memory for the tile);
// activations lie at their pair's number.  Nothing is assumed about how often a token names an expert: routing names one
// several times where no logit compares.
//   BY_PAIR    blockIdx.x is a pair; the workgroup takes the sixteen of its expert's pairs that begins with it, if one does
//   BY_EXPERT  blockIdx.x is an expert; the workgroups along blockIdx.z take its sixteens in turn
// What either costs over the weights' stream is its workgroups without work, so the list with fewer of them is taken:
// pairs up to the number of experts, else experts.  Sorted / by pair / by expert: 1 token by eight of 256 68 / 21 / 33 us, 16 by eight of
// 128 164 / 158 / 157, 16 by four of 32 117 / 116 / 112, 32 by four of 32 138 / 146 / 132.
enum { SORTED, BY_PAIR, BY_EXPERT };
template <bool GATED, int LIST>
__global__ __launch_bounds__(256) void moe_few_tiles_kernel(bf16_t* __restrict__ act_out, float* __restrict__ y,
                                                            const bf16_t* __restrict__ a_rows, int64_t lda,
                                                            const bf16_t* __restrict__ w_first, const bf16_t* __restrict__ w_second,
                                                            const int* __restrict__ order, const float* __restrict__ weights,
                                                            const int4* __restrict__ tiles, int experts, int top, int num_tokens,
                                                            int K, int N, int act_kind) {
  constexpr int BATCH = 2;
  __shared__ f32x4 parts[3][2][PAE_WAVE];
  __shared__ int pair_of[16];
  __shared__ uint64_t of_wave[4];
  const int lane = threadIdx.x % PAE_WAVE, wave = threadIdx.x / PAE_WAVE;
  const int col = lane % 16, kg = lane / 16;
  const int n0 = blockIdx.y * 16;
  int4 tile;  // (expert, first sorted row, rows <= 16, unused)
  int place = -1, from = 0, all = 0;  // this thread's pair among its expert's, where the sixteen begins, how many there are
  if (LIST == SORTED) {
    tile = tiles[blockIdx.x];
    if (tile.z <= 0) return;
  } else {  // order: the pairs' experts
    const int self = blockIdx.x, pairs = num_tokens * top;
    const int expert = LIST == BY_PAIR ? order[min(self, pairs - 1)] : self;
    const bool mine = (int)threadIdx.x < pairs && order[threadIdx.x] == expert;
    const uint64_t found = __ballot(mine);
    if (lane == 0) of_wave[wave] = found;
    __syncthreads();
    int before = 0;  // of the expert's pairs, those of the wavefronts before
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint64_t there = of_wave[w];
      const int ahead = self - w * PAE_WAVE;  // of the wavefront's pairs, those before the workgroup's own
      if (w < wave) before += __popcll(there);
      if (LIST == BY_PAIR) from += __popcll(ahead >= PAE_WAVE ? there : ahead > 0 ? there & ((1ull << ahead) - 1) : 0);
      all += __popcll(there);
    }
    if (LIST == BY_EXPERT) from = blockIdx.z * 16;
    if ((LIST == BY_PAIR && self >= pairs) || from % 16 || from >= all || (unsigned)expert >= (unsigned)experts) return;
    if (mine) place = before + __popcll(found & ((1ull << lane) - 1));
    tile = make_int4(expert, 0, 0, 0);
  }
  if (n0 >= N) return;
  while (true) {  // (once, but BY_EXPERT)
    if (LIST != SORTED) {
      tile.z = min(16, all - from);
      if (place >= from && place < from + 16) pair_of[place - from] = threadIdx.x;
      __syncthreads();
    }
    const int sorted = LIST != SORTED ? pair_of[col < tile.z ? col : 0] : tile.y + (col < tile.z ? col : 0);
    const int pair = LIST != SORTED ? sorted : order[sorted];  // where a result goes: row `sorted` of the activations, the pair's of y
    const int64_t w_row = (int64_t)tile.x * N + min(n0 + col, N - 1);
    const bf16_t* w1 = w_first + w_row * K + 8 * kg;
    const bf16_t* w2 = GATED ? w_second + w_row * K + 8 * kg : nullptr;
    const bf16_t* a = a_rows + (int64_t)(GATED ? pair / top : sorted) * lda + 8 * kg;
    const int steps = K / 32, per = (steps + 3) / 4;
    const int first = wave * per, last = min(steps, first + per);
    f32x4 s1 = {0.f, 0.f, 0.f, 0.f}, s2 = {0.f, 0.f, 0.f, 0.f};
    const auto load = [](const bf16_t* p) { return *reinterpret_cast<const bf16x8*>(p); };
    bf16x8 ca[BATCH], c1[BATCH], c2[BATCH], na[BATCH], n1[BATCH], n2[BATCH];
    const int batches = (last - first) / BATCH;
    if (batches > 0) {
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        c1[i] = load(w1 + 32 * (first + i));
        if (GATED) c2[i] = load(w2 + 32 * (first + i));
      }
#pragma unroll
      for (int i = 0; i < BATCH; ++i) ca[i] = load(a + 32 * (first + i));
    }
    for (int b = 0; b < batches; ++b) {
      const int next = first + BATCH * min(b + 1, batches - 1);  // (the last batch asks for its own lines again)
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        n1[i] = load(w1 + 32 * (next + i));
        if (GATED) n2[i] = load(w2 + 32 * (next + i));
      }
#pragma unroll
      for (int i = 0; i < BATCH; ++i) na[i] = load(a + 32 * (next + i));
      __builtin_amdgcn_sched_barrier(0);  // (asked for before the products, or the loads would sink behind them)
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c1[i], ca[i], s1, 0, 0, 0);
        if (GATED) s2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(c2[i], ca[i], s2, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < BATCH; ++i) {
        ca[i] = na[i]; c1[i] = n1[i];
        if (GATED) c2[i] = n2[i];
      }
    }
    for (int st = first + batches * BATCH; st < last; ++st) {
      const bf16x8 x = load(a + 32 * st), g = load(w1 + 32 * st);
      s1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g, x, s1, 0, 0, 0);
      if (GATED) s2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(load(w2 + 32 * st), x, s2, 0, 0, 0);
    }
    if (wave > 0) {
      parts[wave - 1][0][lane] = s1;
      if (GATED) parts[wave - 1][1][lane] = s2;
    }
    __syncthreads();
    if (wave == 0 && col < tile.z) {
#pragma unroll
      for (int w = 0; w < 3; ++w) {
        s1 += parts[w][0][lane];
        if (GATED) s2 += parts[w][1][lane];
      }
      const int n = n0 + 4 * kg;  // a lane holds features n .. n + 3 of the row col
      if (GATED) {
        bf16_t* o = act_out + (int64_t)sorted * N + n;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) o[i] = __float2bfloat16(act_to<bf16_t>(s1[i], act_kind) * s2[i]);
      } else {
        const float weight = weights[pair];
        float* o = y + ((int64_t)(pair % top) * num_tokens + pair / top) * N + n;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (n + i < N) o[i] = weight * s1[i];
      }
    }
    from += 16 * gridDim.z;
    if (LIST != BY_EXPERT || from >= all) return;
    // (every wavefront has read its pairs, and the first one reads the sums before it comes to the next barrier)
  }
}

// The same two products for prompts, where an expert sees hundreds of tokens: a workgroup takes a tile of 128 rows
// and 128 features with gate and up (or 256 output features of the down product) through the loop of wide_gemm.h, eight wavefronts of
// 64 x 64.  What bounds it: LDS and the lines that a compute unit takes in (wide_gemm.h), so what a workgroup's neighbours
// on the die bring to its L2 counts, and padding: experts see a few hundred rows each.  Measured, 3,001 tokens by four of 32
// experts, 1,536 x 2,240 (165 and 83 GFLOP): with operands through registers, two barriers a stage of 64 of k and
// one workgroup's features after another 594 and 298 us; four wavefronts of 64 x 128 through LDS 382 and 172; with an expert's
// tiles side by side on one die 318 and 140 (three quarters of the lines from L2); with the loads spread among
// the products 306 and 127 us (540 and 650 TFLOP/s); eight wavefronts of 64 x 64, two a
// SIMD, 243 and 121 us (680 TFLOP/s both); the activation as an argument of the template, and worked out as act_to does, both products 384 -> 359 us
// (378 with its code looked at for every number).
typedef wide_gemm::Tile<128, 256, 2, 4, 3> MoeTile;
#define MOE_BIG_ROWS MoeTile::BM
#define MOE_BIG_K wide_gemm::BK
// ACT: the activation's code, an argument of the template as in gemm_wide.hip's epilogue; -1: any, by `act_kind`.
template <bool GATED, int ACT>
__global__ __launch_bounds__(512, 1) void moe_big_tiles_kernel(bf16_t* __restrict__ act_out, float* __restrict__ y,
                                                               const bf16_t* __restrict__ a_rows, int64_t lda,
                                                               const bf16_t* __restrict__ w_first, const bf16_t* __restrict__ w_second,
                                                               const int* __restrict__ order, const float* __restrict__ weights,
                                                               const int4* __restrict__ tiles, int max_tiles, int top,
                                                               int num_tokens, int K, int N, int act_kind) {
  // GATED: a_rows = x (row of a pair = its token), w_first / w_second = gate / up [E][N][K], N = the experts' width;
  // else: a_rows = act in sorted order, w_first = down [E][N][K], N = the hidden width
  extern __shared__ __attribute__((aligned(16))) char big_lds[];
  constexpr int FEATURES = GATED ? 128 : 256;  // output features a workgroup takes
  // Workgroups i, i + 8, i + 16, ... run on one die: they take an eighth of the work in a row, in which an expert's
  // tiles of one block of features follow one another, so that what they share comes to the die's L2 once.
  const int blocks = (N + FEATURES - 1) / FEATURES, total = tiles[max_tiles].x * blocks;
  const int per = (total + 7) / 8, place = blockIdx.x / 8 < per ? blockIdx.x % 8 * per + blockIdx.x / 8 : total;
  if (place >= total) return;
  const int some = place / blocks, mine = tiles[some].w;  // a tile of the expert, its number among the expert's << 16 | how many
  const int first = some - (mine >> 16), within = place - first * blocks;
  const int4 tile = tiles[first + within % (mine & 0xffff)];  // (expert, first sorted row, rows, as above)
  const int n_base = within / (mine & 0xffff) * FEATURES;
  const int lane = threadIdx.x % PAE_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  const int col = lane % 16, kg = lane / 16;
  const int wm = wave / MoeTile::WN, wn = wave % MoeTile::WN;
  MoeTile::Source src;
  src.a = reinterpret_cast<const char*>(a_rows);
  // A wavefront's 64 rows of W in LDS are, gated, 32 of gate's features and the same 32 of up's; a wavefront brings 32 rows
  static_assert(MoeTile::W_LOADS * 8 == 32 && MoeTile::PN == 64, "a wavefront brings rows of one of the two");
  const bf16_t* w = (GATED && wave % 2) ? w_second : w_first;
  src.w = reinterpret_cast<const char*>(w + (int64_t)__builtin_amdgcn_readfirstlane(tile.x) * N * K);
#pragma unroll
  for (int j = 0; j < MoeTile::A_LOADS; ++j) {
    const int r = (wave * MoeTile::A_LOADS + j) * 8 + lane / 8;
    const int sorted = tile.y + (r < tile.z ? r : 0);
    src.a_off[j] = (uint32_t)((GATED ? order[sorted] / top : sorted) * lda * 2) + wide_gemm::piece_of(lane, r);
  }
#pragma unroll
  for (int j = 0; j < MoeTile::W_LOADS; ++j) {
    const int r = (wave * MoeTile::W_LOADS + j) * 8 + lane / 8;
    // gated: row q of group x (of two) holds feature q / 4 * 8 + x * 4 + q % 4 of the 32, so that a lane ends with 8 neighbours
    const int q = r % 16, f = GATED ? r / 64 * 32 + q / 4 * 8 + r / 16 % 2 * 4 + q % 4 : r;
    src.w_off[j] = (uint32_t)min(n_base + f, N - 1) * (uint32_t)(K * 2) + wide_gemm::piece_of(lane, r);
  }
  f32x4 acc[MoeTile::MT][MoeTile::X];
#pragma unroll
  for (int mt = 0; mt < MoeTile::MT; ++mt)
#pragma unroll
    for (int x = 0; x < MoeTile::X; ++x) acc[mt][x] = f32x4{0.f, 0.f, 0.f, 0.f};
  MoeTile::run(acc, big_lds, src, K / MOE_BIG_K);
  // a lane holds rows 16 x + 4 kg .. + 3 (of its wavefront's of W in LDS) of the row wm * 64 + 16 mt + col
#pragma unroll
  for (int mt = 0; mt < MoeTile::MT; ++mt) {
    const int r = wm * MoeTile::PM + 16 * mt + col;
    if (r >= tile.z) continue;
    if (GATED) {
      const int f = n_base + wn * 32 + 8 * kg;  // N is a multiple of 64: all eight or none
      if (f < N) {
        bf16_t eight[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) eight[i] = __float2bfloat16(act_to<bf16_t>(acc[mt][i / 4][i % 4], ACT < 0 ? act_kind : ACT) * acc[mt][2 + i / 4][i % 4]);
        *reinterpret_cast<uint4*>(act_out + (int64_t)(tile.y + r) * N + f) = *reinterpret_cast<const uint4*>(eight);
      }
    } else {
      const int pair = order[tile.y + r];
      const float weight = weights[pair];
      float* o = y + ((int64_t)(pair % top) * num_tokens + pair / top) * N;
#pragma unroll
      for (int x = 0; x < MoeTile::X; ++x) {
        const int n = n_base + wn * MoeTile::PN + 16 * x + 4 * kg;
        if (n < N) *reinterpret_cast<f32x4*>(o + n) = weight * acc[mt][x];
      }
    }
  }
}

// rows a tile holds for a step of that many pairs: 16 while an expert sees a few tokens, 64 in portions, 128 in prompts
// (whose kernel reckons with 32-bit byte offsets within the rows and within an expert's weights)
// (and counts an expert's tiles in 15 bits)
extern "C" int pae_moe_tile_rows(int pairs, int hidden, int inter, int64_t row_bytes) {
  if (pairs <= 512) return 16;
  const int64_t widest = row_bytes > (int64_t)inter * 2 ? row_bytes : (int64_t)inter * 2;
  return (pairs > 4096 && pairs <= 0x7fff * MOE_BIG_ROWS && hidden % MOE_BIG_K == 0 && inter % MOE_BIG_K == 0 && pairs * widest < (1ll << 32) &&
          (int64_t)hidden * inter * 2 < (1ll << 32)) ? MOE_BIG_ROWS : 64;
}
extern "C" int pae_moe_max_tiles(int pairs, int experts) {
  const int rows = pairs <= 512 ? 16 : 64;  // the smallest tiles such a step may get: the most tiles there can be
  return (pairs + rows - 1) / rows + experts;
}
extern "C" int pae_moe_tiles_supported(int hidden, int inter) { return hidden % 32 == 0 && inter % 32 == 0; }

// `order` int32 [pairs], `tiles` int32 [pae_moe_max_tiles + 1][4], `act` bfloat16 [pairs][inter] are work space;
// y float32 [top][num_tokens][hidden] receives every pair's weighted output.
extern "C" int pae_moe_experts_tiles(float* y, const void* x, int64_t ldx, const void* gate_w, const void* up_w,
                                     const void* down_w, const int* chosen, const float* weights, int num_tokens, int top,
                                     int experts, int hidden, int inter, int act_kind, int* order, int* tiles, void* act,
                                     hipStream_t stream) {
  PAE_REQUIRE(top > 0 && experts > 0 && experts <= 4096, "experts: bad sizes top=%d experts=%d", top, experts);
  PAE_REQUIRE(pae_moe_tiles_supported(hidden, inter), "experts: widths %d and %d are no multiples of 32", hidden, inter);
  PAE_REQUIRE(ldx >= hidden && ldx % 8 == 0, "experts: row stride %lld", (long long)ldx);
  if (num_tokens <= 0) return 0;
  const int pairs = num_tokens * top;
  if (num_tokens <= 32 && pairs <= 256) {
    const bool by_pair = pairs <= experts;
    // (an odd number of columns, so that a column's workgroups go round the eight dies and not all to one)
    const dim3 up_grid((by_pair ? pairs : experts) | 1, (inter + 15) / 16, by_pair ? 1 : (num_tokens + 15) / 16);
    const dim3 down_grid(up_grid.x, (hidden + 15) / 16, up_grid.z);
    PAE_REQUIRE(up_grid.y <= 65535 && down_grid.y <= 65535, "experts: widths %d, %d exceed the grid", hidden, inter);
#define MOE_LISTED(LIST)                                                                                                         \
  moe_few_tiles_kernel<true, LIST><<<up_grid, 256, 0, stream>>>((bf16_t*)act, nullptr, (const bf16_t*)x, ldx,                    \
                                                                (const bf16_t*)gate_w, (const bf16_t*)up_w, chosen, weights,     \
                                                                nullptr, experts, top, num_tokens, hidden, inter, act_kind);     \
  moe_few_tiles_kernel<false, LIST><<<down_grid, 256, 0, stream>>>(nullptr, y, (const bf16_t*)act, inter, (const bf16_t*)down_w, \
                                                                   nullptr, chosen, weights, nullptr, experts, top, num_tokens,  \
                                                                   inter, hidden, act_kind)
    if (by_pair) {
      MOE_LISTED(BY_PAIR);
    } else {
      MOE_LISTED(BY_EXPERT);
    }
#undef MOE_LISTED
    return pae_check_launch("moe_experts_few");
  }
  const int tile_rows = pae_moe_tile_rows(pairs, hidden, inter, ldx * 2), max_tiles = pae_moe_max_tiles(pairs, experts);
  moe_sort_kernel<<<1, 1024, (size_t)(4 * experts + 1) * sizeof(int), stream>>>(chosen, pairs, experts, tile_rows, order,
                                                                               (int4*)tiles, max_tiles);
#define MOE_TILES(MT, UP_NT, DOWN_NT)                                                                                      \
  do {                                                                                                                     \
    dim3 up_grid(max_tiles, (inter + 64 * UP_NT - 1) / (64 * UP_NT)), down_grid(max_tiles, (hidden + 64 * DOWN_NT - 1) / (64 * DOWN_NT)); \
    PAE_REQUIRE(up_grid.y <= 65535 && down_grid.y <= 65535, "experts: widths %d, %d exceed the grid", hidden, inter);      \
    moe_tiles_gate_up_kernel<MT, UP_NT><<<up_grid, 256, 0, stream>>>((bf16_t*)act, (const bf16_t*)x, ldx,                   \
                                                                      (const bf16_t*)gate_w, (const bf16_t*)up_w, order,    \
                                                                      (const int4*)tiles, top, hidden, inter, act_kind);    \
    moe_tiles_down_kernel<MT, DOWN_NT><<<down_grid, 256, 0, stream>>>(y, (const bf16_t*)act, (const bf16_t*)down_w, order,  \
                                                                       weights, (const int4*)tiles, top, num_tokens, hidden, \
                                                                       inter);                                              \
  } while (0)
  if (tile_rows == 16) {
    dim3 up_grid(max_tiles, (inter + 15) / 16), down_grid(max_tiles, (hidden + 15) / 16);
    PAE_REQUIRE(up_grid.y <= 65535 && down_grid.y <= 65535, "experts: widths %d, %d exceed the grid", hidden, inter);
    moe_few_tiles_kernel<true, SORTED><<<up_grid, 256, 0, stream>>>((bf16_t*)act, nullptr, (const bf16_t*)x, ldx, (const bf16_t*)gate_w,
                                                                    (const bf16_t*)up_w, order, weights, (const int4*)tiles, experts,
                                                                    top, num_tokens, hidden, inter, act_kind);
    moe_few_tiles_kernel<false, SORTED><<<down_grid, 256, 0, stream>>>(nullptr, y, (const bf16_t*)act, inter, (const bf16_t*)down_w,
                                                                       nullptr, order, weights, (const int4*)tiles, experts, top,
                                                                       num_tokens, inter, hidden, act_kind);
  } else if (tile_rows == 64) MOE_TILES(4, 2, 4);
  else {
    const int64_t up_grid = (int64_t)max_tiles * ((inter + 127) / 128) + 7, down_grid = (int64_t)max_tiles * ((hidden + 255) / 256) + 7;
    PAE_REQUIRE(up_grid < (1ll << 31) && down_grid < (1ll << 31), "experts: widths %d, %d exceed the grid", hidden, inter);
    auto up = act_kind == 2 ? moe_big_tiles_kernel<true, 2> : act_kind == 1 ? moe_big_tiles_kernel<true, 1> : moe_big_tiles_kernel<true, -1>;
    auto down = moe_big_tiles_kernel<false, -1>;
    for (const void* kernel : {(const void*)up, (const void*)down}) {
      const hipError_t err = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MoeTile::LDS_BYTES);
      PAE_REQUIRE(err == hipSuccess, "experts: %d bytes of LDS refused: %s", MoeTile::LDS_BYTES, hipGetErrorString(err));
    }
    up<<<up_grid, 512, MoeTile::LDS_BYTES, stream>>>((bf16_t*)act, nullptr, (const bf16_t*)x, ldx, (const bf16_t*)gate_w, (const bf16_t*)up_w,
                                                     order, weights, (const int4*)tiles, max_tiles, top, num_tokens, hidden, inter, act_kind);
    down<<<down_grid, 512, MoeTile::LDS_BYTES, stream>>>(nullptr, y, (const bf16_t*)act, inter, (const bf16_t*)down_w, nullptr, order, weights,
                                                         (const int4*)tiles, max_tiles, top, num_tokens, inter, hidden, act_kind);
  }
#undef MOE_TILES
  return pae_check_launch("moe_experts_tiles");
}
