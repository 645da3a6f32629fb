// Gated linear attention: a recurrent mixer whose per-request state is one matrix S [D, V] per head, which
// decays per token by a factor of its own for every key channel (every row of S):
//
//   a_t = sigmoid(z_t + bias)^(1 / tau)          (one number per head and key channel)
//   S  <- diag(a_t) S + k_t v_t^T;   o_t = S^T q_t,   q times D^-1/2
//
// then o is divided by its root mean square over V, multiplied by a weight of V numbers that the heads share
// and by act(gate) (SiLU or sigmoid), and rounded to the activation type.  S starts at zero (a slot is zeroed
// when a request takes it).  A step's projected rows hold, per token, [q: H heads of D | k: H heads of D |
// v: H heads of V]; the decay's input z [T][H D] and the gate's rows [T][H V] come as rows of their own.  Three
// kernels:
//
//   gla_prepare      q, k, v to float32 rows (q scaled); the decays as exp(logsigmoid(z + bias) / tau)
//   the delta rule's recurrence kernel (delta_rule.hip) with a decay per key channel and without its
//   read-before-write: a column of S stays in the registers of a group of lanes over the whole step
//   the delta rule's gated norm
//
// Steps whose runs are long on average go by chunks of 16 tokens instead of the first two (see below); a step of single tokens does
// all three in one launch, with the same bits (recurrent_tokens.hip).
//
// Everything but the projected rows, z and the gate's rows is float32: the decay and its logarithm, the state,
// the read-out and the norm.  Token by token the order in which a column's sums are formed depends on D alone; by chunks it
// depends on where in its run a token stands, and which of the two is taken on the step.
#include "common.h"
#include "api.h"
#include "recurrent_tokens.h"

void pae_launch_recurrence(const float* q, const float* k, const float* v, const float* beta, const float* decay,
                           const int4* runs, const int* slots, float* state, int64_t state_slot_stride, int G, int H,
                           int D, int V, int num_tokens, int num_seqs, int channel_decay, int delta, float* o, hipStream_t stream);
int pae_launch_gated_norm(int dtype, const float* o, const void* gates, int64_t gate_stride, int gate_sigmoid,
                          const void* weight, int w_is_f32, float eps, int num_tokens, int H, int V, void* out,
                          hipStream_t stream);

// One workgroup of 128 threads per (token, head).
template <typename T>
__global__ __launch_bounds__(128) void gla_prepare_kernel(const T* __restrict__ proj, int64_t row_stride,
                                                          const T* __restrict__ z_in, int64_t z_stride,
                                                          const void* __restrict__ z_bias, int bias_is_f32, float inv_tau,
                                                          int H, int D, int V, float* __restrict__ q_out,
                                                          float* __restrict__ k_out, float* __restrict__ v_out,
                                                          float* __restrict__ decay_out, float* __restrict__ ones_out) {
  const int64_t t = blockIdx.x;
  const int h = blockIdx.y;
  const T* row = proj + t * row_stride;
  const T* z = z_in + t * z_stride + h * D;
  const float q_scale = 1.0f / sqrtf((float)D);
  const int64_t at = (t * H + h) * D;
  for (int d = threadIdx.x; d < D; d += 128) {
    q_out[at + d] = to_f32(row[h * D + d]) * q_scale;
    k_out[at + d] = to_f32(row[(H + h) * D + d]);
    const float bias = z_bias ? load_param(z_bias, bias_is_f32, h * D + d) : 0.f;
    decay_out[at + d] = expf(gla_log_sigmoid(to_f32(z[d]) + bias) * inv_tau);
  }
  float* v = v_out + (t * H + h) * V;
  for (int i = threadIdx.x; i < V; i += 128) v[i] = to_f32(row[2 * H * D + h * V + i]);
  if (threadIdx.x == 0) ones_out[t * H + h] = 1.0f;  // the recurrence's write strength: every token writes k v^T whole
}

// ------------------------------------------------------------------ runs of many tokens
// Cut into chunks of 16 tokens from the run's first, with L_t the product of the chunk's decays up to and with token t:
//
//   o_t = (q_t L_t)^T S + sum_{j <= t} (sum_d q_td k_jd a_{j+1,d} .. a_td) v_j;    S <- L_16 S + sum_j (k_j a_{j+1} .. a_16) v_j^T
//
// Every product of decays is formed as it stands, by running products: nothing is divided by a decay, however small.
// gla_chunk_prepare forms the factors of v and S chunk by chunk side by side; what remains for gla_chunks, which walks a
// run's chunks one after the other, are two products of float32 matrix instructions a chunk, in whose registers S stays.
//
// Walking a run token by token takes some 40 vector instructions a token, which the one wavefront that a SIMD then has issues in
// 130 ns, and the longest run sets the time; 16 tokens here take 0.85 us, the chain of a chunk's instructions and of its barrier.
// (The places of a chunk's numbers are lane offsets behind a scalar base: reckoned in 64 bits by every lane a chunk took 1.4 us;
// with what lies behind a run's end taken out where it is loaded, which waits for it there, 3.2.)  gla_chunk_prepare is bound by
// its instructions, half of them the decays' logarithms and powers: 36 us for 2,047 tokens of 12 heads, `gla_prepare`'s 25 without the factors.
// Measured, the whole mixer with 12 heads of 128 x 128: a run of 2,047 tokens 308 -> 152 us, four of 2,047 in all 138 -> 96,
// 16 of 4,000 220 -> 152.  Against 64 bits, 12 heads, float32 rows, runs of 300 and of 1,500 tokens: read-outs 2.38e-7 -> 2.24e-7
// and 2.67e-7 -> 2.52e-7, states 2.10e-7 -> 2.00e-7 and 2.62e-7 -> 2.50e-7.
//
// What is infinite or NaN in a token's row reaches its own read-out and those behind it, as token by token.
constexpr int GLA_CHUNK = 16;
// Steps whose runs have that many tokens on average go by chunks: the launch is given counts of tokens and runs, their lengths lie on the
// device (a long run beside many single tokens stays token by token).  Both ways in us, 12 heads of 128:
// one run of 96 24.7 and 26.6, 128 30.6 and 29.1, 160 36.5 and 31.7; 8 runs of 100 57.3 and 60.3, of 138 71.0 and 68.3; 28 heads, two
// runs of 128 45.3 and 47.8; 300 tokens beside 63 single ones 63 and 94.  Heads of up to 32 features have less to share out: 16
// features, one run of 160 21.0 and 24.0, of 200 25.2 and 26.1, 16 runs of 250 55 and 43.
static int gla_chunked_from(int D) { return D <= 32 ? 320 : 160; }

template <int BIT>
__device__ __forceinline__ float gla_across(float v) {  // the number of a lane that differs in bit BIT and agrees in the higher ones
  constexpr int CTRL = BIT == 8 ? 0x140 : BIT == 4 ? 0x141 : BIT == 2 ? 0x4E : 0xB1;  // 16 or 8 lanes mirrored, a quad's exchanged
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), CTRL, 0xF, 0xF, true));
}
// Sums over 16 lanes of 2 BIT numbers a lane: lane i of the 16 is left with that of number i.
template <int BIT>
__device__ __forceinline__ void gla_sums(float* a, int lane) {
  if constexpr (BIT > 0) {
    const bool up = lane & BIT;
#pragma unroll
    for (int j = 0; j < BIT; ++j) a[j] = (up ? a[j + BIT] : a[j]) + gla_across<BIT>(up ? a[j] : a[j + BIT]);
    gla_sums<BIT / 2>(a, lane);
  }
}

// One workgroup per (chunk of the step, head), a thread per key channel (blockDim is D up to whole wavefronts).  Chunks are
// numbered sequence by sequence; workgroups beyond the last do nothing.  Leaves, at the rows of the chunk's tokens, q_t L_t,
// k_j a_{j+1} .. a_16, v and `near` [T][H][16], the factors of v_j in o_t, and L_16 at the first token's row of `decay`.
template <typename T>
__global__ __launch_bounds__(256) void gla_chunk_prepare_kernel(
    const T* __restrict__ proj, int64_t row_stride, const T* __restrict__ z_in, int64_t z_stride, const void* __restrict__ z_bias,
    int bias_is_f32, float inv_tau, const int4* __restrict__ seq_runs, int num_seqs, int H, int D, int V, float* __restrict__ q_out,
    float* __restrict__ k_out, float* __restrict__ v_out, float* __restrict__ decay_out, float* __restrict__ near_out) {
  __shared__ float s_near[16][GLA_CHUNK][GLA_CHUNK + 1];  // by row of 16 lanes: [j][t]
  const int h = blockIdx.y, lane = threadIdx.x % PAE_WAVE;
  // which sequence's chunk this is: 64 sequences at a time, their chunks counted
  int row0 = -1, n = 0, before = 0;
  for (int s0 = 0; s0 < num_seqs && row0 < 0; s0 += PAE_WAVE) {
    const int4 run = s0 + lane < num_seqs ? seq_runs[s0 + lane] : make_int4(0, 0, 0, 0);
    const int mine = (run.y + GLA_CHUNK - 1) / GLA_CHUNK;
    int upto = mine;
    for (int off = 1; off < PAE_WAVE; off <<= 1) {
      const int other = __shfl_up(upto, off, PAE_WAVE);
      if (lane >= off) upto += other;
    }
    const int chunk = blockIdx.x - before - (upto - mine);
    const uint64_t here = __ballot(chunk >= 0 && chunk < mine);
    if (here) {
      const int who = __ffsll((unsigned long long)here) - 1;
      const int first = __shfl(chunk, who, PAE_WAVE) * GLA_CHUNK;
      row0 = __shfl(run.x, who, PAE_WAVE) + first;
      n = min(GLA_CHUNK, __shfl(run.y, who, PAE_WAVE) - first);
    }
    before += __shfl(upto, PAE_WAVE - 1, PAE_WAVE);
  }
  if (row0 < 0) return;
  const int d = threadIdx.x < D ? threadIdx.x : 0;
  const bool live = threadIdx.x < D;
  const float q_scale = 1.0f / sqrtf((float)D), bias = z_bias ? load_param(z_bias, bias_is_f32, h * D + d) : 0.f;
  float q[GLA_CHUNK], k[GLA_CHUNK], a[GLA_CHUNK];
#pragma unroll
  for (int t = 0; t < GLA_CHUNK; ++t) {  // tokens behind the run's last: neither read nor write anything, no decay
    const int64_t row = row0 + min(t, n - 1);
    const bool there = live && t < n;
    const float qt = to_f32(proj[row * row_stride + h * D + d]) * q_scale;
    const float kt = to_f32(proj[row * row_stride + (H + h) * D + d]);
    const float at = expf(gla_log_sigmoid(to_f32(z_in[row * z_stride + h * D + d]) + bias) * inv_tau);
    q[t] = there ? qt : 0.f;
    k[t] = there ? kt : 0.f;
    a[t] = there ? at : 1.f;
  }
  // the factors of v_j and v_{16 - j} are 16 numbers together: for tokens j .. 15 and 16 - j .. 15
#pragma unroll
  for (int j = 0; j <= GLA_CHUNK / 2; ++j) {
    float parts[GLA_CHUNK], p = k[j];
#pragma unroll
    for (int i = 0; i < GLA_CHUNK; ++i) {
      if (j + i < GLA_CHUNK) {
        if (i > 0) p *= a[j + i];
        parts[i] = q[j + i] * p;
      } else {
        parts[i] = 0.f;
      }
    }
    if (live && j < n) k_out[((int64_t)(row0 + j) * H + h) * D + d] = p;
    if (j > 0 && j < GLA_CHUNK / 2) {
      p = k[GLA_CHUNK - j];
#pragma unroll
      for (int t = GLA_CHUNK - j; t < GLA_CHUNK; ++t) {
        if (t > GLA_CHUNK - j) p *= a[t];
        parts[t] = q[t] * p;
      }
      if (live && GLA_CHUNK - j < n) k_out[((int64_t)(row0 + GLA_CHUNK - j) * H + h) * D + d] = p;
    }
    gla_sums<GLA_CHUNK / 2>(parts, lane);
    const int i = lane % 16;
    const bool own = j + i < GLA_CHUNK;
    if (own || j < GLA_CHUNK / 2) s_near[threadIdx.x / 16][own ? j : GLA_CHUNK - j][own ? j + i : i] = parts[0];
  }
  float upto = 1.f;
#pragma unroll
  for (int t = 0; t < GLA_CHUNK; ++t) {
    upto *= a[t];
    if (live && t < n) q_out[((int64_t)(row0 + t) * H + h) * D + d] = q[t] * upto;
  }
  if (live) decay_out[((int64_t)row0 * H + h) * D + d] = upto;
  for (int c = threadIdx.x; c < V; c += blockDim.x) {
#pragma unroll
    for (int t = 0; t < GLA_CHUNK; ++t)
      if (t < n) v_out[((int64_t)(row0 + t) * H + h) * V + c] = to_f32(proj[(int64_t)(row0 + t) * row_stride + 2 * H * D + h * V + c]);
  }
  __syncthreads();
  const int rows = blockDim.x / 16;
  for (int e = threadIdx.x; e < n * GLA_CHUNK; e += blockDim.x) {
    const int t = e / GLA_CHUNK, j = e % GLA_CHUNK;
    float sum = 0.f;
    if (j <= t)
      for (int r = 0; r < rows; ++r) sum += s_near[r][j][t];
    near_out[((int64_t)(row0 + t) * H + h) * GLA_CHUNK + j] = sum;
  }
}

typedef float gla_x4 __attribute__((ext_vector_type(4)));

// One workgroup per (head, 16 columns of S, sequence); wavefront w holds the 16 TW rows of S from 16 TW w on, as tiles of the
// matrix instructions' accumulators: lane (column lane % 16, g = lane / 16), register i: row 4 g + i of the tile.  As the
// instruction's sum over its four lanes' groups may run in any order, the same registers are the right operand of q L S, group g
// bringing row 4 g + i to instruction i, and the left one then is one load of four of q's features.  The wavefronts' parts of the
// read-outs meet in LDS once a chunk, in places that take turns (a barrier that waits for LDS alone: stores stay on their way).
template <int TW>
__global__ __launch_bounds__(256) void gla_chunks_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                         const float* __restrict__ v, const float* __restrict__ decay,
                                                         const float* __restrict__ near, const int4* __restrict__ seq_runs,
                                                         const int* __restrict__ slots, float* __restrict__ state,
                                                         int64_t state_slot_stride, int H, int D, int V, float* __restrict__ out) {
  __shared__ float s_part[2][4][4][PAE_WAVE];
  const int h = blockIdx.x, s = blockIdx.z;
  const int lane = threadIdx.x % PAE_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / PAE_WAVE);
  const int m = lane % 16, g = lane / 16;
  const int4 run = seq_runs[s];
  if (run.y <= 0) return;
  const int col = blockIdx.y * 16 + m, c = col < V ? col : 0;
  float* column = state + (int64_t)slots[s] * state_slot_stride + ((int64_t)h * V + c) * D;
  const int d0 = wave * 16 * TW;
  gla_x4 S[TW];
#pragma unroll
  for (int j = 0; j < TW; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = d0 + 16 * j + 4 * g + i;
      S[j][i] = d < D ? column[d] : 0.f;
    }
  struct Chunk {
    gla_x4 q[TW], through[TW], k[TW], v;
    float near;
  };
  // (places behind D are read at feature 0: there S is zero and stays zero)
  auto load = [&](int first, int n) {
    Chunk x;
    const int64_t at = ((int64_t)run.x + first) * H + h;  // the same in every lane: a scalar base, and offsets of the lanes' own
    const float *qc = q + at * D, *kc = k + at * D, *lc = decay + at * D, *vc = v + at * V, *nc = near + at * GLA_CHUNK;
    const int mine = min(m, n - 1) * H;  // (lanes behind the last token: its numbers, not used)
#pragma unroll
    for (int j = 0; j < TW; ++j) {
      const int d = d0 + 16 * j + 4 * g, dm = d0 + 16 * j + m;  // (D is a multiple of four)
      x.q[j] = *reinterpret_cast<const gla_x4*>(qc + (unsigned)(mine * D + (d < D ? d : 0)));
      x.through[j] = *reinterpret_cast<const gla_x4*>(lc + (unsigned)(d < D ? d : 0));
#pragma unroll
      for (int i = 0; i < 4; ++i) x.k[j][i] = kc[(unsigned)(min(4 * g + i, n - 1) * H * D + (dm < D ? dm : 0))];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) x.v[i] = vc[(unsigned)(min(4 * g + i, n - 1) * H * V + c)];
    x.near = nc[(unsigned)(mine * GLA_CHUNK + 4 * g + wave)];
    return x;
  };
  // Values that are infinite or NaN, among the tokens 4 g + wave, onto the read-outs of their own token and of those behind it (rare).
  auto add_no_numbers = [&](float near, float vw, gla_x4& o) {
    for (int from = 0; from < 4; ++from) {
      const float value = __shfl(vw, 16 * from + m, PAE_WAVE);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float factor = __shfl(near, 16 * from + 4 * g + i, PAE_WAVE);
        if (!__builtin_isfinite(value) && 4 * from + wave <= 4 * g + i) o[i] += factor * value;
      }
    }
  };
  auto advance = [&](const Chunk& x, int first, int n, int turn) {
    // the chunk's own tokens: wavefront w takes those 4 g + w
    const float vw = wave == 0 ? x.v[0] : wave == 1 ? x.v[1] : wave == 2 ? x.v[2] : x.v[3];
    gla_x4 o[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j) o[j % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.q[j][i], S[j][i], o[j % 2], 0, 0, 0);
    // (the instruction multiplies the tokens behind a read-out's own by a factor of zero: what is no number among them goes apart)
    const bool number = __builtin_isfinite(vw);
    o[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(x.near, number ? vw : 0.f, o[1], 0, 0, 0);
    if (__builtin_amdgcn_ballot_w64(!number) != 0) add_no_numbers(x.near, vw, o[1]);
#pragma unroll
    for (int j = 0; j < TW; ++j) S[j] *= x.through[j];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < TW; ++j)
        S[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(d0 + 16 * j + m < D ? x.k[j][i] : 0.f, x.v[i], S[j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) s_part[turn][wave][i][lane] = o[0][i] + o[1][i];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const float sum = (s_part[turn][0][wave][lane] + s_part[turn][1][wave][lane]) +
                      (s_part[turn][2][wave][lane] + s_part[turn][3][wave][lane]);
    const int t = 4 * g + wave;
    if (t < n && col < V) out[(((int64_t)run.x + first) * H + h) * V + (unsigned)(t * H * V + col)] = sum;
  };
  // Whole chunks, AHEAD on their way (behind the last one that one again, not used): a chunk takes less time than a trip to memory.
  constexpr int AHEAD = 2;
  const int whole = run.y / GLA_CHUNK;
  if (whole > 0) {
    Chunk x[AHEAD];
#pragma unroll
    for (int a = 0; a < AHEAD; ++a) x[a] = load(min(a, whole - 1) * GLA_CHUNK, GLA_CHUNK);
    int at = 0;
    for (; at + AHEAD <= whole; at += AHEAD) {
#pragma unroll
      for (int a = 0; a < AHEAD; ++a) {
        advance(x[a], (at + a) * GLA_CHUNK, GLA_CHUNK, a % 2);
        x[a] = load(min(at + a + AHEAD, whole - 1) * GLA_CHUNK, GLA_CHUNK);
      }
    }
#pragma unroll
    for (int a = 0; a < AHEAD - 1; ++a)
      if (at + a < whole) advance(x[a], (at + a) * GLA_CHUNK, GLA_CHUNK, a % 2);
  }
  const int rest = run.y % GLA_CHUNK;
  if (rest > 0) {  // tokens behind the last: no factor, nothing to add
    Chunk x = load(whole * GLA_CHUNK, rest);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      x.v[i] = 4 * g + i < rest ? x.v[i] : 0.f;
#pragma unroll
      for (int j = 0; j < TW; ++j) x.k[j][i] = 4 * g + i < rest ? x.k[j][i] : 0.f;
    }
    x.near = 4 * g + wave < rest ? x.near : 0.f;
    advance(x, whole * GLA_CHUNK, rest, whole % 2);
  }
  if (col < V)
#pragma unroll
    for (int j = 0; j < TW; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = d0 + 16 * j + 4 * g + i;
        if (d < D) column[d] = S[j][i];
      }
}

static int64_t gla_part(int64_t floats) { return (floats + 3) / 4 * 4; }

// Whether a step goes by chunks (four features are read at a time, and a workgroup holds up to 256).
extern "C" int pae_linear_attention_by_chunks(int num_tokens, int num_seqs, int D) {
  return D <= 256 && D % 4 == 0 && num_tokens >= (int64_t)gla_chunked_from(D) * num_seqs;
}

extern "C" int pae_linear_attention_step(int dtype, const void* proj, int64_t row_stride, const void* z_in, int64_t z_stride,
                                         const void* z_bias, int bias_is_f32, float tau, const void* gate_in,
                                         int64_t gate_stride, int gate_sigmoid, int num_tokens, int num_seqs,
                                         const int* seq_runs, const int* slots, int H, int D, int V, float* state,
                                         int64_t state_slot_stride, const void* norm_w, int w_is_f32, float norm_eps,
                                         float* work, void* out, hipStream_t stream) {
  PAE_REQUIRE(H > 0 && D > 0 && V > 0, "linear attention: bad head sizes H=%d D=%d V=%d", H, D, V);
  PAE_REQUIRE(D <= 1024 && V <= 1024, "linear attention: key width %d or value width %d exceeds 1024", D, V);
  PAE_REQUIRE(H <= 65535 && num_seqs <= 65535, "linear attention: %d heads, %d sequences exceed the grid", H, num_seqs);
  PAE_REQUIRE(row_stride >= 2 * (int64_t)H * D + (int64_t)H * V, "linear attention: row stride %lld too small", (long long)row_stride);
  PAE_REQUIRE(z_stride >= (int64_t)H * D && gate_stride >= (int64_t)H * V, "linear attention: the decay's or the gate's rows are too narrow");
  PAE_REQUIRE(tau > 0.f, "linear attention: the decay's temperature must be positive, got %g", (double)tau);
  PAE_REQUIRE(z_in && gate_in, "linear attention: the decay's and the gate's rows are needed");
  PAE_REQUIRE(dtype == PAE_F32 || dtype == PAE_BF16, "linear attention: unknown dtype code %d", dtype);
  if (num_tokens <= 0 || num_seqs <= 0) return 0;
  if (takes_tokens_step(num_tokens, num_seqs, H, H, D, V, state, state_slot_stride)) {
    const TokensStep p = {proj, row_stride, (const int4*)seq_runs, slots, state, state_slot_stride, H, H, D, V, z_in, z_stride,
                          gate_in, gate_stride, gate_sigmoid, norm_w, w_is_f32, norm_eps, out, nullptr, nullptr, 0, 0,
                          nullptr, nullptr, 0.f, nullptr, 0, z_bias, bias_is_f32, 1.0f / tau};
    launch_tokens_step(TOKENS_LINEAR, dtype, p, num_seqs, stream);
    return pae_check_launch("linear_attention_step (single tokens)");
  }
  // work: q [T][H][D], k [T][H][D], decay [T][H][D], v [T][H][V], ones [T][H] (by chunks: near [T][H][16]), o [T][H][V], each on a
  // 16-byte boundary
  const int64_t T = num_tokens;
  float* q = work;
  float* k = q + gla_part(T * H * D);
  float* decay = k + gla_part(T * H * D);
  float* v = decay + gla_part(T * H * D);
  float* ones = v + gla_part(T * H * V);
  const bool chunks = pae_linear_attention_by_chunks(num_tokens, num_seqs, D);
  float* o = ones + gla_part(T * H * (chunks ? GLA_CHUNK : 1));
  const int4* runs = (const int4*)seq_runs;
  if (chunks) {
    // (a run of n tokens has at most (n + 15) / 16 chunks)
    const dim3 chunk_heads((unsigned)((T + (GLA_CHUNK - 1) * (int64_t)num_seqs) / GLA_CHUNK), H);
    const int threads = (D + PAE_WAVE - 1) / PAE_WAVE * PAE_WAVE;
#define GLA_PREPARE(T)                                                                                                            \
  gla_chunk_prepare_kernel<T><<<chunk_heads, threads, 0, stream>>>((const T*)proj, row_stride, (const T*)z_in, z_stride, z_bias, \
                                                                   bias_is_f32, 1.0f / tau, runs, num_seqs, H, D, V, q, k, v, decay, ones)
    if (dtype == PAE_F32) {
      GLA_PREPARE(float);
    } else {
      GLA_PREPARE(bf16_t);
    }
#undef GLA_PREPARE
    const dim3 grid(H, (V + 15) / 16, num_seqs);
#define GLA_CHUNKS(TW) \
  gla_chunks_kernel<TW><<<grid, 256, 0, stream>>>(q, k, v, decay, ones, runs, slots, state, state_slot_stride, H, D, V, o)
    if (D <= 64) GLA_CHUNKS(1);
    else if (D <= 128) GLA_CHUNKS(2);
    else if (D <= 192) GLA_CHUNKS(3);
    else GLA_CHUNKS(4);
#undef GLA_CHUNKS
  } else {
    const dim3 token_heads(num_tokens, H);
    if (dtype == PAE_F32)
      gla_prepare_kernel<float><<<token_heads, 128, 0, stream>>>((const float*)proj, row_stride, (const float*)z_in, z_stride,
                                                                 z_bias, bias_is_f32, 1.0f / tau, H, D, V, q, k, v, decay, ones);
    else
      gla_prepare_kernel<bf16_t><<<token_heads, 128, 0, stream>>>((const bf16_t*)proj, row_stride, (const bf16_t*)z_in, z_stride,
                                                                  z_bias, bias_is_f32, 1.0f / tau, H, D, V, q, k, v, decay, ones);
    pae_launch_recurrence(q, k, v, ones, decay, runs, slots, state, state_slot_stride, H, H, D, V, num_tokens, num_seqs, 1, 0, o, stream);
  }
  const int code = pae_launch_gated_norm(dtype, o, gate_in, gate_stride, gate_sigmoid, norm_w, w_is_f32, norm_eps,
                                         num_tokens, H, V, out, stream);
  if (code) return code;
  return pae_check_launch("linear_attention_step");
}

// floats of `work` that pae_linear_attention_step needs for a step of `num_tokens` rows
extern "C" int64_t pae_linear_attention_work_floats(int num_tokens, int H, int D, int V) {
  const int64_t T = num_tokens;
  return 3 * gla_part(T * H * D) + 2 * gla_part(T * H * V) + gla_part(T * H * (pae_linear_attention_by_chunks(num_tokens, 1, D) ? GLA_CHUNK : 1));
}
