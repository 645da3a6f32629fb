// The gated delta rule and gated linear attention where every sequence of a step brings one token (decoding): what
// delta_rule.hip and linear_attention.hip do in three or four launches (convolution, unit vectors and decays; the convolution's
// inputs moved on; the recurrence; the gated norm) in one.
//
// What bounds such a step is launches: each of those kernels takes 3 to 6 us beside the state's way from memory and back, 64 KB a head
// each way.  Here a workgroup of 16 wavefronts takes a (sequence, key head) with the value heads that read it, so that it alone reads
// and moves on its channels of the convolution, and has the whole head, over which the norm goes, in one place.  A column of S belongs to L
// lanes of 8 rows each, as in delta_recurrence_group_kernel, a lane holds them of up to two columns; the state is asked for first, before
// the token's numbers are made.  Every sum is formed in the order of the separate kernels: the same bits.
//
// Measured in a recorded graph, us for 1 / 8 / 64 sequences, separate kernels and this: delta rule with 12 heads of 128 by 128 12.2 / 14.9 / 42.1
// and 7.9 / 8.7 / 24.1, with channel decays 12.7 / 15.1 / 43.3 and 8.5 / 9.5 / 26.1; 28 heads 12.3 / 21.5 / 73.0 and 8.0 / 10.2 / 48.6; linear attention with 12
// heads 8.9 / 11.4 / 37.9 and 4.3 / 5.2 / 20.5, 14 heads of 64 8.4 / 8.8 / 17.8 and 3.9 / 4.4 / 13.9.  What is left of the delta rule's 8 us is
// a chain: the run and its slot, the convolution's inputs, the unit vectors' sums, the state's products, the norm's sum.
#include "api.h"
#include "recurrent_tokens.h"

namespace {

constexpr int THREADS = 1024, R = 8, COLUMNS = 2;  // rows and columns of S a lane holds
constexpr int MOST_VALUES = 4096;                  // of the value heads of a key head, in LDS

typedef float f32x4 __attribute__((ext_vector_type(4)));

template <typename T, int L, int KIND>
__global__ __launch_bounds__(THREADS) void recurrent_tokens_kernel(TokensStep p) {
  constexpr bool DELTA = KIND != TOKENS_LINEAR, CHANNEL = KIND != TOKENS_DELTA;
  constexpr int DP = L * R, EACH = THREADS / L;  // a key head's rows, padded; columns side by side
  extern __shared__ __attribute__((aligned(16))) float s_values[];  // v [heads][V], then decays [heads][DP] (CHANNEL)
  __shared__ __attribute__((aligned(16))) float s_q[DP], s_k[DP];
  __shared__ float s_out[2][EACH * COLUMNS], s_sums[4];
  const int s = blockIdx.y, g = blockIdx.x, tid = threadIdx.x, lane = tid % PAE_WAVE;
  const int G = p.G, H = p.H, D = p.D, V = p.V, heads = H / G, h0 = g * heads;
  const int4 run = p.runs[s];
  const int slot = p.slots[s];
  float* s_dec = s_values + (heads * V + 3) / 4 * 4;
  float* s_scalars = s_dec + (CHANNEL ? heads * DP : 0);  // beta, then decay (one a head)
  const int sub = tid % L, column = tid / L;
  float* state = p.state + (int64_t)slot * p.state_slot_stride;
  auto load_state = [&](float (&S)[COLUMNS][R], int h) {
#pragma unroll
    for (int c = 0; c < COLUMNS; ++c) {
      const int col = c * EACH + column;
      const float* from = state + (uint32_t)((h * V + min(col, V - 1)) * D);
#pragma unroll
      for (int r4 = 0; r4 < R / 4; ++r4) {
        const int d = r4 * (4 * L) + sub * 4;
        const f32x4 x = *reinterpret_cast<const f32x4*>(from + min(d, D - 4));
#pragma unroll
        for (int e = 0; e < 4; ++e) S[c][4 * r4 + e] = d < D ? x[e] : 0.f;
      }
    }
  };
  const int64_t C = 2 * (int64_t)G * D + (int64_t)H * V;
  float* tail = DELTA ? p.conv_tail + (int64_t)slot * p.tail_slot_stride : nullptr;
  const int keep = p.taps - 1;
  // channel c of the token `in_step` rows behind the run's first, convolved and activated
  auto convolved = [&](int in_step, int64_t c) {
    const T* row = (const T*)p.proj + (int64_t)(run.x + in_step) * p.row_stride + c;
    const float* before = keep > 0 ? tail + c : p.conv_w;  // (one tap: no tail, and nothing of it is used)
    float sum = 0.f;
    for (int j0 = 0; j0 < p.taps; j0 += 4) {  // four taps asked for together, of rows and tail, from places that there are
      float x[4], w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = min(j0 + u, keep), back = keep - j;
        const float here = to_f32(row[-(int64_t)min(back, in_step) * p.row_stride]), held = before[(int64_t)min(keep - back + in_step, max(keep - 1, 0)) * C];
        x[u] = back <= in_step ? here : held;
        w[u] = p.conv_w[c * p.taps + j];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j0 + u < p.taps) sum = fmaf(w[u], x[u], sum);
    }
    return silu_f(sum);
  };
  // the convolution's inputs of channel c moved on by the run's rows (entries read lie above those written before)
  auto move_on = [&](int64_t c) {
    for (int j0 = 0; j0 < keep; j0 += 4) {
      float x[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int j = min(j0 + u, keep - 1), r = run.y - keep + j;
        x[u] = r >= 0 ? to_f32(((const T*)p.proj)[(int64_t)(run.x + r) * p.row_stride + c]) : tail[(int64_t)(j + run.y) * C + c];
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (j0 + u < keep) tail[(int64_t)(j0 + u) * C + c] = x[u];
    }
  };

  int parity = 0;
  for (int i = 0; i < run.y; ++i) {
    const int64_t t = run.x + i;
    const T* row = (const T*)p.proj + t * p.row_stride;
    float S[COLUMNS][R];
    load_state(S, h0);
    // the token's numbers: threads 0 to 127 q, 128 to 255 k, the others values, decays and strengths
    const int wave = tid / PAE_WAVE;
    float unit = 0.f;
    if (wave < 4) {
      const int d = tid % 128, which = tid / 128;
      if (DELTA) {
        const int64_t c = ((int64_t)which * G + g) * D + d;
        if (d < D) {
          unit = convolved(i, c);
          if (i == run.y - 1) move_on(c);
        }
        const float sum = wave_sum(fmaf(unit, unit, 0.f));
        if (lane == 0) s_sums[wave] = sum;
      } else if (d < DP) {
        float x = 0.f;
        if (d < D) x = to_f32(row[((int64_t)which * H + g) * D + d]);
        if (which == 0) s_q[d] = x * (1.0f / sqrtf((float)D));
        else s_k[d] = x;
      }
    } else {
      for (int v = tid - 256; v < heads * V; v += THREADS - 256) {
        if (DELTA) {
          const int64_t c = 2 * (int64_t)G * D + (int64_t)h0 * V + v;
          s_values[v] = convolved(i, c);
          if (i == run.y - 1) move_on(c);
        } else {
          s_values[v] = to_f32(row[2 * (int64_t)H * D + (int64_t)h0 * V + v]);
        }
      }
      const T* decay_row = (const T*)p.decay_in + t * p.decay_stride;
      if (CHANNEL) {
        for (int e = tid - 256; e < heads * DP; e += THREADS - 256) {
          const int hh = e / DP, d = e % DP, c = (h0 + hh) * D + d;
          float dec = 0.f;
          if (d < D) {
            if (DELTA) dec = expf(-expf(p.a_log[h0 + hh]) * softplus_f(to_f32(decay_row[c]) + p.dt_bias[c]));
            else dec = expf(gla_log_sigmoid(to_f32(decay_row[c]) + (p.decay_bias ? load_param(p.decay_bias, p.bias_is_f32, c) : 0.f)) * p.inv_tau);
          }
          s_dec[e] = dec;
        }
      }
      if (DELTA) {
        for (int hh = THREADS - 1 - tid; hh < heads; hh += THREADS - 256) {
          const int h = h0 + hh;
          s_scalars[2 * hh] = 1.0f / (1.0f + expf(-to_f32(((const T*)p.beta_in)[t * p.beta_stride + h])));
          if (!CHANNEL) s_scalars[2 * hh + 1] = expf(-expf(p.a_log[h]) * softplus_f(to_f32(decay_row[h]) + p.dt_bias[h]));
        }
      }
    }
    __syncthreads();
    if (DELTA) {  // q and k become unit vectors, q also divided by sqrt(D)
      if (wave < 4 && tid % 128 < DP) {
        const int which = tid / 128;
        float total = 0.f;
        total += s_sums[2 * which];
        total += s_sums[2 * which + 1];
        const float inv = 1.0f / sqrtf(total + p.unit_eps);
        if (which == 0) s_q[tid % 128] = unit * inv * (1.0f / sqrtf((float)D));
        else s_k[tid % 128] = unit * inv;
      }
      __syncthreads();
    }

    for (int hh = 0; hh < heads; ++hh) {
      const int h = h0 + hh;
      // what the norm reads, and the next head's state, are on their way beside this head's sums
      const T* gate = (const T*)p.gate + t * p.gate_stride + (int64_t)h * V;
      const float z = to_f32(gate[min(tid, V - 1)]), w = load_param(p.norm_w, p.w_is_f32, min(tid, V - 1));
      float next[COLUMNS][R];
      if (hh + 1 < heads) load_state(next, h + 1);
      f32x4 k4[R / 4], q4[R / 4], d4[R / 4];
#pragma unroll
      for (int r4 = 0; r4 < R / 4; ++r4) {
        const int at = r4 * (4 * L) + sub * 4;
        k4[r4] = *reinterpret_cast<const f32x4*>(s_k + at);
        q4[r4] = *reinterpret_cast<const f32x4*>(s_q + at);
        if (CHANNEL) d4[r4] = *reinterpret_cast<const f32x4*>(s_dec + hh * DP + at);
        else d4[r4] = f32x4{s_scalars[2 * hh + 1], s_scalars[2 * hh + 1], s_scalars[2 * hh + 1], s_scalars[2 * hh + 1]};
      }
      const float beta = DELTA ? s_scalars[2 * hh] : 1.f;
#pragma unroll
      for (int c = 0; c < COLUMNS; ++c) {
        const int col = c * EACH + column;
        if (c * EACH >= V) break;
        const float v = s_values[hh * V + min(col, V - 1)];
        float dot = 0.f, o = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) S[c][r] *= d4[r / 4][r % 4];
        if (DELTA) {
#pragma unroll
          for (int r = 0; r < R; ++r) dot = fmaf(S[c][r], k4[r / 4][r % 4], dot);
          dot = group_sum<L>(dot);
        }
        const float u = DELTA ? beta * (v - dot) : beta * v;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          S[c][r] = fmaf(k4[r / 4][r % 4], u, S[c][r]);
          o = fmaf(S[c][r], q4[r / 4][r % 4], o);
        }
        o = group_sum<L>(o);
        if (sub == 0) s_out[parity][col] = o;
      }
      __syncthreads();
#pragma unroll
      for (int c = 0; c < COLUMNS; ++c) {
        const int col = c * EACH + column;
        if (col >= V) break;
        float* to = state + (uint32_t)((h * V + col) * D);
#pragma unroll
        for (int r4 = 0; r4 < R / 4; ++r4) {
          const int d = r4 * (4 * L) + sub * 4;
          if (d < D) *reinterpret_cast<f32x4*>(to + d) = f32x4{S[c][4 * r4], S[c][4 * r4 + 1], S[c][4 * r4 + 2], S[c][4 * r4 + 3]};
        }
      }
      if (tid < (V + PAE_WAVE - 1) / PAE_WAVE * PAE_WAVE) {  // whole wavefronts
        float ss = 0.f;
        for (int v = lane; v < V; v += PAE_WAVE) ss = fmaf(s_out[parity][v], s_out[parity][v], ss);
        ss = wave_sum(ss);
        const float inv = 1.0f / sqrtf(ss / (float)V + p.norm_eps);
        const float gz = p.gate_sigmoid ? 1.0f / (1.0f + expf(-z)) : silu_f(z);
        if (tid < V) ((T*)p.out)[(t * H + h) * V + tid] = from_f32<T>(s_out[parity][tid] * inv * w * gz);
      }
      parity ^= 1;
#pragma unroll
      for (int c = 0; c < COLUMNS; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) S[c][r] = next[c][r];
    }
  }
}

template <typename T, int L>
void launch_of(int kind, const TokensStep& p, int num_seqs, hipStream_t stream) {
  const int heads = p.H / p.G;
  const int lds = ((heads * p.V + 3) / 4 * 4 + (kind == TOKENS_DELTA ? 0 : heads * L * R) + 2 * heads) * 4;
  const dim3 grid(p.G, num_seqs);
  if (kind == TOKENS_DELTA) recurrent_tokens_kernel<T, L, TOKENS_DELTA><<<grid, THREADS, lds, stream>>>(p);
  else if (kind == TOKENS_CHANNEL_DELTA) recurrent_tokens_kernel<T, L, TOKENS_CHANNEL_DELTA><<<grid, THREADS, lds, stream>>>(p);
  else recurrent_tokens_kernel<T, L, TOKENS_LINEAR><<<grid, THREADS, lds, stream>>>(p);
}

}  // namespace

// Whether a step of that many single tokens is ahead in one launch.  A workgroup takes the value heads of its key head one after another, 2 us each:
// always up to four of them, beyond that where workgroups are so many that the units are busy anyway (us, separate kernels and one launch, heads of 128 by
// 128: 4 key and 16 value heads for 1 / 8 / 64 sequences 12.2 / 16.2 / 49.3 and 11.6 / 12.7 / 26.4; 2 and 16 for 1 / 16 / 32 / 64 12.2 / 21.8 / 33.1 / 48.7 and
// 19.9 / 21.9 / 29.0 / 34.6; 1 and 16 for 1 / 64 / 128 11.9 / 48.7 / 78.3 and 35.1 / 52.4 / 61.3; 2 and 28 of 64 by 64 for 32 / 64 21.0 / 30.7 and 24.1 / 29.9).
extern "C" int pae_tokens_step_pays(int num_seqs, int G, int H) { return H <= 4 * G || (int64_t)num_seqs * G * G >= 8 * (int64_t)H; }

// As many tokens as sequences: single tokens (a run of several beside empty ones is worked on token by token here).  The other
// bounds are what a workgroup holds, lanes of 8 rows by two columns and what the value heads of a key head have in LDS, and that four rows of
// a column are read at a time.
bool takes_tokens_step(int num_tokens, int num_seqs, int G, int H, int D, int V, const float* state, int64_t slot_stride) {
  const int lanes = D <= 64 ? 8 : 16;
  return num_tokens == num_seqs && pae_tokens_step_pays(num_seqs, G, H) && D % 4 == 0 && slot_stride % 4 == 0 && (uintptr_t)state % 16 == 0 && D > 32 &&
         D <= 128 && V <= COLUMNS * THREADS / lanes && (int64_t)(H / G) * (V + lanes * R) <= MOST_VALUES;
}

void launch_tokens_step(int kind, int dtype, const TokensStep& p, int num_seqs, hipStream_t stream) {
  if (dtype == PAE_F32) {
    if (p.D <= 64) launch_of<float, 8>(kind, p, num_seqs, stream);
    else launch_of<float, 16>(kind, p, num_seqs, stream);
  } else {
    if (p.D <= 64) launch_of<bf16_t, 8>(kind, p, num_seqs, stream);
    else launch_of<bf16_t, 16>(kind, p, num_seqs, stream);
  }
}
