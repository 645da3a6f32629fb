// Causal attention over the paged cache in float32 arithmetic, two kernels that compute the same bits: one wavefront per
// (token, query head) for any size, and a workgroup for the query heads of one key/value head and
// a few tokens, which brings the keys and values to LDS once for all of them (below).
//
// These are the kernels every size goes through in float32 and the ones bfloat16
// falls back to when the matrix-core kernels do not take a shape.  A step's
// tokens are flat: token t belongs to sequence tok_seq[t] and stands at
// positions[t]; its keys are the cache slots of positions start..pos of that
// sequence, start = max(0, pos - window + 1) (window 0: every earlier key).  The
// rule is the reference's mask (engine/attention.py:474-487: key j is visible iff
// j <= query position and j < kv length) plus the window, which it lacks.
// KV head j serves query heads j*g .. (j+1)*g-1 (engine/attention.py:72-74).
//
// Keys are taken in chunks of 64 aligned to multiples of 64 from position 0,
// lane = key within the chunk: every chunk's weights have the chunk's largest score for their reference, and the
// chunks' sums are added in order, in float32 (`add_chunk`).  What a
// (token, head) computes therefore depends on nothing but its own position:
// not on how the step was cut, nor on what else is in the batch, nor on whether a workgroup walks the chunks or
// several share them out (few tokens at many keys: `split_chunks`).
//
// Three things beyond the reference's attention, each switched by a parameter: values of their own
// width `vd` (keys and queries stay `hd` wide), a cap on the scores (s <- cap * tanh(s / cap),
// cap 0: none), and one learned sink per query head, a number that joins the softmax's denominator
// as exp(sink) without a key or a value of its own (sinks null: none).
//
// And four more, for designs that have them: a mask in chunks (`chunked`: the `window` is then a
// chunk length, and position p sees the keys from p - p % window on, chunk borders at multiples of the length from the first token
// of the sequence); a bias by distance, score -= slopes[head] * (p - key) (slopes null: none); a gate
// on the output, out *= sigmoid(gate[token][head][feature]), or with one number a head, gate[token][head]
// (`gate_per_head`) (gate null: none); and values that are
// the first `vd` features of the key rows themselves (`shared_kv`, one latent row per token that
// serves as key and as value: v_cache is then not read).
#include "common.h"
#include "api.h"

// What a chunk's weights are taken relative to: its largest score, or the least number there is where all its scores are minus infinity (numbers that
// overflowed, or a bias that hides a key), whose weights are then zero as they are beside a score that is a number.  (Once a chunk and not
// where chunks are added: there it cost 2.5 % of a prompt of 1,500 tokens.)
__device__ __forceinline__ float reference_of(float largest) { return fmaxf(largest, -3.402823466e38f); }

// A chunk's sums (its largest score, the sum of its weights, the weighted values) onto those of the chunks before it.
template <int MAXD>
__device__ __forceinline__ void add_chunk(float (&acc)[MAXD], float& m, float& l, const float (&sum)[MAXD], float m_chunk, float l_chunk) {
  const float m_new = fmaxf(m, m_chunk);
  const float before = expf(m - m_new), now = expf(m_chunk - m_new);  // 0 and 1 on the first chunk (m = -inf)
  l = l * before + l_chunk * now;
  m = m_new;
#pragma unroll
  for (int i = 0; i < MAXD; ++i) acc[i] = acc[i] * before + sum[i] * now;
}

// The row's output from its sums: the sink joins the denominator, then the gate.
template <typename T, int MAXD>
__device__ __forceinline__ void finish_row(T* __restrict__ o, const float (&acc)[MAXD], float m, float l, int vd, int lane,
                                           const float* __restrict__ sink, const T* __restrict__ gate, int gate_per_head) {
  float keep = 1.f;  // what the sums keep when the sink raises the reference point
  if (sink) {
    const float m_all = fmaxf(m, *sink);
    keep = expf(m - m_all);
    l = l * keep + expf(*sink - m_all);
  }
  const float inv = keep / l;
#pragma unroll
  for (int i = 0; i < MAXD; ++i) {
    const int d = lane + i * PAE_WAVE;
    if (d < vd) {
      float v = acc[i] * inv;
      if (gate) v *= 1.0f / (1.0f + expf(-to_f32(gate[gate_per_head ? 0 : d])));
      o[d] = from_f32<T>(v);
    }
  }
}

template <typename T, int MAXD>  // MAXD: output features per lane, value width <= 64 * MAXD
__global__ void paged_attention_generic_kernel(
    T* __restrict__ out, int64_t out_stride, const T* __restrict__ q, int64_t q_stride,
    const T* __restrict__ k_cache, const T* __restrict__ v_cache, const int* __restrict__ positions,
    const int* __restrict__ tok_seq, const int* __restrict__ block_tables, int max_blocks, int bs,
    int nh, int nkv, int hd, int vd, float scale, int window, float cap, const float* __restrict__ sinks,
    int chunked, const float* __restrict__ slopes, const T* __restrict__ gate, int64_t gate_stride, int gate_per_head,
    int shared_kv) {
  extern __shared__ float lds[];  // [hd] query, [64] probabilities
  float* q_lds = lds;
  float* p_lds = lds + hd;
  const int t = blockIdx.x;
  const int head = blockIdx.y;
  const int lane = threadIdx.x;
  const int kvh = head / (nh / nkv);
  const int pos = positions[t];
  const int* table = block_tables + (int64_t)tok_seq[t] * max_blocks;
  const int start = window <= 0 ? 0 : (chunked ? pos - pos % window : (pos - window + 1 > 0 ? pos - window + 1 : 0));
  const float slope = slopes ? slopes[head] : 0.f;

  const T* q_row = q + (int64_t)t * q_stride + (int64_t)head * hd;
  for (int d = lane; d < hd; d += PAE_WAVE) q_lds[d] = to_f32(q_row[d]);
  __syncthreads();

  float acc[MAXD];
#pragma unroll
  for (int i = 0; i < MAXD; ++i) acc[i] = 0.f;
  float m = -INFINITY, l = 0.f;

  for (int base = (start / PAE_WAVE) * PAE_WAVE; base <= pos; base += PAE_WAVE) {
    const int key = base + lane;
    const bool valid = key >= start && key <= pos;
    int row = 0;  // this lane's key row in the pool, in units of head_dim elements
    float s = -INFINITY;
    if (valid) {
      const int blk = table[key / bs];
      row = (blk * nkv + kvh) * bs + key % bs;
      const T* kr = k_cache + (int64_t)row * hd;
      float dot = 0.f;
      for (int d = 0; d < hd; ++d) dot = fmaf(q_lds[d], to_f32(kr[d]), dot);
      s = dot * scale;
      if (slopes) s -= slope * (float)(pos - key);
      if (cap > 0.f) s = cap * tanhf(s / cap);
    }
    const float m_chunk = reference_of(wave_max(s));
    const float p = valid ? expf(s - m_chunk) : 0.f;
    const float l_chunk = wave_sum(p);
    p_lds[lane] = p;
    __syncthreads();
    const int first = (start > base ? start - base : 0);
    const int last = (pos - base < PAE_WAVE - 1 ? pos - base : PAE_WAVE - 1);
    float sum[MAXD];
#pragma unroll
    for (int i = 0; i < MAXD; ++i) sum[i] = 0.f;
    for (int j = first; j <= last; ++j) {
      const float pj = p_lds[j];
      const int rj = __shfl(row, j, PAE_WAVE);
      // values are transposed within a page: [block][kv head][feature][offset in page]; shared with
      // the keys they are the head of the key row
      const T* vr = shared_kv ? k_cache + (int64_t)rj * hd : v_cache + (int64_t)(rj / bs) * bs * vd + rj % bs;
      const int64_t step = shared_kv ? 1 : bs;
#pragma unroll
      for (int i = 0; i < MAXD; ++i) {
        const int d = lane + i * PAE_WAVE;
        if (d < vd) sum[i] = fmaf(pj, to_f32(vr[(int64_t)d * step]), sum[i]);
      }
    }
    add_chunk<MAXD>(acc, m, l, sum, m_chunk, l_chunk);
    __syncthreads();
  }
  finish_row<T, MAXD>(out + (int64_t)t * out_stride + (int64_t)head * vd, acc, m, l, vd, lane, sinks ? sinks + head : nullptr,
                      gate ? gate + (int64_t)t * gate_stride + (gate_per_head ? head : (int64_t)head * vd) : nullptr, gate_per_head);
}

// The same for float32 rows that can be read four numbers at a time: a workgroup of eight wavefronts takes up to 16 (token,
// query head) rows that share a key/value head, and walks the chunks of 64 keys that any of them
// sees.  A chunk's keys and values come to LDS once, by 16-byte loads, the next chunk's on their way
// meanwhile; a wavefront computes up to two rows together, lane = key for the scores, lane = feature for
// the sums, so that a key or value read from LDS serves two rows.  Every row does the operations of the
// kernel above in its order and over its own keys only: the bits are the same, and a row never touches a
// key it does not see.
//
// What bound the kernel above: every lane read its own key row number by number (64 rows of 512 bytes, a
// load instruction per number), and every (token, head) read the keys and values again.  Measured, 12 heads over 2
// of 128, float32: three prompts of 601 tokens in all 262 -> 58 us, a token each behind them 92 -> 27, one prompt of 601 tokens 647 ->
// 117, eight single tokens at 4,096 1,551 -> 338; 8 heads over 2 of 256, where six of 256 registers do not fit and lie in memory, 399 -> 77,
// 177 -> 47, 900 -> 132, 2,534 -> 521.  What is left is the chain of a workgroup's chunks, 5 us each, which few tokens share out
// (`split_chunks`).  Where a workgroup has
// eight rows or fewer (a token's heads, mostly) a wavefront takes one: the chain is a row's then, and registers are left to ask
// LDS for more at once (a token at 4,096 330 -> 275 us, three at 250 25.6 -> 22.2, at heads of 64 18.6 -> 14.0; eight at 1,000, heads
// of 256, 136 -> 114).  Loads
// under conditions (keys beside those in sight) had the compiler wait for each in turn (twice the time for prompts), and
// four wavefronts of four rows instead of eight of two took half as long again.
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define PAE_ROWS_WAVES 8
#define PAE_ROWS_EACH 2
#define PAE_ROWS_MOST (PAE_ROWS_WAVES * PAE_ROWS_EACH)
#define SPLIT_GROUPS 128         // up to so many workgroups' chunks are shared out
#define SPLIT_UNITS 256          // over so many workgroups
#define SPLIT_FLOATS (16 << 20)  // numbers that their sums may take: 64 MiB

// SPLIT: the workgroup looks at every gridDim.z-th chunk of 64 keys from chunk blockIdx.z on, and every row's sums over each go to
// `chunk_sums` [(token, head)][chunk][vd] and `chunk_ml` [(token, head)][chunk][2], for the kernel below to add up in the order of the chunks
// (`chunks` is how many the tables have room for).
template <int MAXD, int EACH, bool SPLIT>  // keys and values at most 64 * MAXD wide; rows of a wavefront: one where eight rows are all there are
__global__ __launch_bounds__(PAE_WAVE * PAE_ROWS_WAVES) void paged_attention_rows_kernel(
    float* __restrict__ out, int64_t out_stride, const float* __restrict__ q, int64_t q_stride,
    const float* __restrict__ k_cache, const float* __restrict__ v_cache, const int* __restrict__ positions,
    const int* __restrict__ tok_seq, const int* __restrict__ block_tables, int max_blocks, int bs, int num_tokens,
    int nh, int nkv, int hd, int vd, float scale, int window, float cap, const float* __restrict__ sinks,
    int chunked, const float* __restrict__ slopes, const float* __restrict__ gate, int64_t gate_stride,
    int gate_per_head, int toks, int heads_each, int chunks, float* __restrict__ chunk_sums, float* __restrict__ chunk_ml) {
  constexpr int FOURS = 16 * MAXD / PAE_ROWS_WAVES;  // that a thread brings of a chunk's keys, and of its values
  extern __shared__ float lds[];
  const int kst = hd + 4, vst = vd + 4;  // row strides that spread a quad's reads and writes over the banks
  float* k_lds = lds;                    // [64 keys][kst]
  float* v_lds = lds + PAE_WAVE * kst;   // [64 keys][vst]
  float* p_lds = v_lds + PAE_WAVE * vst; // [wavefront][row][64]
  float* q_lds = p_lds + PAE_ROWS_MOST * PAE_WAVE;  // [row][hd]
  const int tid = threadIdx.x, lane = tid % PAE_WAVE;
  const int wave = __builtin_amdgcn_readfirstlane(tid / PAE_WAVE);
  const int g = nh / nkv;
  const int parts = (g + heads_each - 1) / heads_each;
  const int kvh = blockIdx.y / parts, head0 = (blockIdx.y % parts) * heads_each;
  const int heads = min(heads_each, g - head0);
  const int t0 = blockIdx.x * toks;
  p_lds += wave * EACH * PAE_WAVE;

  // the wavefront's rows: row = token of the tile * heads + head
  int tok[EACH], head[EACH], pos[EACH], start[EACH];
  float acc[EACH][MAXD], m[EACH], l[EACH];
  bool live[EACH];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int row = wave + i * PAE_ROWS_WAVES;
    live[i] = row < toks * heads && t0 + row / heads < num_tokens;
    tok[i] = live[i] ? t0 + row / heads : t0;
    head[i] = kvh * g + head0 + row % heads;
    pos[i] = __builtin_amdgcn_readfirstlane(positions[tok[i]]);
    start[i] = window <= 0 ? 0 : (chunked ? pos[i] - pos[i] % window : (pos[i] - window + 1 > 0 ? pos[i] - window + 1 : 0));
    m[i] = -INFINITY;
    l[i] = 0.f;
#pragma unroll
    for (int d = 0; d < MAXD; ++d) acc[i][d] = 0.f;
  }

  // the tile's queries, and which fours of a chunk a thread brings
  for (int c = tid; c < toks * heads * (hd / 4); c += PAE_WAVE * PAE_ROWS_WAVES) {
    const int row = c / (hd / 4), d = (c % (hd / 4)) * 4;
    const int t = min(t0 + row / heads, num_tokens - 1);
    const float* src = q + (int64_t)t * q_stride + (int64_t)(kvh * g + head0 + row % heads) * hd + d;
    *(float4*)(q_lds + row * hd + d) = make_float4(src[0], src[1], src[2], src[3]);
  }
  // (threads without a four of their own bring the last one again)
  const int span = min(bs, PAE_WAVE);  // keys of a chunk that lie in one page; a power of two
  int k_key[FOURS], k_dim[FOURS], v_key[FOURS], v_dim[FOURS];
#pragma unroll
  for (int u = 0; u < FOURS; ++u) {
    const int c = tid + u * PAE_WAVE * PAE_ROWS_WAVES;
    const int ck = min(c, PAE_WAVE * hd / 4 - 1), cv = min(c, PAE_WAVE * vd / 4 - 1);
    k_key[u] = ck / (hd / 4);
    k_dim[u] = (ck % (hd / 4)) * 4;
    // neighbouring threads take a feature's run of keys within a page, then the next feature
    v_key[u] = cv / (span / 4 * vd) * span + cv % (span / 4) * 4;
    v_dim[u] = cv % (span / 4 * vd) / (span / 4);
  }

  // tokens of one sequence at a time (neighbours in a step mostly are); the first barrier below is behind the queries, too
  int at = t0;
  const int t_end = min(t0 + toks, num_tokens);
  while (at < t_end) {
    const int s = __builtin_amdgcn_readfirstlane(tok_seq[at]);
    int low = 0x7fffffff, high = -1, next = at;
    for (; next < t_end && __builtin_amdgcn_readfirstlane(tok_seq[next]) == s; ++next) {
      const int p = __builtin_amdgcn_readfirstlane(positions[next]);
      const int first = window <= 0 ? 0 : (chunked ? p - p % window : (p - window + 1 > 0 ? p - window + 1 : 0));
      low = min(low, first);
      high = max(high, p);
    }
    if (high < low) {  // tokens that see no key, position -1: their table need not name a page
      at = next;
      continue;
    }
    const int* table = block_tables + (int64_t)s * max_blocks;
    // A chunk's keys and values, four numbers at a time (keys [key][feature], values [page][feature][offset]); what a
    // thread brings lies at the same places of every chunk.
    // No load stands under a condition: pages before and behind those in sight are read as the nearest one in
    // sight, and what lies beside the keys in sight is never looked at.
    const int page_low = low / bs, page_high = high / bs;
    f32x4 k_reg[FOURS], v_reg[FOURS];
    auto fetch = [&](int base) {
      const int page0 = base / bs, off0 = base % bs;
      int k_page[FOURS], v_page[FOURS];
#pragma unroll
      for (int u = 0; u < FOURS; ++u) {
        k_page[u] = table[min(max(page0 + k_key[u] / span, page_low), page_high)];
        v_page[u] = table[min(max(page0 + v_key[u] / span, page_low), page_high)];
      }
#pragma unroll
      for (int u = 0; u < FOURS; ++u)
        k_reg[u] = *(const f32x4*)(k_cache + (((int64_t)k_page[u] * nkv + kvh) * bs + off0 + k_key[u] % span) * hd + k_dim[u]);
#pragma unroll
      for (int u = 0; u < FOURS; ++u)
        v_reg[u] = *(const f32x4*)(v_cache + (((int64_t)v_page[u] * nkv + kvh) * vd + v_dim[u]) * bs + off0 + v_key[u] % span);
    };
    const int step = SPLIT ? gridDim.z * PAE_WAVE : PAE_WAVE;
    int base0 = (low / PAE_WAVE) * PAE_WAVE;
    if (SPLIT) {
      base0 = blockIdx.z * PAE_WAVE;
      if (base0 + PAE_WAVE <= low) base0 += (low - base0) / step * step;
      if (base0 + PAE_WAVE <= low) base0 += step;  // the first of the workgroup's chunks with a key in sight
      if (base0 > high) {
        at = next;
        continue;
      }
    }
    // (shared out, heads of more than 192 have no registers for the chunk after this one: eight tokens at 1,000 keys 25.4 us with it, 21 without)
    constexpr bool AHEAD = !SPLIT || MAXD < 4;
    if (AHEAD) fetch(base0);
    for (int base = base0; base <= high; base += step) {
      if (!AHEAD) fetch(base);
      __syncthreads();  // the chunk before has been read
#pragma unroll
      for (int u = 0; u < FOURS; ++u) *(f32x4*)(k_lds + k_key[u] * kst + k_dim[u]) = k_reg[u];
#pragma unroll
      for (int u = 0; u < FOURS; ++u) {
        float* v = v_lds + v_key[u] * vst + v_dim[u];
        v[0] = v_reg[u].x;
        v[vst] = v_reg[u].y;
        v[2 * vst] = v_reg[u].z;
        v[3 * vst] = v_reg[u].w;
      }
      __syncthreads();
      if (AHEAD && base + step <= high) fetch(base + step);
      bool on[EACH];
      bool any = false, whole = true;
#pragma unroll
      for (int i = 0; i < EACH; ++i) {
        on[i] = live[i] && tok[i] >= at && tok[i] < next && base <= pos[i] && base + PAE_WAVE > start[i];
        any = any || on[i];
        whole = whole && (!live[i] || (on[i] && start[i] <= base && pos[i] >= base + PAE_WAVE - 1));
      }
      if (!any) continue;
      // scores: the lane's key against every row
      float dot[EACH];
      int q_row[EACH];
#pragma unroll
      for (int i = 0; i < EACH; ++i) {
        dot[i] = 0.f;
        q_row[i] = live[i] ? (wave + i * PAE_ROWS_WAVES) * hd : 0;
      }
      const float* kr = k_lds + lane * kst;
#pragma unroll(EACH == 1 && MAXD <= 2 ? 8 : 4)
      for (int d = 0; d < hd; d += 4) {
        const float4 k4 = *(const float4*)(kr + d);
#pragma unroll
        for (int i = 0; i < EACH; ++i) {
          const float4 q4 = *(const float4*)(q_lds + q_row[i] + d);
          dot[i] = fmaf(q4.x, k4.x, dot[i]);
          dot[i] = fmaf(q4.y, k4.y, dot[i]);
          dot[i] = fmaf(q4.z, k4.z, dot[i]);
          dot[i] = fmaf(q4.w, k4.w, dot[i]);
        }
      }
      const int key = base + lane;
      float sc[EACH], m_chunk[EACH], p[EACH], l_chunk[EACH], sum[EACH][MAXD];
#pragma unroll
      for (int i = 0; i < EACH; ++i) {
        sc[i] = dot[i] * scale;
        if (slopes) sc[i] -= slopes[head[i]] * (float)(pos[i] - key);
        if (cap > 0.f) sc[i] = cap * tanhf(sc[i] / cap);
        if (!(key >= start[i] && key <= pos[i])) sc[i] = -INFINITY;
        m_chunk[i] = reference_of(wave_max(sc[i]));
      }
#pragma unroll
      for (int i = 0; i < EACH; ++i) {  // the rows' reductions side by side; rows that are not on keep what they have
        p[i] = key >= start[i] && key <= pos[i] ? expf(sc[i] - m_chunk[i]) : 0.f;
        l_chunk[i] = wave_sum(p[i]);
      }
#pragma unroll
      for (int i = 0; i < EACH; ++i) {
        if (on[i]) p_lds[i * PAE_WAVE + lane] = p[i];
#pragma unroll
        for (int d = 0; d < MAXD; ++d) sum[i][d] = 0.f;
      }
      // sums: the lane's features over the keys in order (the wavefront's own p: no barrier, its LDS operations are in order)
      __builtin_amdgcn_wave_barrier();
      if (whole) {
#pragma unroll(EACH == 1 && MAXD <= 2 ? 4 : 2)
        for (int j = 0; j < PAE_WAVE; j += 4) {
          float v[4][MAXD];
#pragma unroll
          for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int d = 0; d < MAXD; ++d) v[u][d] = v_lds[(j + u) * vst + min(lane + d * PAE_WAVE, vd - 1)];
#pragma unroll
          for (int i = 0; i < EACH; ++i) {
            if (!live[i]) continue;
            const float4 p4 = *(const float4*)(p_lds + i * PAE_WAVE + j);
#pragma unroll
            for (int d = 0; d < MAXD; ++d) {
              sum[i][d] = fmaf(p4.x, v[0][d], sum[i][d]);
              sum[i][d] = fmaf(p4.y, v[1][d], sum[i][d]);
              sum[i][d] = fmaf(p4.z, v[2][d], sum[i][d]);
              sum[i][d] = fmaf(p4.w, v[3][d], sum[i][d]);
            }
          }
        }
      } else {
#pragma unroll
        for (int i = 0; i < EACH; ++i) {
          if (!on[i]) continue;
          const int first = max(0, start[i] - base), last = min(PAE_WAVE - 1, pos[i] - base);
          auto add = [&](int j, float p) {
#pragma unroll
            for (int d = 0; d < MAXD; ++d)
              if (lane + d * PAE_WAVE < vd) sum[i][d] = fmaf(p, v_lds[j * vst + lane + d * PAE_WAVE], sum[i][d]);
          };
          int j = first;
#pragma unroll 1
          for (; j <= last && j % 4; ++j) add(j, p_lds[i * PAE_WAVE + j]);
#pragma unroll 1
          for (; j + 3 <= last; j += 4) {
            const float4 p4 = *(const float4*)(p_lds + i * PAE_WAVE + j);
            float v[4][MAXD];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
              for (int d = 0; d < MAXD; ++d) v[u][d] = v_lds[(j + u) * vst + min(lane + d * PAE_WAVE, vd - 1)];
#pragma unroll
            for (int d = 0; d < MAXD; ++d) {
              sum[i][d] = fmaf(p4.x, v[0][d], sum[i][d]);
              sum[i][d] = fmaf(p4.y, v[1][d], sum[i][d]);
              sum[i][d] = fmaf(p4.z, v[2][d], sum[i][d]);
              sum[i][d] = fmaf(p4.w, v[3][d], sum[i][d]);
            }
          }
#pragma unroll 1
          for (; j <= last; ++j) add(j, p_lds[i * PAE_WAVE + j]);
        }
      }
#pragma unroll
      for (int i = 0; i < EACH; ++i) {
        if (!on[i]) continue;
        if (!SPLIT) {
          add_chunk<MAXD>(acc[i], m[i], l[i], sum[i], m_chunk[i], l_chunk[i]);
          continue;
        }
        const int64_t part = ((int64_t)tok[i] * nh + head[i]) * chunks + base / PAE_WAVE;
        if (lane == 0) *reinterpret_cast<float2*>(chunk_ml + 2 * part) = make_float2(m_chunk[i], l_chunk[i]);
#pragma unroll
        for (int d = 0; d < MAXD; ++d)
          if (lane + d * PAE_WAVE < vd) chunk_sums[part * vd + lane + d * PAE_WAVE] = sum[i][d];
      }
    }
    at = next;
  }
  if (SPLIT) return;
#pragma unroll
  for (int i = 0; i < EACH; ++i)
    if (live[i])
      finish_row<float, MAXD>(out + (int64_t)tok[i] * out_stride + (int64_t)head[i] * vd, acc[i], m[i], l[i], vd, lane, sinks ? sinks + head[i] : nullptr,
                              gate ? gate + (int64_t)tok[i] * gate_stride + (gate_per_head ? head[i] : (int64_t)head[i] * vd) : nullptr, gate_per_head);
}

// A row's chunks, added in their order as the kernels above add them: one wavefront per (token, query head), eight chunks'
// sums on their way together.
template <int MAXD>
__global__ __launch_bounds__(PAE_WAVE) void paged_attention_chunks_kernel(
    float* __restrict__ out, int64_t out_stride, const float* __restrict__ chunk_sums, const float* __restrict__ chunk_ml, int chunks,
    const int* __restrict__ positions, int nh, int vd, int window, const float* __restrict__ sinks, int chunked,
    const float* __restrict__ gate, int64_t gate_stride, int gate_per_head) {
  constexpr int AHEAD = 8;
  const int t = blockIdx.x, head = blockIdx.y, lane = threadIdx.x, pos = positions[t];
  const int start = window <= 0 ? 0 : (chunked ? pos - pos % window : (pos - window + 1 > 0 ? pos - window + 1 : 0));
  const int64_t row = ((int64_t)t * nh + head) * chunks;
  const int last = pos < 0 ? -1 : pos / PAE_WAVE;
  float acc[MAXD], m = -INFINITY, l = 0.f;
#pragma unroll
  for (int i = 0; i < MAXD; ++i) acc[i] = 0.f;
  for (int c0 = start / PAE_WAVE; c0 <= last; c0 += AHEAD) {
    float2 ml[AHEAD];
    float sum[AHEAD][MAXD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const int64_t part = row + min(c0 + u, last);
      ml[u] = *reinterpret_cast<const float2*>(chunk_ml + 2 * part);
#pragma unroll
      for (int i = 0; i < MAXD; ++i) sum[u][i] = chunk_sums[part * vd + min(lane + i * PAE_WAVE, vd - 1)];
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (c0 + u <= last) add_chunk<MAXD>(acc, m, l, sum[u], ml[u].x, ml[u].y);
  }
  finish_row<float, MAXD>(out + (int64_t)t * out_stride + (int64_t)head * vd, acc, m, l, vd, lane, sinks ? sinks + head : nullptr,
                          gate ? gate + (int64_t)t * gate_stride + (gate_per_head ? head : (int64_t)head * vd) : nullptr, gate_per_head);
}

// Whether the rows kernel takes a call: rows and pages that can be read four numbers at a time, and a chunk's keys and values
// in a compute unit's LDS (150 KB at heads of 256).
static bool rows_kernel_takes(const void* k_cache, const void* v_cache, int bs, int hd, int vd, int shared_kv) {
  return !shared_kv && bs % 4 == 0 && (bs >= PAE_WAVE ? bs % PAE_WAVE == 0 : PAE_WAVE % bs == 0) && hd % 4 == 0 && vd <= 256 &&
         hd <= 256 && (uintptr_t)k_cache % 16 == 0 && (uintptr_t)v_cache % 16 == 0;
}

// Tokens that share a workgroup's keys, its heads of each, and the parts of a key/value head's query heads.  Several tokens where
// there are workgroups enough (decode steps: a token each).
static int rows_of_a_workgroup(int num_tokens, int nh, int nkv, int& heads_each, int& parts) {
  const int g = nh / nkv;
  heads_each = g < PAE_ROWS_MOST ? g : PAE_ROWS_MOST;
  parts = (g + heads_each - 1) / heads_each;
  return (int64_t)num_tokens * nkv * parts >= 512 ? PAE_ROWS_MOST / heads_each : 1;
}

// Chunks of keys that are shared out, or 1: a workgroup walks them all.  Shared out where the walks would leave half the chip idle and more
// and the tables have room for three chunks (a token at 60 keys 10.0 and 12.1; 14 heads of 64 at 75 about 8 and 9), over one workgroup a compute unit
// in all: a count by the tables' room would launch one for every chunk that a longer sequence or a rounded width makes room for, which costs its
// start also where it finds no key.  12 heads over 2 of 128, in us, walked, shared, and with a workgroup for every chunk in the tables: three
// tokens at 200 keys of 1,024 21.4, 12.8 and 12.7; eight at 1,000 73, 14.6 and 14.6, at 4,000 278, 42 and 53; 32 at 200 21.6, 13.2 and 22.3; 64 at
// 130 17.9, 16.0 and 37.6, at 1,000 78, 49 and 70; one at 2,000 beside 63 at 130 143, 80 and 99.  Over 783 such calls (9 kinds of heads) 0.473 of the walk's
// time and 1.36 at worst (60 keys), by the tables' room 0.523 and 3.1, with two workgroups a unit 0.49 and 1.5.  Prompts walk (200 tokens, 400 workgroups, 33 us,
// by chunks 44).  (All with a token a workgroup: where several share one, from 512 such workgroups on, they walk.)
static int split_chunks(int num_tokens, int nh, int nkv, int vd, int max_blocks, int bs) {
  int heads_each, parts;
  rows_of_a_workgroup(num_tokens, nh, nkv, heads_each, parts);
  const int64_t chunks = ((int64_t)max_blocks * bs + PAE_WAVE - 1) / PAE_WAVE;
  const int64_t groups = (int64_t)num_tokens * nkv * parts;
  if (chunks < 3 || chunks > 65535 || groups > SPLIT_GROUPS || (int64_t)num_tokens * nh * chunks * (vd + 2) > SPLIT_FLOATS) return 1;
  return (int)chunks;
}

static int launch_rows(float* out, int64_t out_stride, const float* q, int64_t q_stride, const float* k_cache,
                       const float* v_cache, const int* positions, const int* tok_seq, const int* block_tables,
                       int max_blocks, int bs, int num_tokens, int nh, int nkv, int hd, int vd, float scale, int window,
                       float cap, const float* sinks, int chunked, const float* slopes, const float* gate,
                       int64_t gate_stride, int gate_per_head, float* scratch, hipStream_t stream) {
  int heads_each, parts;
  const int toks = rows_of_a_workgroup(num_tokens, nh, nkv, heads_each, parts);
  const int chunks = scratch ? split_chunks(num_tokens, nh, nkv, vd, max_blocks, bs) : 1;
  float* part_ml = scratch;
  float* part_sums = scratch ? scratch + (int64_t)2 * num_tokens * nh * chunks : nullptr;
  const size_t lds = (size_t)(PAE_WAVE * (hd + 4 + vd + 4) + PAE_ROWS_MOST * (PAE_WAVE + hd)) * sizeof(float);
  const dim3 grid((num_tokens + toks - 1) / toks, nkv * parts, chunks > 1 ? min(chunks, SPLIT_UNITS / (num_tokens * nkv * parts)) : 1);
#define PAE_LAUNCH_EACH(MAXD, EACH, SPLIT)                                                                            \
  do {                                                                                                                \
    if (lds > 65536) {                                                                                                \
      const hipError_t err = hipFuncSetAttribute((const void*)paged_attention_rows_kernel<MAXD, EACH, SPLIT>,         \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);               \
      if (err != hipSuccess) return pae_fail("attention: %zu bytes of LDS refused: %s", lds, hipGetErrorString(err)); \
    }                                                                                                                 \
    paged_attention_rows_kernel<MAXD, EACH, SPLIT><<<grid, PAE_WAVE * PAE_ROWS_WAVES, lds, stream>>>(                 \
        out, out_stride, q, q_stride, k_cache, v_cache, positions, tok_seq, block_tables, max_blocks, bs, num_tokens, \
        nh, nkv, hd, vd, scale, window, cap, sinks, chunked, slopes, gate, gate_stride, gate_per_head, toks, heads_each, \
        chunks, part_sums, part_ml);                                                                                          \
  } while (0)
#define PAE_LAUNCH(MAXD)                                                                                              \
  do {                                                                                                                \
    if (chunks > 1) {                                                                                                 \
      if (toks * heads_each <= PAE_ROWS_WAVES) PAE_LAUNCH_EACH(MAXD, 1, true);                                        \
      else PAE_LAUNCH_EACH(MAXD, PAE_ROWS_EACH, true);                                                                \
      paged_attention_chunks_kernel<MAXD><<<dim3(num_tokens, nh), PAE_WAVE, 0, stream>>>(                             \
          out, out_stride, part_sums, part_ml, chunks, positions, nh, vd, window, sinks, chunked, gate, gate_stride, gate_per_head); \
    } else if (toks * heads_each <= PAE_ROWS_WAVES) PAE_LAUNCH_EACH(MAXD, 1, false);                                  \
    else PAE_LAUNCH_EACH(MAXD, PAE_ROWS_EACH, false);                                                                 \
  } while (0)
  const int wide = hd > vd ? hd : vd;
  if (wide <= 64) PAE_LAUNCH(1);
  else if (wide <= 128) PAE_LAUNCH(2);
  else if (wide <= 192) PAE_LAUNCH(3);
  else PAE_LAUNCH(4);
#undef PAE_LAUNCH
#undef PAE_LAUNCH_EACH
  return pae_check_launch("paged_attention_rows");
}

template <typename T>
static int launch_generic(void* out, int64_t out_stride, const void* q, int64_t q_stride, const void* k_cache,
                          const void* v_cache, const int* positions, const int* tok_seq,
                          const int* block_tables, int max_blocks, int bs, int num_tokens, int nh, int nkv,
                          int hd, int vd, float scale, int window, float cap, const float* sinks, int chunked,
                          const float* slopes, const void* gate, int64_t gate_stride, int gate_per_head, int shared_kv,
                          hipStream_t stream) {
  dim3 grid(num_tokens, nh);
  const size_t lds = (size_t)(hd + PAE_WAVE) * sizeof(float);
#define PAE_LAUNCH(MAXD)                                                                              \
  paged_attention_generic_kernel<T, MAXD><<<grid, PAE_WAVE, lds, stream>>>(                           \
      (T*)out, out_stride, (const T*)q, q_stride, (const T*)k_cache, (const T*)v_cache, positions,    \
      tok_seq, block_tables, max_blocks, bs, nh, nkv, hd, vd, scale, window, cap, sinks, chunked,   \
      slopes, (const T*)gate, gate_stride, gate_per_head, shared_kv)
  if (vd <= 64) PAE_LAUNCH(1);
  else if (vd <= 128) PAE_LAUNCH(2);
  else if (vd <= 192) PAE_LAUNCH(3);
  else if (vd <= 256) PAE_LAUNCH(4);
  else PAE_LAUNCH(8);
#undef PAE_LAUNCH
  return pae_check_launch("paged_attention_generic");
}

// Floats of scratch for the calls below (16-byte aligned), 0: none is used.  Without it a workgroup walks its chunks; the bits are the same.
extern "C" int64_t pae_paged_attention_scratch(int dtype, const void* k_cache, const void* v_cache, int max_blocks, int bs, int num_tokens,
                                               int nh, int nkv, int hd, int vd, int shared_kv) {
  if (dtype != PAE_F32 || num_tokens <= 0 || nh <= 0 || nkv <= 0 || nh % nkv || nkv > 65535 || bs <= 0 || vd <= 0 ||
      !rows_kernel_takes(k_cache, v_cache, bs, hd, vd, shared_kv))
    return 0;
  const int chunks = split_chunks(num_tokens, nh, nkv, vd, max_blocks, bs);
  return chunks > 1 ? (int64_t)num_tokens * nh * chunks * (vd + 2) : 0;
}

extern "C" int pae_paged_attention_masked(int dtype, void* out, int64_t out_stride, const void* q,
                                          int64_t q_stride, const void* k_cache, const void* v_cache,
                                          const int* positions, const int* tok_seq,
                                          const int* block_tables, int max_blocks, int bs,
                                          int num_tokens, int nh, int nkv, int hd, int vd, float scale,
                                          int window, float cap, const float* sinks, int chunked,
                                          const float* slopes, const void* gate, int64_t gate_stride, int gate_per_head,
                                          int shared_kv, float* scratch, hipStream_t stream) {
  PAE_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0, "attention: %d query heads over %d key/value heads", nh, nkv);
  PAE_REQUIRE(hd > 0 && hd <= 1024, "attention: head_dim %d is outside 1..1024", hd);
  PAE_REQUIRE(vd > 0 && vd <= 512, "attention: value width %d is outside 1..512", vd);
  PAE_REQUIRE(!shared_kv || (nkv == 1 && vd <= hd), "attention: values shared with the keys need one key head at least as wide");
  PAE_REQUIRE(!gate || gate_stride >= (gate_per_head ? nh : (int64_t)nh * vd), "attention: gate row stride %lld too small", (long long)gate_stride);
  PAE_REQUIRE(shared_kv || v_cache, "attention: no values");
  PAE_REQUIRE(bs > 0 && max_blocks > 0, "attention: bad cache geometry bs=%d max_blocks=%d", bs, max_blocks);
  PAE_REQUIRE(window >= 0, "attention: negative window %d", window);
  PAE_REQUIRE(cap >= 0.f, "attention: negative score cap %g", (double)cap);
  PAE_REQUIRE(nh <= 65535, "attention: %d query heads exceed the grid", nh);
  if (num_tokens <= 0) return 0;
  if (dtype == PAE_F32 && rows_kernel_takes(k_cache, v_cache, bs, hd, vd, shared_kv) && nkv <= 65535)
    return launch_rows((float*)out, out_stride, (const float*)q, q_stride, (const float*)k_cache, (const float*)v_cache, positions,
                       tok_seq, block_tables, max_blocks, bs, num_tokens, nh, nkv, hd, vd, scale, window, cap, sinks, chunked,
                       slopes, (const float*)gate, gate_stride, gate_per_head, scratch, stream);
  if (dtype == PAE_F32)
    return launch_generic<float>(out, out_stride, q, q_stride, k_cache, v_cache, positions, tok_seq, block_tables,
                                 max_blocks, bs, num_tokens, nh, nkv, hd, vd, scale, window, cap, sinks, chunked, slopes, gate,
                                 gate_stride, gate_per_head, shared_kv, stream);
  if (dtype == PAE_BF16)
    return launch_generic<bf16_t>(out, out_stride, q, q_stride, k_cache, v_cache, positions, tok_seq, block_tables,
                                  max_blocks, bs, num_tokens, nh, nkv, hd, vd, scale, window, cap, sinks, chunked, slopes, gate,
                                  gate_stride, gate_per_head, shared_kv, stream);
  return pae_fail("attention: unknown dtype code %d", dtype);
}

extern "C" int pae_paged_attention_capped(int dtype, void* out, int64_t out_stride, const void* q,
                                          int64_t q_stride, const void* k_cache, const void* v_cache,
                                          const int* positions, const int* tok_seq,
                                          const int* block_tables, int max_blocks, int bs,
                                          int num_tokens, int nh, int nkv, int hd, int vd, float scale,
                                          int window, float cap, const float* sinks, float* scratch, hipStream_t stream) {
  PAE_REQUIRE(vd > 0 && vd <= 256, "attention: value width %d is outside 1..256", vd);
  return pae_paged_attention_masked(dtype, out, out_stride, q, q_stride, k_cache, v_cache, positions, tok_seq,
                                    block_tables, max_blocks, bs, num_tokens, nh, nkv, hd, vd, scale, window, cap, sinks,
                                    0, nullptr, nullptr, 0, 0, 0, scratch, stream);
}

extern "C" int pae_paged_attention_generic(int dtype, void* out, int64_t out_stride, const void* q,
                                           int64_t q_stride, const void* k_cache, const void* v_cache,
                                           const int* positions, const int* tok_seq,
                                           const int* block_tables, int max_blocks, int bs,
                                           int num_tokens, int nh, int nkv, int hd, float scale,
                                           int window, float* scratch, hipStream_t stream) {
  PAE_REQUIRE(hd > 0 && hd <= 256, "attention: head_dim %d is outside 1..256", hd);
  return pae_paged_attention_capped(dtype, out, out_stride, q, q_stride, k_cache, v_cache, positions, tok_seq,
                                    block_tables, max_blocks, bs, num_tokens, nh, nkv, hd, hd, scale, window, 0.f,
                                    nullptr, scratch, stream);
}
