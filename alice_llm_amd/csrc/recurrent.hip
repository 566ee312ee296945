// Recurrent mixers whose state per head is a matrix S [d, dv] that is carried from token to token, and the short
// causal convolutions that stand before them.  Two recurrences share one kernel:
//
//   state space (plain):  S_t = diag(a_t) S_(t-1) + k_t (b_t v_t)^T,             o_t = S_t^T q_t + skip_h v_t
//   delta rule:           S' = diag(a_t) S_(t-1);  u = b_t (v_t - S'^T k_t);  S_t = S' + k_t u^T,  o_t = S_t^T q_t
//
// a_t is a decay per key channel (or one number a head, spread over the channels), b_t one number a head (the step
// size, or the write strength), q and k may be shared by groups of heads.  o is taken after the token's write.
//
// Everything here is 32-bit on both paths: the operands arrive as float32 rows of the projections and of the
// convolutions, the decays, step sizes and unit vectors are made with the full-precision functions, the state lives
// in float32 rows of the cache, one per slot, and the read-out is left in float32 for the norm that follows.
//
// recurrence_kernel: one wave per (sequence, head, CB value columns), four of them a block, walks through the sequence's tokens of the
// step with its part of the state in registers: lane (rg, col) holds RPT neighbouring rows of one column, reads
// them once and writes them once; a single token is the same walk of one step.  The tokens go through LDS TC at a
// time, the next TC tokens' operands already on their way from memory; sums over the rows of a column meet by lane
// exchanges inside a row of 16 lanes (the 64 / CB row groups of a column are neighbouring lanes), so the delta rule's
// sum a token needs no barrier and no trip through LDS; the read-outs' sums are taken once per TC tokens.  CB is 16 where that fills the chip's SIMDs, else 8 or 4 (more waves, fewer rows a lane).  Which rows belong to the sequence and which state row is
// its own are read on the device (cu_seqlens, slots), so a launch depends on sizes only.
//
// short_conv: y[t, c] = act(bias_c + sum_j w[c, j] x[t - (taps - 1) + j, c]) over the tokens of the token's own
// sequence; before the step's first token come the last taps - 1 inputs of the sequence's earlier steps, kept in
// a state row per slot (zeros at the start), which then takes the step's last inputs.  ssm_enter and delta_enter do
// the same and make, in the same launch, what else the recurrence takes from the projection's row.
#include "common.h"
#include "alice_hip.h"

namespace {

__device__ __forceinline__ float silu_full(float z) { return z / (1.f + expf(-z)); }
__device__ __forceinline__ float sigmoid_full(float z) { return 1.f / (1.f + expf(-z)); }
__device__ __forceinline__ float softplus_full(float z) { return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z))); }

// ------------------------------------------------------------------------------------------ short convolution

__global__ __launch_bounds__(256) void short_conv_kernel(const float* __restrict__ rows, int row_w, int col0, int C, int taps,
                                                         const float* __restrict__ w, const float* __restrict__ bias,
                                                         const float* __restrict__ state, float* __restrict__ out, int act,
                                                         const int* __restrict__ cu_seqlens, const int* __restrict__ seq_of_token,
                                                         const int* __restrict__ slots) {
  const int t = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int s = seq_of_token[t];
  const int i = t - cu_seqlens[s];                     // the token's place among its sequence's tokens of this step
  const int K = taps - 1;
  const float* st = state ? state + ((size_t)slots[s] * C + c) * K : nullptr;
  float acc = bias ? bias[c] : 0.f;
  for (int j = 0; j < taps; ++j) {
    const int back = K - j;                            // how many tokens before this one
    float x;
    if (back <= i) x = rows[(size_t)(t - back) * row_w + col0 + c];
    else x = st[K + i - back];                         // the input `back - i` places before the step's first token
    acc = fmaf(w[(size_t)c * taps + j], x, acc);
  }
  out[(size_t)t * C + c] = act ? silu_full(acc) : acc;
}

constexpr int MAX_TAPS = 16;

__global__ __launch_bounds__(256) void short_conv_state_kernel(const float* __restrict__ rows, int row_w, int col0, int C, int taps,
                                                               float* __restrict__ state, const int* __restrict__ cu_seqlens,
                                                               const int* __restrict__ slots) {
  const int s = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int t0 = cu_seqlens[s], n = cu_seqlens[s + 1] - t0, K = taps - 1;
  if (n <= 0) return;
  float* st = state + ((size_t)slots[s] * C + c) * K;
  float keep[MAX_TAPS];
#pragma unroll
  for (int m = 0; m < MAX_TAPS; ++m) {
    if (m < K) {
      const int off = n - K + m;                       // the step's token that lands at place m (negative: an older input)
      keep[m] = off >= 0 ? rows[(size_t)(t0 + off) * row_w + col0 + c] : st[n + m];
    }
  }
#pragma unroll
  for (int m = 0; m < MAX_TAPS; ++m)
    if (m < K) st[m] = keep[m];
}

// ------------------------------------------------------------------------------------------ what enters the recurrences

// A launch of the convolution with what else is made of the projection's rows.
struct Enter {
  const float* rows; int row_w, col0, C, taps;
  const float* w; const float* bias; float* state; float* out; int act;
  const int* cu; const int* seq; const int* slots; int T, n_seqs;
  // Unit heads (unit_d 0: none): the convolution's columns [0, unit_cols) are heads of unit_d that become unit vectors
  // x / sqrt(sum x^2 + unit_eps); those of the first q_cols columns also times q_scale.
  int unit_d, q_cols, unit_cols; float unit_eps, q_scale;
  // State space (step not null): step = softplus(rows[dt_col + h] + dt_bias[h]), decay = exp(-exp(a_log[h]) step), with
  // as_log its logarithm, which the chunk kernels take; both [T, H].
  int dt_col; const float* dt_bias; const float* a_log; float* step; float* decay; int H, as_log;
  // Delta rule (beta not null): beta[t, h] = sigmoid(rows[b_col + h]); the columns [low_col, low_col + n0) and the n1 behind
  // them to the matrices low0 [T, n0] and low1 [T, n1], in bfloat16 or as they are.
  int b_col; float* beta; int low_col, n0, n1; void* low0; void* low1; int low_bf16;
};

// The numbers of token t that are no convolution, dealt out to a block's threads.
__device__ void enter_small(const Enter& a, int t, int tid, int threads) {
  const float* r = a.rows + (size_t)t * a.row_w;
  if (a.step) {
    for (int h = tid; h < a.H; h += threads) {
      const float dt = softplus_full(r[a.dt_col + h] + a.dt_bias[h]);
      const float l = -expf(a.a_log[h]) * dt;
      a.step[(size_t)t * a.H + h] = dt;
      a.decay[(size_t)t * a.H + h] = a.as_log ? l : expf(l);
    }
  }
  if (a.beta) {
    for (int h = tid; h < a.H; h += threads) a.beta[(size_t)t * a.H + h] = sigmoid_full(r[a.b_col + h]);
    for (int e = tid; e < a.n0 + a.n1; e += threads) {
      const float x = r[a.low_col + e];
      void* m = e < a.n0 ? a.low0 : a.low1;
      const size_t i = e < a.n0 ? (size_t)t * a.n0 + e : (size_t)t * a.n1 + (e - a.n0);
      if (a.low_bf16) store_f32((bf16_t*)m, i, x); else store_f32((float*)m, i, x);
    }
  }
}
__global__ __launch_bounds__(128) void enter_small_kernel(Enter a) { enter_small(a, blockIdx.x, threadIdx.x, 128); }

// The unit heads in place, a wave a head: where the kernels below do not cover the head size.
__global__ __launch_bounds__(64) void enter_unit_kernel(Enter a) {
  const int t = blockIdx.x, c = blockIdx.y * a.unit_d;
  float* x = a.out + (size_t)t * a.C + c;
  float ss = 0.f;
  for (int e = threadIdx.x; e < a.unit_d; e += 64) ss = fmaf(x[e], x[e], ss);
  ss = wave_sum(ss);
  const float f = (c < a.q_cols ? a.q_scale : 1.f) / sqrtf(ss + a.unit_eps);
  for (int e = threadIdx.x; e < a.unit_d; e += 64) x[e] *= f;
}

// Four neighbouring channels of one token from the inputs x[0 .. TAPS - 1] (oldest first) to the output.  A head of
// unit_d channels is unit_d / 4 neighbouring lanes (a power of two, at most the wave).
template <int TAPS>
__device__ __forceinline__ void enter_token(const Enter& a, int t, int c, const float4 (&x)[TAPS], const float (&w)[4][TAPS],
                                            const float4 bias, bool unit) {
  float y[4] = {bias.x, bias.y, bias.z, bias.w};
#pragma unroll
  for (int j = 0; j < TAPS; ++j) {
    y[0] = fmaf(w[0][j], x[j].x, y[0]);
    y[1] = fmaf(w[1][j], x[j].y, y[1]);
    y[2] = fmaf(w[2][j], x[j].z, y[2]);
    y[3] = fmaf(w[3][j], x[j].w, y[3]);
  }
  if (a.act) {
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = silu_full(y[i]);
  }
  if (unit) {                                        // (the whole head or none of it)
    float ss = fmaf(y[0], y[0], y[1] * y[1]) + fmaf(y[2], y[2], y[3] * y[3]);
    for (int m = 1; m < (a.unit_d >> 2); m <<= 1) ss += __shfl_xor(ss, m);
    const float f = (c < a.q_cols ? a.q_scale : 1.f) / sqrtf(ss + a.unit_eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] *= f;
  }
  *reinterpret_cast<float4*>(a.out + (size_t)t * a.C + c) = make_float4(y[0], y[1], y[2], y[3]);
}

template <int TAPS>
__device__ __forceinline__ void enter_weights(const Enter& a, int c, float (&w)[4][TAPS], float4& bias) {
  float4 raw[TAPS];
#pragma unroll
  for (int i = 0; i < TAPS; ++i) raw[i] = reinterpret_cast<const float4*>(a.w + (size_t)c * TAPS)[i];
  const float* f = reinterpret_cast<const float*>(raw);
#pragma unroll
  for (int i = 0; i < 4 * TAPS; ++i) w[i / TAPS][i % TAPS] = f[i];
  bias = a.bias ? *reinterpret_cast<const float4*>(a.bias + c) : make_float4(0.f, 0.f, 0.f, 0.f);
}
// The state of four neighbouring channels: K inputs each, oldest first.
template <int K>
__device__ __forceinline__ void enter_state(const float* st, float4 (&x)[K]) {
  float4 raw[K];
#pragma unroll
  for (int i = 0; i < K; ++i) raw[i] = reinterpret_cast<const float4*>(st)[i];
  const float* f = reinterpret_cast<const float*>(raw);
#pragma unroll
  for (int m = 0; m < K; ++m) x[m] = make_float4(f[m], f[K + m], f[2 * K + m], f[3 * K + m]);
}

constexpr int ENTER_TT = 8, ENTER_THREADS = 128;

// By tokens: a thread takes four channels of ENTER_TT tokens, all inputs loaded before the first product (an input serves
// TAPS tokens and is read from memory once).  Memory-bound, with two full-precision exponential-and-divide a number
// beside it: 2,048 tokens of 6,144 channels 29 us (3.5 TB/s), channel by channel 64; with unit heads, step sizes and the
// small matrices 34 against 86 in launches of their own.
// grid: (tiles of tokens, blocks of 512 channels + one a token for the small numbers).
template <int TAPS>
__global__ __launch_bounds__(ENTER_THREADS) void enter_tokens_kernel(Enter a) {
  constexpr int K = TAPS - 1, TT = ENTER_TT;
  const int t0 = blockIdx.x * TT, n = min(TT, a.T - t0);
  const int c = (blockIdx.y * ENTER_THREADS + threadIdx.x) * 4;
  if (blockIdx.y * ENTER_THREADS * 4 >= (unsigned)a.C) {
    const int j = (int)blockIdx.y - (a.C + ENTER_THREADS * 4 - 1) / (ENTER_THREADS * 4);
    if (j < n) enter_small(a, t0 + j, threadIdx.x, ENTER_THREADS);
    return;
  }
  if (c >= a.C) return;
  float w[4][TAPS];
  float4 bias, x[K + TT];
  const float* col = a.rows + a.col0 + c;
#pragma unroll
  for (int m = 0; m < K + TT; ++m)
    x[m] = *reinterpret_cast<const float4*>(col + (size_t)min(max(t0 + m - K, 0), a.T - 1) * a.row_w);
  enter_weights<TAPS>(a, c, w, bias);
  const bool unit = c < a.unit_cols;
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    if (j >= n) break;
    const int t = t0 + j, s = a.seq[t], i = t - a.cu[s];     // the token's place among its sequence's tokens of this step
    float4 v[TAPS];
#pragma unroll
    for (int m = 0; m < TAPS; ++m) v[m] = x[j + m];
    if (i < K) {                                             // the sequence's first tokens: earlier inputs from its state
      float4 st[K];
      enter_state<K>(a.state + ((size_t)a.slots[s] * a.C + c) * K, st);
#pragma unroll
      for (int m = 0; m < K; ++m)                            // place m of the window is the input K - m before this token
#pragma unroll
        for (int o = 0; o < K; ++o)
          if (K - m > i && o == m + i) v[m] = st[o];
    }
    enter_token<TAPS>(a, t, c, v, w, bias, unit);
  }
}

// By sequences: a thread takes four channels of a sequence's tokens one after the other, its window and so the state in
// registers; the state's next inputs need no launch of their own.  Latency-bound: 8 single tokens 2.7 us where the launches of
// their own take 8.2; about a microsecond more for every further token of a sequence.
// grid: (sequences, blocks of 512 channels + one for the small numbers).
template <int TAPS>
__global__ __launch_bounds__(ENTER_THREADS) void enter_sequences_kernel(Enter a) {
  constexpr int K = TAPS - 1;
  const int s = blockIdx.x, c = (blockIdx.y * ENTER_THREADS + threadIdx.x) * 4;
  if (blockIdx.y * ENTER_THREADS * 4 >= (unsigned)a.C) {
    for (int t = s; t < a.T; t += a.n_seqs) enter_small(a, t, threadIdx.x, ENTER_THREADS);
    return;
  }
  if (c >= a.C) return;
  const int t0 = a.cu[s], n = a.cu[s + 1] - t0;
  if (n <= 0) return;
  float w[4][TAPS];
  float4 bias, x[TAPS], old[K];
  float* st = a.state + ((size_t)a.slots[s] * a.C + c) * K;
  const float* col = a.rows + (size_t)t0 * a.row_w + a.col0 + c;
  float4 next = *reinterpret_cast<const float4*>(col);
  enter_state<K>(st, old);
  enter_weights<TAPS>(a, c, w, bias);
#pragma unroll
  for (int m = 0; m < K; ++m) x[m] = old[m];
  const bool unit = c < a.unit_cols;
  for (int i = 0; i < n; ++i) {
    x[K] = next;
    next = *reinterpret_cast<const float4*>(col + (size_t)min(i + 1, n - 1) * a.row_w);
    enter_token<TAPS>(a, t0 + i, c, x, w, bias, unit);
#pragma unroll
    for (int m = 0; m < K; ++m) x[m] = x[m + 1];
  }
  float f[4 * K];
#pragma unroll
  for (int m = 0; m < K; ++m) {
    f[m] = x[m].x;
    f[K + m] = x[m].y;
    f[2 * K + m] = x[m].z;
    f[3 * K + m] = x[m].w;
  }
#pragma unroll
  for (int i = 0; i < K; ++i) reinterpret_cast<float4*>(st)[i] = make_float4(f[4 * i], f[4 * i + 1], f[4 * i + 2], f[4 * i + 3]);
}

// Delta rule: z [T, H d] into the decays exp(-exp(a_log[h]) softplus(z + dt_bias)), with as_log their logarithms, in place;
// V neighbouring numbers of one head a thread.
template <int V>
__global__ __launch_bounds__(256) void delta_decay_kernel(float* __restrict__ z, const float* __restrict__ dt_bias,
                                                          const float* __restrict__ a_log, long n, int H, int d, int as_log) {
  const long i = ((long)blockIdx.x * 256 + threadIdx.x) * V;
  if (i >= n) return;
  const int col = (int)(i % ((long)H * d));
  const float rate = expf(a_log[col / d]);
  float x[V];
  if constexpr (V == 4) *reinterpret_cast<float4*>(x) = *reinterpret_cast<const float4*>(z + i);
  else x[0] = z[i];
#pragma unroll
  for (int e = 0; e < V; ++e) {
    const float l = -rate * softplus_full(x[e] + dt_bias[col + e]);
    x[e] = as_log ? l : expf(l);
  }
  if constexpr (V == 4) *reinterpret_cast<float4*>(z + i) = *reinterpret_cast<const float4*>(x);
  else z[i] = x[0];
}

// ------------------------------------------------------------------------------------------ the recurrence

struct RecurrenceArgs {
  const float* q; int q_w, q_col;          // q[t, q_col + (h / per) * d + r]
  const float* k; int k_w, k_col;          // k likewise (q and k share the grouping)
  const float* v; int v_w, v_col;          // v[t, v_col + h * dv + c]
  const float* decay; int decay_per_row;   // [T, H d] or [T, H]
  const float* b;                          // [T, H]
  const float* skip;                       // [H] or null
  float* out;                              // [T, H dv]
  const int* cu_seqlens; const int* slots;
  float* S;                                // [slots, H, d, dv]
  int H, per, d, dv;
};

// x plus the x of the lane that a DPP control names (lanes a fixed distance apart inside a row of 16)
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
// The sum over the RG neighbouring lanes that hold one column's row groups (RG 4, 8 or 16, aligned): every one of them
// gets it.  Lanes 1 and 2 apart inside a quad, then the other quad of the half row, then the other half of the row.
template <int RG>
__device__ __forceinline__ float sum_row_groups(float x) {
  x = dpp_add<0xB1>(x);                    // quad_perm [1, 0, 3, 2]
  x = dpp_add<0x4E>(x);                    // quad_perm [2, 3, 0, 1]
  if (RG >= 8) x = dpp_add<0x141>(x);      // row_half_mirror
  if (RG >= 16) x = dpp_add<0x140>(x);     // row_mirror
  return x;
}

template <int CB, int RPT, int TC, int WPB, bool DELTA>
__global__ __launch_bounds__(64 * WPB) void recurrence_kernel(RecurrenceArgs a) {
  constexpr int RG = 64 / CB, DP = RG * RPT, NT = 64 * WPB, CBB = CB * WPB;
  constexpr int NL = TC * DP / NT;
  constexpr int NV = (TC * CBB + NT - 1) / NT;
  static_assert(RPT % 4 == 0 && (TC * DP) % NT == 0 && TC <= 64 && (RG == 4 || RG == 8 || RG == 16), "rows are read four at a time");
  __shared__ __align__(16) float sq[TC][DP];
  __shared__ __align__(16) float sk[TC][DP];
  __shared__ __align__(16) float sa[TC][DP];
  __shared__ float sv[TC][CBB];
  __shared__ float sb[TC];
  // the row groups of a column are neighbouring lanes, so that their sums meet without a trip through LDS; the waves of
  // a block take neighbouring columns and share the tokens' q, k and decays
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int col = wave * CB + lane / RG, rg = lane % RG;
  const int j = blockIdx.z * CBB + col;
  const bool col_ok = j < a.dv;
  const int t0 = a.cu_seqlens[s], t1 = a.cu_seqlens[s + 1];
  if (t1 <= t0) return;
  const int H = a.H, d = a.d, dv = a.dv;
  float* Sh = a.S + ((size_t)a.slots[s] * H + h) * d * dv;
  float st[RPT];
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = rg * RPT + i;
    st[i] = (r < d && col_ok) ? Sh[(size_t)r * dv + j] : 0.f;
  }
  const int qk_head = h / a.per;
  const float skip = a.skip ? a.skip[h] : 0.f;
  // what this thread fetches for TC tokens: element (t, r) = (idx / DP, idx % DP) of q, k and the decay; (t, c) of v; b of token `tid`
  float pq[NL], pk[NL], pa[NL], pv[NV], pb = 0.f;
  auto fetch = [&](int tc) {
#pragma unroll
    for (int n = 0; n < NL; ++n) {
      const int idx = tid + n * NT, t = tc + idx / DP, r = idx % DP;
      pq[n] = pk[n] = pa[n] = 0.f;
      if (t < t1 && r < d) {
        pq[n] = a.q[(size_t)t * a.q_w + a.q_col + qk_head * d + r];
        pk[n] = a.k[(size_t)t * a.k_w + a.k_col + qk_head * d + r];
        pa[n] = a.decay_per_row ? a.decay[((size_t)t * H + h) * d + r] : a.decay[(size_t)t * H + h];
      }
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int idx = tid + n * NT, t = tc + idx / CBB, c = blockIdx.z * CBB + idx % CBB;
      pv[n] = (idx < TC * CBB && t < t1 && c < dv) ? a.v[(size_t)t * a.v_w + a.v_col + h * dv + c] : 0.f;
    }
    pb = (tid < TC && tc + tid < t1) ? a.b[(size_t)(tc + tid) * H + h] : 0.f;
  };
  fetch(t0);
  for (int tc = t0; tc < t1; tc += TC) {
    const int n_tok = min(TC, t1 - tc);
    __syncthreads();                                   // the last tokens' operands have been read
#pragma unroll
    for (int n = 0; n < NL; ++n) {
      const int idx = tid + n * NT;
      sq[idx / DP][idx % DP] = pq[n];
      sk[idx / DP][idx % DP] = pk[n];
      sa[idx / DP][idx % DP] = pa[n];                  // (rows beyond d hold zeros and stay zero)
    }
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      const int idx = tid + n * NT;
      if (idx < TC * CBB) sv[idx / CBB][idx % CBB] = pv[n];
    }
    if (tid < TC) sb[tid] = pb;
    __syncthreads();
    if (tc + TC < t1) fetch(tc + TC);                  // the next tokens' operands are on their way during the walk
    float part[TC], vs[TC];                            // the lanes' shares of the read-outs meet once per TC tokens
#pragma unroll
    for (int tt = 0; tt < TC; ++tt) {
      part[tt] = 0.f;
      vs[tt] = 0.f;
      if (tt < n_tok) {
        const float vj = sv[tt][col], bt = sb[tt];
        vs[tt] = vj;
        float u = bt * vj;
        float4 kk[RPT / 4];
#pragma unroll
        for (int i = 0; i < RPT; i += 4) kk[i / 4] = *reinterpret_cast<const float4*>(&sk[tt][rg * RPT + i]);
        if (DELTA) {
          float p0 = 0.f, p1 = 0.f, p2 = 0.f, p3 = 0.f;   // four sums side by side: no chain of dependent additions
#pragma unroll
          for (int i = 0; i < RPT; i += 4) {
            const float4 aa = *reinterpret_cast<const float4*>(&sa[tt][rg * RPT + i]);
            st[i] *= aa.x;      p0 = fmaf(st[i], kk[i / 4].x, p0);
            st[i + 1] *= aa.y;  p1 = fmaf(st[i + 1], kk[i / 4].y, p1);
            st[i + 2] *= aa.z;  p2 = fmaf(st[i + 2], kk[i / 4].z, p2);
            st[i + 3] *= aa.w;  p3 = fmaf(st[i + 3], kk[i / 4].w, p3);
          }
          u = bt * (vj - sum_row_groups<RG>((p0 + p1) + (p2 + p3)));
        }
        float o0 = 0.f, o1 = 0.f, o2 = 0.f, o3 = 0.f;
#pragma unroll
        for (int i = 0; i < RPT; i += 4) {
          const float4 qq = *reinterpret_cast<const float4*>(&sq[tt][rg * RPT + i]);
          if (DELTA) {
            st[i] = fmaf(kk[i / 4].x, u, st[i]);
            st[i + 1] = fmaf(kk[i / 4].y, u, st[i + 1]);
            st[i + 2] = fmaf(kk[i / 4].z, u, st[i + 2]);
            st[i + 3] = fmaf(kk[i / 4].w, u, st[i + 3]);
          } else {
            const float4 aa = *reinterpret_cast<const float4*>(&sa[tt][rg * RPT + i]);
            st[i] = fmaf(aa.x, st[i], kk[i / 4].x * u);
            st[i + 1] = fmaf(aa.y, st[i + 1], kk[i / 4].y * u);
            st[i + 2] = fmaf(aa.z, st[i + 2], kk[i / 4].z * u);
            st[i + 3] = fmaf(aa.w, st[i + 3], kk[i / 4].w * u);
          }
          o0 = fmaf(st[i], qq.x, o0);
          o1 = fmaf(st[i + 1], qq.y, o1);
          o2 = fmaf(st[i + 2], qq.z, o2);
          o3 = fmaf(st[i + 3], qq.w, o3);
        }
        part[tt] = (o0 + o1) + (o2 + o3);
      }
    }
#pragma unroll
    for (int tt = 0; tt < TC; ++tt) {
      const float o = sum_row_groups<RG>(part[tt]);
      if (tt < n_tok && rg == 0 && col_ok) a.out[(size_t)(tc + tt) * H * dv + h * dv + j] = fmaf(skip, vs[tt], o);
    }
  }
#pragma unroll
  for (int i = 0; i < RPT; ++i) {
    const int r = rg * RPT + i;
    if (r < d && col_ok) Sh[(size_t)r * dv + j] = st[i];
  }
}

// ------------------------------------------------------------------------------------------ norm and gate behind a read-out

// A block per (token, part): the row's part of n elements is RMS-normed (eps inside the root) and multiplied by a
// weight (of the part's length, shared by the parts, or of the row's length).  gate_act 1: silu of the gate row,
// applied before the norm; 2: sigmoid of the gate row, applied after it; 0: no gate.
template <typename TO, typename TG>
__global__ __launch_bounds__(1024) void norm_gate_kernel(const float* __restrict__ x, int width, int parts, const TG* __restrict__ gate,
                                                        int gate_w, int gate_col, int gate_act, const float* __restrict__ w,
                                                        int w_shared, float eps, TO* __restrict__ out) {
  __shared__ float red[16];
  const int t = blockIdx.x, g = blockIdx.y, n = width / parts;
  const float* xr = x + (size_t)t * width + (size_t)g * n;
  const TG* gr = gate ? gate + (size_t)t * gate_w + gate_col + (size_t)g * n : nullptr;
  float ss = 0.f;
  for (int e = threadIdx.x; e < n; e += blockDim.x) {
    float y = xr[e];
    if (gate_act == 1) y *= silu_full(load_f32(gr, e));
    ss = fmaf(y, y, ss);
  }
  ss = block_sum(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)n + eps);
  for (int e = threadIdx.x; e < n; e += blockDim.x) {
    float y = xr[e];
    if (gate_act == 1) y *= silu_full(load_f32(gr, e));
    y = y * inv * w[w_shared ? e : g * n + e];
    if (gate_act == 2) y *= sigmoid_full(load_f32(gr, e));
    store_f32(out + (size_t)t * width + (size_t)g * n, e, y);
  }
}

// The same with the part in registers: LANES lanes a part (a part of a row of at most 16 LANES wide elements, V units of
// four a lane), so that x and the gate are read once and the gate's exponential is taken once.
template <typename T>
__device__ __forceinline__ void load4(const T* p, float (&v)[4]) {
  if constexpr (std::is_same_v<T, float>) {
    const float4 r = *reinterpret_cast<const float4*>(p);
    v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w;
  } else {
    const uint2 r = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(r.x << 16); v[1] = __uint_as_float(r.x & 0xffff0000u);
    v[2] = __uint_as_float(r.y << 16); v[3] = __uint_as_float(r.y & 0xffff0000u);
  }
}
template <typename TO, typename TG, int LANES, int V>
__global__ __launch_bounds__(LANES > 256 ? LANES : 256) void norm_gate_regs_kernel(const float* __restrict__ x, int width, int parts, long rows,
                                                                                  const TG* __restrict__ gate, int gate_w, int gate_col,
                                                                                  int gate_act, const float* __restrict__ w, int w_shared,
                                                                                  float eps, TO* __restrict__ out) {
  constexpr int THREADS = LANES > 256 ? LANES : 256, PPB = THREADS / LANES;
  __shared__ float red[16];
  const int lane = threadIdx.x % LANES, n = width / parts;
  const long p = (long)blockIdx.x * PPB + threadIdx.x / LANES;       // (token, part); beyond the last: computed on it, not stored
  const bool in = p < rows;
  const long pc = in ? p : rows - 1;
  const long t = pc / parts;
  const int g = (int)(pc % parts);
  const float* xr = x + t * width + (long)g * n;
  const TG* gr = gate + t * gate_w + gate_col + (long)g * n;
  float y[V][4], s[V][4];
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int e = min((v * LANES + lane) * 4, n - 4);
    load4(xr + e, y[v]);
    if (gate_act) load4(gr + e, s[v]);
  }
  float ss = 0.f;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    if ((v * LANES + lane) * 4 >= n) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (gate_act == 1) y[v][i] *= silu_full(s[v][i]);
      ss = fmaf(y[v][i], y[v][i], ss);
    }
  }
  if constexpr (LANES <= 64) {
#pragma unroll
    for (int m = 1; m < LANES; m <<= 1) ss += __shfl_xor(ss, m);
  } else {
    ss = block_sum(ss, red);
  }
  const float inv = 1.f / sqrtf(ss / (float)n + eps);
  TO* o = out + t * width + (long)g * n;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    const int e = (v * LANES + lane) * 4;
    if (e >= n || !in) continue;
    float ww[4];
    load4(w + (w_shared ? e : g * n + e), ww);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      y[v][i] = y[v][i] * inv * ww[i];
      if (gate_act == 2) y[v][i] *= sigmoid_full(s[v][i]);
    }
    if constexpr (std::is_same_v<TO, float>) {
      *reinterpret_cast<float4*>(o + e) = make_float4(y[v][0], y[v][1], y[v][2], y[v][3]);
    } else {
      union { bf16_t h[4]; uint2 u; } r;
#pragma unroll
      for (int i = 0; i < 4; ++i) r.h[i] = f32_to_bf16(y[v][i]);
      *reinterpret_cast<uint2*>(o + e) = r.u;
    }
  }
}

}  // namespace

namespace {

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// form 1 and 2: by tokens (the state behind it) or by sequences, where the channels come in whole units of four with two
// to four taps, else as form 3: channel by channel, which takes everything.
int launch_enter(const Enter& a, int form, hipStream_t stream) {
  ALICE_CHECK(a.rows && a.w && a.out && a.cu && a.seq && a.slots, "short_conv: a pointer is missing");
  ALICE_CHECK(a.T >= 0 && a.n_seqs >= 0 && a.C >= 1 && a.taps >= 1 && a.taps <= MAX_TAPS, "short_conv: bad sizes (taps 1..%d)", MAX_TAPS);
  ALICE_CHECK(a.col0 >= 0 && a.col0 + a.C <= a.row_w, "short_conv: rows of %d elements are too short for the channels", a.row_w);
  ALICE_CHECK(a.taps == 1 || a.state != nullptr, "short_conv: more than one tap needs the state rows");
  ALICE_CHECK(ceil_div(a.C, 256) <= 65534, "short_conv: too many channels for one launch");
  ALICE_CHECK(form >= 1 && form <= 3, "short_conv: unknown form %d", form);
  if (a.T == 0 || a.n_seqs == 0) return 0;
  const bool whole_heads = a.unit_d == 0 || (a.unit_d >= 4 && a.unit_d <= 256 && (a.unit_d & (a.unit_d - 1)) == 0);
  const bool units = a.taps >= 2 && a.taps <= 4 && a.C % 4 == 0 && a.row_w % 4 == 0 && a.col0 % 4 == 0 && whole_heads && aligned16(a.rows) &&
                     aligned16(a.w) && aligned16(a.bias) && aligned16(a.state) && aligned16(a.out);
  const bool small = a.step || a.beta;
  if (units && form != 3) {
    const bool by_sequences = form == 2;
    const dim3 grid(by_sequences ? a.n_seqs : ceil_div(a.T, ENTER_TT), ceil_div(a.C, 4 * ENTER_THREADS) + (!small ? 0 : by_sequences ? 1 : ENTER_TT));
#define GO(TAPS)                                                                          \
  do {                                                                                    \
    if (by_sequences) enter_sequences_kernel<TAPS><<<grid, ENTER_THREADS, 0, stream>>>(a); \
    else enter_tokens_kernel<TAPS><<<grid, ENTER_THREADS, 0, stream>>>(a);                 \
  } while (0)
    if (a.taps == 4) GO(4); else if (a.taps == 3) GO(3); else GO(2);
#undef GO
    ALICE_LAUNCH_CHECK();
    if (by_sequences) return 0;
  } else {
    dim3 grid(a.T, ceil_div(a.C, 256));
    short_conv_kernel<<<grid, 256, 0, stream>>>(a.rows, a.row_w, a.col0, a.C, a.taps, a.w, a.bias, a.taps > 1 ? a.state : nullptr, a.out,
                                                a.act, a.cu, a.seq, a.slots);
    ALICE_LAUNCH_CHECK();
    if (a.unit_d) {
      ALICE_CHECK(a.unit_cols / a.unit_d <= 65535, "delta_enter: too many heads for one launch");
      enter_unit_kernel<<<dim3(a.T, a.unit_cols / a.unit_d), 64, 0, stream>>>(a);
      ALICE_LAUNCH_CHECK();
    }
    if (small) {
      enter_small_kernel<<<a.T, 128, 0, stream>>>(a);
      ALICE_LAUNCH_CHECK();
    }
  }
  if (a.taps > 1) {
    dim3 g2(a.n_seqs, ceil_div(a.C, 256));
    short_conv_state_kernel<<<g2, 256, 0, stream>>>(a.rows, a.row_w, a.col0, a.C, a.taps, a.state, a.cu, a.slots);
    ALICE_LAUNCH_CHECK();
  }
  return 0;
}

Enter enter_of(const float* rows, int row_w, int col0, int channels, int taps, const float* w, const float* bias, float* state, float* out,
               int act, const int* cu, const int* seq, const int* slots, int T, int n_seqs) {
  Enter a{};
  a.rows = rows; a.row_w = row_w; a.col0 = col0; a.C = channels; a.taps = taps; a.w = w; a.bias = bias; a.state = state; a.out = out;
  a.act = act; a.cu = cu; a.seq = seq; a.slots = slots; a.T = T; a.n_seqs = n_seqs;
  return a;
}

}  // namespace

extern "C" int alice_short_conv(const float* rows, int row_w, int col0, int channels, int taps, const float* w, const float* bias,
                                float* state, float* out, int act, const int* cu_seqlens, const int* seq_of_token,
                                const int* slots, int T, int n_seqs, int form, hipStream_t stream) {
  return launch_enter(enter_of(rows, row_w, col0, channels, taps, w, bias, state, out, act, cu_seqlens, seq_of_token, slots, T, n_seqs), form, stream);
}

extern "C" int alice_ssm_enter(const float* rows, int row_w, int col0, int channels, int taps, const float* w, const float* bias,
                               float* state, float* out, int dt_col, const float* dt_bias, const float* a_log, float* step,
                               float* decay, int H, int as_log, const int* cu_seqlens, const int* seq_of_token, const int* slots,
                               int T, int n_seqs, int form, hipStream_t stream) {
  ALICE_CHECK(dt_bias && a_log && step && decay, "ssm_enter: a pointer is missing");
  ALICE_CHECK(H >= 1 && dt_col >= 0 && dt_col + H <= row_w, "ssm_enter: bad sizes");
  Enter a = enter_of(rows, row_w, col0, channels, taps, w, bias, state, out, 1, cu_seqlens, seq_of_token, slots, T, n_seqs);
  a.dt_col = dt_col; a.dt_bias = dt_bias; a.a_log = a_log; a.step = step; a.decay = decay; a.H = H; a.as_log = as_log;
  return launch_enter(a, form, stream);
}

extern "C" int alice_delta_enter(const float* rows, int row_w, int channels, int taps, const float* w, float* state, float* out, int G,
                                 int d, float unit_eps, float q_scale, int b_col, int H, float* beta, int low_col, int n0, int n1,
                                 void* low0, void* low1, int low_dtype, const int* cu_seqlens, const int* seq_of_token,
                                 const int* slots, int T, int n_seqs, int form, hipStream_t stream) {
  ALICE_CHECK(beta && low0 && low1 && dtype_ok(low_dtype), "delta_enter: a pointer is missing or the dtype is unknown");
  ALICE_CHECK(H >= 1 && G >= 1 && d >= 1 && unit_eps >= 0.f && n0 >= 1 && n1 >= 1, "delta_enter: bad sizes");
  ALICE_CHECK(2L * G * d <= channels && b_col >= 0 && b_col + H <= row_w && low_col >= 0 && (long)low_col + n0 + n1 <= row_w,
              "delta_enter: the rows are too short for the heads");
  Enter a = enter_of(rows, row_w, 0, channels, taps, w, nullptr, state, out, 1, cu_seqlens, seq_of_token, slots, T, n_seqs);
  a.unit_d = d; a.q_cols = G * d; a.unit_cols = 2 * G * d; a.unit_eps = unit_eps; a.q_scale = q_scale;
  a.b_col = b_col; a.H = H; a.beta = beta; a.low_col = low_col; a.n0 = n0; a.n1 = n1; a.low0 = low0; a.low1 = low1;
  a.low_bf16 = low_dtype == DT_BF16;
  return launch_enter(a, form, stream);
}

extern "C" int alice_delta_decay(float* z, const float* dt_bias, const float* a_log, int T, int H, int d, int as_log, hipStream_t stream) {
  ALICE_CHECK(z && dt_bias && a_log, "delta_decay: a pointer is missing");
  ALICE_CHECK(T >= 0 && H >= 1 && d >= 1, "delta_decay: bad sizes");
  const long n = (long)T * H * d;
  if (n == 0) return 0;
  if (d % 4 == 0 && aligned16(z)) delta_decay_kernel<4><<<ceil_div(n / 4, 256), 256, 0, stream>>>(z, dt_bias, a_log, n, H, d, as_log);
  else delta_decay_kernel<1><<<ceil_div(n, 256), 256, 0, stream>>>(z, dt_bias, a_log, n, H, d, as_log);
  ALICE_LAUNCH_CHECK();
  return 0;
}

// Value columns a wave: 16 where (sequences x heads x columns) fill the chip's SIMDs, else 8 or 4: more waves, each with
// fewer rows a lane (the rows of a column are then spread over 8 or 16 lanes).
extern "C" int alice_matrix_recurrence_columns(int n_seqs, int H, int d, int dv) {
  const long waves16 = (long)n_seqs * H * ceil_div(dv, 16);
  return (waves16 >= 1024 || d <= 32) ? 16 : ((waves16 >= 512 || d <= 64) ? 8 : 4);
}

extern "C" int alice_matrix_recurrence(const float* q, int q_w, int q_col, const float* k, int k_w, int k_col, const float* v, int v_w,
                                       int v_col, const float* decay, int decay_per_row, const float* b, const float* skip, float* out,
                                       const int* cu_seqlens, const int* slots, float* S, int n_seqs, int n_slots, int H, int qk_heads,
                                       int d, int dv, int delta, int columns, hipStream_t stream) {
  ALICE_CHECK(q && k && v && decay && b && out && cu_seqlens && slots && S, "matrix_recurrence: a pointer is missing");
  ALICE_CHECK(n_seqs >= 0 && n_slots >= 1 && H >= 1 && qk_heads >= 1 && H % qk_heads == 0 && d >= 1 && dv >= 1, "matrix_recurrence: bad sizes");
  ALICE_CHECK(d <= 256, "matrix_recurrence: key size %d is beyond 256, the range of this kernel", d);
  ALICE_CHECK(q_col >= 0 && k_col >= 0 && v_col >= 0 && q_col + qk_heads * d <= q_w && k_col + qk_heads * d <= k_w && v_col + H * dv <= v_w,
              "matrix_recurrence: the rows are too short for the heads");
  ALICE_CHECK(H <= 65535 && ceil_div(dv, 16) <= 65535, "matrix_recurrence: too many heads or value columns for one launch");
  if (n_seqs == 0) return 0;
  RecurrenceArgs a{q, q_w, q_col, k, k_w, k_col, v, v_w, v_col, decay, decay_per_row, b, skip, out, cu_seqlens, slots, S, H, H / qk_heads, d, dv};
  int cb = columns ? columns : alice_matrix_recurrence_columns(n_seqs, H, d, dv);
  ALICE_CHECK(cb == 16 || cb == 8 || cb == 4, "matrix_recurrence: %d value columns a wave are not built (4, 8, 16; 0: by the step's size)", columns);
  if (d <= 32 || (cb == 4 && d <= 64)) cb = d <= 32 ? 16 : 8;      // (fewer than four rows a lane are not built)
  constexpr int WPB = 4;                       // waves a block: they share the staged q, k and decays of a head's tokens
  dim3 grid(n_seqs, H, ceil_div(dv, cb * WPB));
#define GO(CB, RPT, TC)                                                                     \
  do {                                                                                      \
    if (delta) recurrence_kernel<CB, RPT, TC, WPB, true><<<grid, 64 * WPB, 0, stream>>>(a); \
    else recurrence_kernel<CB, RPT, TC, WPB, false><<<grid, 64 * WPB, 0, stream>>>(a);      \
  } while (0)
  if (cb == 16) {
    if (d <= 16) GO(16, 4, 16);
    else if (d <= 32) GO(16, 8, 16);
    else if (d <= 64) GO(16, 16, 16);
    else if (d <= 128) GO(16, 32, 8);
    else GO(16, 64, 8);
  } else if (cb == 8) {
    if (d <= 64) GO(8, 8, 16);
    else if (d <= 128) GO(8, 16, 8);
    else GO(8, 32, 8);
  } else {
    if (d <= 128) GO(4, 8, 8);
    else GO(4, 16, 8);
  }
#undef GO
  ALICE_LAUNCH_CHECK();
  return 0;
}

extern "C" int alice_norm_gate(const float* x, int width, int parts, const void* gate, int gate_dtype, int gate_w, int gate_col, int gate_act,
                               const float* w, int w_shared, float eps, void* out, int out_dtype, int T, hipStream_t stream) {
  ALICE_CHECK(x && w && out && dtype_ok(out_dtype) && dtype_ok(gate_dtype), "norm_gate: a pointer is missing or the dtype is unknown");
  ALICE_CHECK(T >= 0 && width >= 1 && parts >= 1 && width % parts == 0 && parts <= 65535, "norm_gate: %d parts must divide the width %d", parts, width);
  ALICE_CHECK(gate_act >= 0 && gate_act <= 2 && (gate_act == 0 || (gate && gate_col >= 0 && gate_col + width <= gate_w)),
              "norm_gate: the gate rows are missing or too short");
  ALICE_CHECK(eps > 0.f, "norm_gate: eps must be positive");
  if (T == 0) return 0;
  const int n = width / parts;
  // Whole units of four, in registers: 32, 64 or 256 lanes a part by its length, 1,024 where the rows are few.  2,048 rows
  // of 16 parts of 128: 9.3 us (4.5 TB/s), element by element 18.7; of one part of 4,096: 16.2 us (5.2 TB/s) and 28.
  const bool units = n % 4 == 0 && n <= 4096 && aligned16(x) && aligned16(w) && aligned16(out) &&
                     (gate_act == 0 || (aligned16(gate) && gate_w % 4 == 0 && gate_col % 4 == 0));
  const long rows = (long)T * parts;
#define GO3(TO, TG, LANES, V) norm_gate_regs_kernel<TO, TG, LANES, V><<<ceil_div(rows, LANES > 256 ? 1 : 256 / LANES), LANES > 256 ? LANES : 256, 0, stream>>>( \
    x, width, parts, rows, (const TG*)gate, gate_w, gate_col, gate_act, w, w_shared, eps, (TO*)out)
#define GO2(TO, TG)                              \
  do {                                           \
    if (n <= 128) GO3(TO, TG, 32, 1);            \
    else if (n <= 512) GO3(TO, TG, 64, 2);       \
    else if (n > 1024 && rows <= 256) GO3(TO, TG, 1024, 1); \
    else if (n <= 1024) GO3(TO, TG, 256, 1);     \
    else GO3(TO, TG, 256, 4);                    \
  } while (0)
  if (units) {
    if (gate_dtype == DT_F32) { if (out_dtype == DT_F32) GO2(float, float); else GO2(bf16_t, float); }
    else { if (out_dtype == DT_F32) GO2(float, bf16_t); else GO2(bf16_t, bf16_t); }
    ALICE_LAUNCH_CHECK();
    return 0;
  }
#undef GO2
#undef GO3
  dim3 grid(T, parts);
  const int threads = n > 1024 && (long)T * parts <= 256 ? 1024 : (n > 128 ? 256 : 64);      // few rows: more lanes a row
#define GO(TO, TG) norm_gate_kernel<TO, TG><<<grid, threads, 0, stream>>>(x, width, parts, (const TG*)gate, gate_w, gate_col, gate_act, w, w_shared, eps, (TO*)out)
  if (gate_dtype == DT_F32) { if (out_dtype == DT_F32) GO(float, float); else GO(bf16_t, float); }
  else { if (out_dtype == DT_F32) GO(float, bf16_t); else GO(bf16_t, bf16_t); }
#undef GO
  ALICE_LAUNCH_CHECK();
  return 0;
}
