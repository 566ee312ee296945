// The matrix recurrences of recurrent.hip (state space, delta rule) over pieces of many tokens, 16 tokens at a time on
// the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32).  With S the state [d, dv] ahead of a chunk, A_t the product of
// the decays of the chunk's tokens up to t (a number a key channel, or one a head), n the chunk's last token:
//
//   state space:  o_t = A_t (S^T q_t) + sum_(r <= t) (A_t / A_r) b_r (q_t . k_r) v_r + skip v_t
//                 S'  = A_n S + sum_r (A_n / A_r) b_r k_r v_r^T
//   delta rule:   u   = (I + diag(b) M)^(-1) diag(b) (V - K~ S),   M_tr = sum_c k_t[c] k_r[c] A_t[c] / A_r[c]  (r < t)
//                 o_t = S^T (A_t q_t) + sum_(r <= t) P_tr u_r,     P_tr = sum_c q_t[c] k_r[c] A_t[c] / A_r[c]
//                 S'  = diag(A_n) S + sum_r (A_n / A_r k_r) u_r^T,  K~_t = A_t k_t
//
// Everything that does not depend on the state is made for all chunks side by side first (ssm_chunk_kernel,
// delta_chunk_kernel) and left in a workspace; recurrence_chunks_kernel then walks a sequence's chunks for 16 value
// columns of a head with the state in the matrix instruction's accumulators.  For the delta rule that leaves of a chunk,
// with T = (I + diag(b) M)^(-1) diag(b),   W = T K~,   u = T V - W S,   o = (A q - P W) S + P T V:
// one product with the state between two states, and the read-outs off that chain.
// Decays arrive as logarithms; their sums over a chunk are kept in 64-bit (base 2) and only differences of two of them (never
// above zero) are exponentiated, so that no quotient of small products is ever formed.  32-bit everywhere else, as in the
// token-by-token kernel.  What is no finite number reaches the tokens from its own on and no earlier one of its chunk: where
// there is any, the products with a triangle of zeros are made token by token (lower_product).
//
// The walk: a wave holds TW tiles of 16 channels.  A tile of the state as it stands in the accumulators (lane group g: rows 4 g ..
// 4 g + 3) is the second operand of the products with it, if product e takes channel 4 g + e of the group on both sides,
// and so are u's rows for the update.  All other operands come straight from memory in the order of their use, four chunks ahead; the
// waves' shares of W S meet in LDS with one barrier a chunk that waits for LDS only, those of the read-outs every four chunks,
// of which each wave finishes one.
//
// What bounds it: the chain of a chunk's products and its barrier, in H dv / 16 blocks.  2,048 tokens, 64 heads of a state of
// 128 x 64: 479 us token by token, 89 in all so; delta rule, 16 heads of 128 x 128: 557 us, 190 so (131 the walk, whose 24 KB of
// operands a chunk and block take a quarter of it, 60 what stands before it).
#include "common.h"
#include "alice_hip.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int C = 16;                      // tokens a chunk

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

constexpr double LOG2E = 1.4426950408889634;
// 2^x for a difference x <= 0 of two sums: the hardware's instruction (1 ulp), on an argument that was scaled in 64-bit
__device__ __forceinline__ float power(double x) { return __builtin_amdgcn_exp2f((float)x); }

// A decay's logarithm to base 2.  One so low that the decay is zero in 32 bits (minus infinity among them) counts as -10,000, so that
// differences of sums with it stay finite; what is no number stays so.
__device__ __forceinline__ double log2_decay(float l) { return (double)(l < -1e4f ? -1e4f : l) * LOG2E; }

struct ChunkArgs {
  const float* q; int q_w, q_col;          // as in recurrent.hip
  const float* k; int k_w, k_col;
  const float* v; int v_w, v_col;
  const float* log_decay;                  // [T, H] or (delta) [T, H d]
  const float* b;                          // [T, H]
  const float* skip;                       // [H] or null
  float* out;                              // [T, H dv]
  float* work;
  const int* cu_seqlens; const int* slots;
  float* S;                                // [slots, H, d, dv]
  int n_seqs, H, G, d, dv;
  int first, run;                          // of every sequence the chunks first .. first + run - 1
  long max_chunks;                         // of all sequences
};

// Floats of the workspace.  State space: a chunk and group K^T [DP][16]; a chunk and head A [16], (A_n / A_r) b [16], P [16][16].
// Delta rule: a chunk and head W [16][DP], A q - P W [16][DP], (A_n / A k)^T [DP][16], A_n [DP], T V [16][dv to 16], P T V likewise.
constexpr int SS_HEAD = 2 * C + C * C;
__host__ __device__ __forceinline__ int delta_head(int DP, int dv) { return 3 * C * DP + DP + 2 * C * ((dv + 15) & ~15); }

// How many chunks of a run are a sequence's of n tokens.
__device__ __forceinline__ int run_chunks(const ChunkArgs& a, int n) { return min(max((n + C - 1) / C - a.first, 0), a.run); }
// Which 16 tokens chunk `at` of the run is: the chunks are dealt to the sequences in order.
__device__ __forceinline__ bool find_chunk(const ChunkArgs& a, int at, int& t0, int& len) {
  for (int s = 0; s < a.n_seqs; ++s) {
    const int b = a.cu_seqlens[s], n = a.cu_seqlens[s + 1] - b, nc = run_chunks(a, n);
    if (at < nc) {
      t0 = b + (a.first + at) * C;
      len = min(C, n - (a.first + at) * C);
      return true;
    }
    at -= nc;
  }
  return false;
}

template <int N>
__device__ __forceinline__ float tree_sum(float (&x)[N]) {
#pragma unroll
  for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i) x[i] += x[i + n];
  return x[0];
}

// o + L x for a chunk's lower triangle L (lane: row c, columns 4 g .. 4 g + 3) and rows x (lane: column c, rows 4 g .. 4 g + 3).  A zero of
// the triangle would not keep an infinity out of an earlier row: if x holds one, or NaN, a token at a time, and the rows before it
// get back what they had.
__device__ __forceinline__ f32x4 lower_product(const float* L, const float* x, f32x4 o, int g) {
  bool odd = false;
#pragma unroll
  for (int e = 0; e < 4; ++e) odd = odd || !(fabsf(x[e]) < INFINITY);
  if (__ballot(odd) == 0ull) {
#pragma unroll
    for (int e = 0; e < 4; ++e) o = mfma(L[e], x[e], o);
  } else {
#pragma unroll 1
    for (int t4 = 0; t4 < 4; ++t4)
#pragma unroll
      for (int e = 0; e < 4; ++e) {                           // token 4 t4 + e
        const f32x4 after = mfma(g == t4 ? L[e] : 0.f, g == t4 ? x[e] : 0.f, o);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = g * 4 + i >= t4 * 4 + e ? after[i] : o[i];
      }
  }
  return o;
}

// ------------------------------------------------------------------------------------------ what does not depend on the state

// State space: a block a (chunk, group of heads with one q and k, 16 of its heads).
constexpr int HB = 16;                     // (times C tokens: a block's threads)
template <int DP>
__global__ __launch_bounds__(256) void ssm_chunk_kernel(ChunkArgs a) {
  __shared__ float qs[C][DP + 1], ks[C][DP + 1];
  __shared__ double ls[HB][C + 1];
  __shared__ float bs[HB][C + 1];
  const int tid = threadIdx.x, grp = blockIdx.y, d = a.d;
  int t0, len;
  if (!find_chunk(a, blockIdx.x, t0, len)) return;
  const int per = a.H / a.G;
  for (int i = tid; i < C * DP; i += 256) {
    const int t = i / DP, c = i % DP;
    const bool in = t < len && c < d;
    const size_t row = t0 + min(t, len - 1);
    const int cc = grp * d + min(c, d - 1);
    const float qv = a.q[row * a.q_w + a.q_col + cc], kv = a.k[row * a.k_w + a.k_col + cc];
    qs[t][c] = in ? qv : 0.f;
    ks[t][c] = in ? kv : 0.f;
  }
  __syncthreads();
  if (blockIdx.z == 0) {
    float* kT = a.work + ((size_t)blockIdx.x * a.G + grp) * DP * C;
    for (int i = tid; i < DP * C; i += 256) kT[i] = ks[i % C][i / C];
  }
  const int t = tid / C, r = tid % C;
  float qk = 0.f;
  if (r <= t) {                                               // sixteen sums: the error of one grows with the key size (zeros behind d)
    float part[16] = {};
    for (int c = 0; c < d; c += 16)
#pragma unroll
      for (int e = 0; e < 16; ++e) part[e] = fmaf(qs[t][c + e], ks[r][c + e], part[e]);
    qk = tree_sum(part);
  }
  const int h0 = blockIdx.z * HB, nh = min(HB, per - h0);      // of the group's heads
  float* heads = a.work + (size_t)a.max_chunks * a.G * DP * C + ((size_t)blockIdx.x * a.H + grp * per + h0) * SS_HEAD;
  {
    const int hh = tid % HB, i = tid / HB;
    const size_t at = (size_t)(t0 + min(i, len - 1)) * a.H + grp * per + h0 + min(hh, nh - 1);
    const float x = a.log_decay[at], w = a.b[at];
    ls[hh][i] = i < len ? log2_decay(x) : 0.0;
    bs[hh][i] = i < len ? w : 0.f;
  }
  __syncthreads();
  if (tid < nh) {
    double l = 0.0;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      l += ls[tid][i];
      ls[tid][i] = l;
    }
  }
  __syncthreads();
  for (int hh = 0; hh < nh; ++hh) {
    float* o = heads + (size_t)hh * SS_HEAD;
    o[2 * C + tid] = r <= t ? qk * (power(ls[hh][t] - ls[hh][r]) * bs[hh][r]) : 0.f;
  }
  if (tid < nh * C) {
    const int hh = tid / C, j = tid % C;
    float* o = heads + (size_t)hh * SS_HEAD;
    o[j] = power(ls[hh][j]);
    o[C + j] = power(ls[hh][C - 1] - ls[hh][j]) * bs[hh][j];
  }
}

// Delta rule: a block a (chunk, head).
template <int DP>
__global__ __launch_bounds__(256) void delta_chunk_kernel(ChunkArgs a) {
  __shared__ float qs[C][DP + 1], ks[C][DP + 1];
  __shared__ double ls[C][DP + 1];
  __shared__ float ms[C][C + 1], ps[C][C + 1], ts[C][C + 1], bs[C];
  const int tid = threadIdx.x, h = blockIdx.y, d = a.d, H = a.H;
  int t0, len;
  if (!find_chunk(a, blockIdx.x, t0, len)) return;
  const int qk_head = h / (H / a.G);
  for (int i = tid; i < C * DP; i += 256) {
    const int t = i / DP, c = i % DP;
    const bool in = t < len && c < d;
    const size_t row = t0 + min(t, len - 1);
    const int cc = qk_head * d + min(c, d - 1);
    const float qv = a.q[row * a.q_w + a.q_col + cc], kv = a.k[row * a.k_w + a.k_col + cc];
    const float lv = a.log_decay[(row * H + h) * d + min(c, d - 1)];
    qs[t][c] = in ? qv : 0.f;
    ks[t][c] = in ? kv : 0.f;
    ls[t][c] = in ? log2_decay(lv) : 0.0;
  }
  if (tid < C) bs[tid] = tid < len ? a.b[(size_t)(t0 + tid) * H + h] : 0.f;
  __syncthreads();
  for (int c = tid; c < DP; c += 256) {
    double l = 0.0;
#pragma unroll
    for (int t = 0; t < C; ++t) {
      l += ls[t][c];
      ls[t][c] = l;
    }
  }
  __syncthreads();
  const int dvp = (a.dv + 15) & ~15;
  float* o = a.work + ((size_t)blockIdx.x * H + h) * delta_head(DP, a.dv);
  for (int i = tid; i < C * DP; i += 256) {
    const int c = i / C, t = i % C;
    o[2 * C * DP + i] = power(ls[C - 1][c] - ls[t][c]) * ks[t][c];
  }
  for (int c = tid; c < DP; c += 256) o[3 * C * DP + c] = power(ls[C - 1][c]);
  // the pairs (t, r <= t): those off the diagonal by two threads, (t, r) for the lower half of the channels and its mirror image for
  // the upper half
  const int t = tid / C, r = tid % C, ht = max(t, r), hr = min(t, r), mid = (d / 2 + 7) & ~7;
  float m, p;
  {
    float mp[8] = {}, pp[8] = {};                             // eight sums each: the error of one grows with the key size (zeros behind d)
    const int c1 = r < t ? mid : d;
    for (int c = r > t ? mid : 0; c < c1; c += 8)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float kk = ks[hr][c + e] * power(ls[ht][c + e] - ls[hr][c + e]);
        mp[e] = fmaf(ks[ht][c + e], kk, mp[e]);
        pp[e] = fmaf(qs[ht][c + e], kk, pp[e]);
      }
    m = tree_sum(mp);
    p = tree_sum(pp);
  }
  ms[t][r] = m;
  ps[t][r] = p;
  __syncthreads();
  if (r < t) {
    m += ms[r][t];
    p += ps[r][t];
  }
  __syncthreads();
  ps[t][r] = r <= t ? p : 0.f;
  if (r < t) ms[t][r] = m;
  // (the pairs are done with the keys and queries: they take their decays to the chunk's start)
  for (int i = tid; i < C * DP; i += 256) {
    const int tt = i / DP, c = i % DP;
    const float A = power(ls[tt][c]);
    ks[tt][c] *= A;
    qs[tt][c] *= A;
  }
  __syncthreads();
  if (tid < C) {                                              // column `tid` of T, from the top
    float x[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
      float s = i == tid ? 1.f : 0.f;
#pragma unroll
      for (int j = 0; j < i; ++j) s = fmaf(-ms[i][j], x[j], s);
      x[i] = bs[i] * s;
      ts[i][tid] = x[i];
    }
  }
  __syncthreads();
  // 16 columns a tile: W and A q - P W, then T V and P T V; what one product leaves is the next one's operand as it stands
  const int lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  float T4[4], P4[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    T4[e] = ts[c][g * 4 + e];
    P4[e] = ps[c][g * 4 + e];
  }
  for (int tile = wave; tile < DP / 16; tile += 4) {
    f32x4 q;
    float k[4], w[4], minus[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      k[e] = ks[g * 4 + e][tile * 16 + c];
      q[e] = qs[g * 4 + e][tile * 16 + c];
      minus[e] = -P4[e];
    }
    const f32x4 w4 = lower_product(T4, k, f32x4{0.f, 0.f, 0.f, 0.f}, g);
#pragma unroll
    for (int e = 0; e < 4; ++e) w[e] = w4[e];
    q = lower_product(minus, w, q, g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[(g * 4 + e) * DP + tile * 16 + c] = w[e];
      o[C * DP + (g * 4 + e) * DP + tile * 16 + c] = q[e];
    }
  }
  float* tv = o + 3 * C * DP + DP;
  for (int tile = wave; tile < dvp / 16; tile += 4) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    float v[4], u[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = a.v[(size_t)(t0 + min(g * 4 + e, len - 1)) * a.v_w + a.v_col + h * a.dv + min(tile * 16 + c, a.dv - 1)];
      v[e] = g * 4 + e < len ? x : 0.f;
    }
    const f32x4 u4 = lower_product(T4, v, zero, g);
#pragma unroll
    for (int e = 0; e < 4; ++e) u[e] = u4[e];
    const f32x4 y = lower_product(P4, u, zero, g);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      tv[(g * 4 + e) * dvp + tile * 16 + c] = u[e];
      tv[C * dvp + (g * 4 + e) * dvp + tile * 16 + c] = y[e];
    }
  }
}

// ------------------------------------------------------------------------------------------ the walk

template <int NW>
__device__ __forceinline__ f32x4 shares_sum(const f32x4 (*r)[64], int lane) {
  f32x4 o = (r[0][lane] + r[1][lane]) + (r[2][lane] + r[3][lane]);
  if constexpr (NW == 8) o += (r[4][lane] + r[5][lane]) + (r[6][lane] + r[7][lane]);
  return o;
}

// A block: one sequence, one head, 16 value columns, all chunks in order, four at a time; wave w holds the state's channels
// w TW 16 .. + TW 16 - 1.
template <int NW, int TW, bool DELTA>
__global__ __launch_bounds__(64 * NW, NW / 4) void recurrence_chunks_kernel(ChunkArgs a) {
  constexpr int DP = 16 * NW * TW;
  __shared__ __align__(16) f32x4 read[2][4][NW][64];          // the waves' shares of four chunks' read-outs, twice
  __shared__ __align__(16) f32x4 part[2][NW][64];             // (delta) of a chunk's W S, twice
  const int h = blockIdx.x, s = blockIdx.y, v0 = blockIdx.z * 16, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int c = lane & 15, g = lane >> 4;
  const int n = run_chunks(a, a.cu_seqlens[s + 1] - a.cu_seqlens[s]);
  if (n <= 0) return;
  const int t0 = a.cu_seqlens[s] + a.first * C, t1 = min(a.cu_seqlens[s + 1], t0 + n * C);
  size_t chunk0 = 0;                                          // this sequence's first chunk in the workspace
  for (int i = 0; i < s; ++i) chunk0 += run_chunks(a, a.cu_seqlens[i + 1] - a.cu_seqlens[i]);
  const int H = a.H, d = a.d, dv = a.dv, last = t1 - 1, grp = h / (H / a.G), dvp = (dv + 15) & ~15;
  const int col = min(v0 + c, dv - 1);
  const bool col_ok = v0 + c < dv;
  float* Sh = a.S + ((size_t)a.slots[s] * H + h) * d * dv;
  f32x4 st[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = (wave * TW + i) * 16 + g * 4 + e;
      const float x = Sh[(size_t)min(r, d - 1) * dv + col];
      st[i][e] = r < d ? x : 0.f;
    }
  const float skip = a.skip ? a.skip[h] : 0.f;

  struct Operands {
    f32x4 q[TW], kT[TW];
    f32x4 w[DELTA ? TW : 1], an[DELTA ? TW : 1];              // W and A_n; (state space) w: (A_n / A_r) b of the lane's four tokens
    float u[4], a_last;                                       // rows of T V; (state space) of V
  };
  struct Finish {                                             // what the chunk that this wave finishes needs
    f32x4 A, P;                                               // (state space)
    float x[4];                                               // rows of P T V; (state space) of V
  };
  // Addresses: a base for the whole wave, moved on chunk by chunk, and lane offsets in bytes that do not change but for the rows of
  // a last, shorter chunk (rows behind the last token repeat it).
  const int head_w = DELTA ? delta_head(DP, dv) : SS_HEAD, len_last = t1 - t0 - (n - 1) * C;
  const char* heads = reinterpret_cast<const char*>(a.work + (DELTA ? 0 : (size_t)a.max_chunks * a.G * DP * C) + (chunk0 * H + h) * head_w);
  const char* keys = reinterpret_cast<const char*>(a.work + (chunk0 * a.G + grp) * DP * C);
  const char* qrows = reinterpret_cast<const char*>(a.q + (size_t)t0 * a.q_w + a.q_col + grp * d);
  const char* vrows = reinterpret_cast<const char*>(a.v + (size_t)t0 * a.v_w + a.v_col + h * dv);
  const char *fin_heads = heads, *fin_v = vrows;
  const size_t head_step = (size_t)H * head_w * 4, key_step = (size_t)a.G * DP * C * 4, q_step = (size_t)C * a.q_w * 4, v_step = (size_t)C * a.v_w * 4;
  const unsigned o_rows = (c * DP + wave * TW * 16 + g * 4) * 4, o_kT = ((wave * TW * 16 + c) * C + g * 4) * 4, o_an = (wave * TW * 16 + g * 4) * 4;
  unsigned o_q[TW], o_ql[TW], o_u[4], o_ul[4];
  if (DELTA) {
#pragma unroll
    for (int e = 0; e < 4; ++e) o_u[e] = o_ul[e] = (3 * C * DP + DP + (g * 4 + e) * dvp + v0 + c) * 4;
  } else {
#pragma unroll
    for (int w = 0; w < TW; ++w) {
      const int k = min((wave * TW + w) * 16 + g * 4, d - 4);        // channels beyond d meet a zero of the state
      o_q[w] = (c * a.q_w + k) * 4;
      o_ql[w] = (min(c, len_last - 1) * a.q_w + k) * 4;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o_u[e] = ((g * 4 + e) * a.v_w + col) * 4;
      o_ul[e] = (min(g * 4 + e, len_last - 1) * a.v_w + col) * 4;
    }
  }
  auto ld4 = [](const char* base, unsigned off) { return *reinterpret_cast<const f32x4*>(base + off); };
  auto ld1 = [](const char* base, unsigned off) { return *reinterpret_cast<const float*>(base + off); };
  int next = 0;                                               // the chunk that the bases stand at
  auto fetch = [&](Operands& x) {
    if (DELTA) {
#pragma unroll
      for (int w = 0; w < TW; ++w) {
        x.w[w] = ld4(heads, o_rows + w * 64);
        x.q[w] = ld4(heads, o_rows + C * DP * 4 + w * 64);
        x.kT[w] = ld4(heads, o_kT + 2 * C * DP * 4 + w * 16 * C * 4);
        x.an[w] = ld4(heads, o_an + 3 * C * DP * 4 + w * 64);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) x.u[e] = ld1(heads, o_u[e]);
    } else {
      const bool short_one = next == n - 1;
#pragma unroll
      for (int w = 0; w < TW; ++w) {
        x.kT[w] = ld4(keys, o_kT + w * 16 * C * 4);
        x.q[w] = ld4(qrows, short_one ? o_ql[w] : o_q[w]);
      }
      x.w[0] = ld4(heads, C * 4 + g * 16);                    // (zero at the places behind the last token)
      x.a_last = ld1(heads, (C - 1) * 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) x.u[e] = ld1(vrows, short_one ? o_ul[e] : o_u[e]);
    }
    if (++next < n) {
      heads += head_step;
      keys += key_step;
      qrows += q_step;
      vrows += v_step;
    } else {
      next = n - 1;
    }
  };
  auto fetch_finish = [&](Finish& fin, int i) {
    const char* o = fin_heads + (size_t)i * head_step;
    if (DELTA) {
#pragma unroll
      for (int e = 0; e < 4; ++e) fin.x[e] = ld1(o, o_u[e] + C * dvp * 4);
    } else {
      fin.A = ld4(o, g * 16);
      fin.P = ld4(o, (2 * C + c * C + g * 4) * 4);
      const char* v = fin_v + (size_t)i * v_step;
#pragma unroll
      for (int e = 0; e < 4; ++e) fin.x[e] = ld1(v, i == n - 1 ? o_ul[e] : o_u[e]);
    }
  };
  auto step = [&](const Operands& x, int i) {
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const int half = i & 1;
    if (DELTA) {                                              // this wave's share of W S
      f32x4 w0 = zero, w1 = zero;
#pragma unroll
      for (int w = 0; w < TW; ++w)
#pragma unroll
        for (int e = 0; e < 4; e += 2) {
          w0 = mfma(x.w[w][e], st[w][e], w0);
          w1 = mfma(x.w[w][e + 1], st[w][e + 1], w1);
        }
      part[half][wave][lane] = w0 + w1;
      lds_barrier();
    }
    f32x4 q0 = zero, q1 = zero;                               // its share of the read-outs of the state ahead of the chunk
#pragma unroll
    for (int w = 0; w < TW; ++w)
#pragma unroll
      for (int e = 0; e < 4; e += 2) {
        q0 = mfma(x.q[w][e], st[w][e], q0);
        q1 = mfma(x.q[w][e + 1], st[w][e + 1], q1);
      }
    f32x4 up;                                                 // the rows that the four tokens of the lane's group write
    if (DELTA) {
      const f32x4 ws = shares_sum<NW>(part[half], lane);
#pragma unroll
      for (int e = 0; e < 4; ++e) up[e] = x.u[e] - ws[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) up[e] = x.w[0][e] * x.u[e];
    }
#pragma unroll
    for (int w = 0; w < TW; ++w) st[w] *= DELTA ? x.an[w] : f32x4{x.a_last, x.a_last, x.a_last, x.a_last};
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int w = 0; w < TW; ++w) st[w] = mfma(x.kT[w][e], up[e], st[w]);
    read[(i >> 2) & 1][i & 3][wave][lane] = q0 + q1;
  };
  auto finish = [&](const Finish& fin, int i) {
    const f32x4(*r)[64] = read[(i >> 2) & 1][i & 3];
    const int tb = t0 + i * C + g * 4;
    f32x4 o = shares_sum<NW>(r, lane);
    if (DELTA) {
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] += fin.x[e];
    } else {
      const float P[4] = {fin.P[0], fin.P[1], fin.P[2], fin.P[3]};
      o = lower_product(P, fin.x, o * fin.A, g);
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = fmaf(skip, fin.x[e], o[e]);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (col_ok && tb + e < t1) a.out[(size_t)(tb + e) * H * dv + h * dv + v0 + c] = o[e];
  };
  // Fetches are unconditional (a chunk beyond the last repeats it): behind a condition the compiler could not tell how many
  // loads are younger than the ones it waits for, and would wait for all of them.  For the same reason the last chunks, fewer than
  // four, are fetched anew: what the loop carries then has one place, and no copy of it waits for the youngest loads.
  int base = 0;
  if (n >= 4) {
    Operands buf[4];
    Finish fin;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      fetch(buf[u]);
      __builtin_amdgcn_sched_barrier(0);                      // (the order of the loads is the order of their use)
    }
    fetch_finish(fin, wave & 3);
    for (; base + 4 <= n; base += 4) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        step(buf[u], base + u);
        __builtin_amdgcn_sched_barrier(0);
        fetch(buf[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
      lds_barrier();
      if (wave < 4) finish(fin, base + wave);
      fetch_finish(fin, min(base + 4 + (wave & 3), n - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (base < n) {
    const size_t back = next - base;
    heads -= back * head_step;
    keys -= back * key_step;
    qrows -= back * q_step;
    vrows -= back * v_step;
    next = base;
    Operands buf[3];
    Finish fin;
#pragma unroll
    for (int u = 0; u < 3; ++u) fetch(buf[u]);
    fetch_finish(fin, min(base + (wave & 3), n - 1));
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (base + u < n) step(buf[u], base + u);
    lds_barrier();
    if (wave < 4 && base + wave < n) finish(fin, base + wave);
  }
#pragma unroll
  for (int i = 0; i < TW; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int r = (wave * TW + i) * 16 + g * 4 + e;
      if (col_ok && r < d) Sh[(size_t)r * dv + v0 + c] = st[i][e];
    }
}

int padded(int d) { return d <= 64 ? 64 : (d <= 128 ? 128 : 256); }

template <int NW, int TW>
int launch(const ChunkArgs& a, int delta, hipStream_t stream) {
  constexpr int DP = 16 * NW * TW;
  const dim3 walk(a.H, a.n_seqs, ceil_div(a.dv, 16));
  if (delta) {
    delta_chunk_kernel<DP><<<dim3((unsigned)a.max_chunks, a.H), 256, 0, stream>>>(a);
    ALICE_LAUNCH_CHECK();
    recurrence_chunks_kernel<NW, TW, true><<<walk, 64 * NW, 0, stream>>>(a);
  } else {
    ssm_chunk_kernel<DP><<<dim3((unsigned)a.max_chunks, a.G, ceil_div(a.H / a.G, HB)), 256, 0, stream>>>(a);
    ALICE_LAUNCH_CHECK();
    recurrence_chunks_kernel<NW, TW, false><<<walk, 64 * NW, 0, stream>>>(a);
  }
  ALICE_LAUNCH_CHECK();
  return 0;
}

// The workspace holds a step's chunks at once up to WORK_MOST floats (256 MB: 6,400 tokens with 16 heads of 128 x 128 under the delta rule,
// 41 KB a token; the state space takes 5 KB a token with 64 heads).  A longer step goes in runs of that many chunks, each with the
// state that the one before left: the same numbers, and a microsecond or two a run.
constexpr long WORK_MOST = 1l << 26;
struct Runs {
  int run;                                 // chunks of every sequence a run
  long chunks;                             // chunks of all sequences a run, at most
};
long chunk_floats(int H, int G, int d, int dv, int delta) {
  return delta ? (long)H * delta_head(padded(d), dv) : G * (long)padded(d) * C + H * (long)SS_HEAD;
}
Runs runs_of(int T, int n_seqs, int H, int G, int d, int dv, int delta) {
  const long all = (long)T / C + n_seqs, fit = WORK_MOST / chunk_floats(H, G, d, dv, delta);
  if (all <= fit) return {T / C + 1, all};
  const long run = fit / n_seqs > 1 ? fit / n_seqs : 1;
  return {(int)run, run * n_seqs < all ? run * n_seqs : all};
}

}  // namespace

// Float32 workspace of alice_recurrence_chunks for a step of T tokens in n_seqs sequences; 0 where the sizes are outside
// its range (key sizes that are no multiples of four: the queries are read 16 bytes at a time).
extern "C" long alice_recurrence_chunks_workspace(int T, int n_seqs, int H, int qk_heads, int d, int dv, int delta) {
  if (T < 0 || dv < 1 || n_seqs < 1 || H < 1 || qk_heads < 1 || H % qk_heads || d < 4 || d > 256 || d % 4 || H > 65535 || n_seqs > 65535) return 0;
  return runs_of(T, n_seqs, H, qk_heads, d, dv, delta).chunks * chunk_floats(H, qk_heads, d, dv, delta);
}

// longest: tokens of the longest sequence.
extern "C" int alice_recurrence_chunks(const float* q, int q_w, int q_col, const float* k, int k_w, int k_col, const float* v, int v_w,
                                       int v_col, const float* log_decay, const float* b, const float* skip, float* out, float* work,
                                       const int* cu_seqlens, const int* slots, float* S, int T, int n_seqs, int longest, int H,
                                       int qk_heads, int d, int dv, int delta, hipStream_t stream) {
  ALICE_CHECK(q && k && v && log_decay && b && out && work && cu_seqlens && slots && S, "recurrence_chunks: a pointer is missing");
  ALICE_CHECK(T >= 0 && n_seqs >= 0 && longest >= 0 && longest <= T && dv >= 1 && ceil_div(dv, 16) <= 65535, "recurrence_chunks: bad sizes");
  if (n_seqs == 0 || T == 0) return 0;
  ALICE_CHECK(alice_recurrence_chunks_workspace(T, n_seqs, H, qk_heads, d, dv, delta) > 0, "recurrence_chunks: heads %d / %d of size %d are outside this kernel's range", H, qk_heads, d);
  ALICE_CHECK(q_col >= 0 && k_col >= 0 && v_col >= 0 && q_col + qk_heads * d <= q_w && k_col + qk_heads * d <= k_w && v_col + H * dv <= v_w,
              "recurrence_chunks: the rows are too short for the heads");
  ALICE_CHECK(((uintptr_t)q & 15) == 0 && q_w % 4 == 0 && q_col % 4 == 0 && ((uintptr_t)work & 15) == 0, "recurrence_chunks: operands are not aligned");
  const Runs r = runs_of(T, n_seqs, H, qk_heads, d, dv, delta);
  ALICE_CHECK(r.chunks < (1l << 31), "recurrence_chunks: too many chunks for one launch");
  for (int first = 0; first * C < longest; first += r.run) {
    const ChunkArgs a{q, q_w, q_col, k, k_w, k_col, v, v_w, v_col, log_decay, b, skip, out, work, cu_seqlens, slots, S, n_seqs, H, qk_heads, d,
                      dv, first, r.run, r.chunks};
    int rc;
    // Eight waves a block while the blocks are few (2,048 tokens: 131 against 138 us, state space 81 against 91), four where several
    // blocks share a CU (8 sequences of 1,000: 503 against 534 us with the preparation, 295 against 344).
    if (d <= 64) rc = launch<4, 1>(a, delta, stream);
    else if (d <= 128) rc = (long)H * n_seqs * ceil_div(dv, 16) < 512 ? launch<8, 1>(a, delta, stream) : launch<4, 2>(a, delta, stream);
    else rc = launch<8, 2>(a, delta, stream);
    if (rc) return rc;
  }
  return 0;
}
