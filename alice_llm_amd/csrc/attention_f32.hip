// Attention of the true 32-bit path over a row-major paged cache on the 32-bit matrix instruction
// (v_mfma_f32_16x16x4_f32: 32-bit products and sums): prompts, pieces and single tokens alike, causal, with a window and
// a softcap, in the order of the reference (llama3.rs:5622-5688): dot product, times scale, cap * tanh(s / cap), softmax
// over the keys max(0, pos + 1 - window) .. pos, weighted sum of the values.
//
// A tile's 16 columns are (query, head) pairs: 16 / (heads a kv head) neighbouring queries of one sequence with all heads
// of one kv head's group, so that a key serves the group.  A block of four waves takes one tile; the keys go in tiles
// of 16 to the waves of the `splits` blocks in turn.  S^T = K Q^T has the keys as rows: a lane ends up with four scores of ONE
// column, which are, as they stand, the second operand of O^T = V^T P^T (product i takes key 4 g + i of lane group g on
// both sides).  Keys, values and queries come straight from memory in 16-byte pieces into the matrix instruction's
// operands: in a chunk of 16 dimensions lane group g holds the dimensions 4 g .. 4 g + 3 of its key (the order of the
// inner dimension is the same for the queries), in a chunk of 64 value dimensions lane c holds 4 c .. 4 c + 3, which
// permutes the rows of O^T and nothing else.  No LDS but for the four waves' results at the end.  A tile's values are on their way while its
// scores are made, the next tile's keys while its values are used.
//
// What bounds it: with a prompt the matrix instruction (4,096 cycles a wave for 16 keys by 16 columns at size 256, half
// of it for columns and keys that the causal mask hides near the diagonal); with single tokens the way of a key from
// memory.  500 tokens, 8 heads over 4 of 256: 1,048 us with a block a (token, head) on scalar loads before, 40 us so;
// 4 single tokens at 300 to 700 keys 608 us before, 17 us with the combine.
#include "common.h"
#include "alice_hip.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct F32Args {
  const float* q;
  const float* k_pool;
  const float* v_pool;
  float* out;
  const int* positions;
  const int* cu_seqlens;      // null: every sequence brings one token
  const int* block_table;
  int bt_stride, n_seqs, nH, nKV, page_size;
  float scale, cap;
  int window, splits;
  float* part_ml;             // [T, nH, splits, 2]   (splits > 1)
  float* part_o;              // [T, nH, splits, D]
};

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <int D>
__global__ __launch_bounds__(256) void attn_f32_kernel(F32Args a) {
  constexpr int KC = D / 16, VC = D / 64;
  __shared__ float osh[3][D / 4][64];
  __shared__ float msh[4][16], lsh[4][16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  const int kvh = blockIdx.y, split = blockIdx.z, per = a.nH / a.nKV, qpt = 16 / per;

  // which queries: the tiles are dealt to the sequences in order; the last queries of a sequence have the most keys, so
  // they go first
  int seq = -1, q0 = 0, nq = 0;
  if (a.cu_seqlens == nullptr) {
    seq = q0 = blockIdx.x;
    nq = 1;
  } else {
    int idx = gridDim.x - 1 - blockIdx.x;
    for (int s = 0; s < a.n_seqs; ++s) {
      const int b = a.cu_seqlens[s], e = a.cu_seqlens[s + 1], n = (e - b + qpt - 1) / qpt;
      if (idx < n) {
        seq = s;
        q0 = b + idx * qpt;
        nq = min(qpt, e - q0);
        break;
      }
      idx -= n;
    }
  }
  if (seq < 0) return;
  const int* bt = a.block_table + (size_t)seq * a.bt_stride;
  const int p_first = a.positions[q0], p_last = p_first + nq - 1;
  const bool valid = c < nq * per;
  const int qi = valid ? c / per : 0, h = kvh * per + (valid ? c % per : 0), t = q0 + qi;
  const int qpos = p_first + qi;
  const int lo_q = a.window > 0 ? max(0, qpos + 1 - a.window) : 0;
  const int lo = a.window > 0 ? max(0, p_first + 1 - a.window) : 0;
  const int lo_last = a.window > 0 ? max(0, p_last + 1 - a.window) : 0;       // keys lo_last .. p_first: every query sees them

  f32x4 qf[KC];
  const float* qrow = a.q + ((size_t)t * a.nH + h) * D + g * 4;
#pragma unroll
  for (int k = 0; k < KC; ++k) qf[k] = *reinterpret_cast<const f32x4*>(qrow + k * 16);

  f32x4 o[D / 16];
#pragma unroll
  for (int k = 0; k < D / 16; ++k) o[k] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_run = 0.f;

  const int t_hi = p_last >> 4, step = 4 * a.splits;
  int kt = (lo >> 4) + split * 4 + wave;
  f32x4 kf[KC];
  // the 16 keys of a tile lie in one page (pages are multiples of 16 positions)
  auto page_row = [&](int tile) -> size_t {
    const int key0 = tile * 16;
    return ((size_t)bt[key0 / a.page_size] * a.nKV + kvh) * a.page_size + key0 % a.page_size;
  };
  auto fetch_keys = [&](size_t row) {
    const float* p = a.k_pool + (row + c) * D + g * 4;
#pragma unroll
    for (int k = 0; k < KC; ++k) kf[k] = *reinterpret_cast<const f32x4*>(p + k * 16);
  };
  size_t row = 0, row_next = 0;
  if (kt <= t_hi) {
    row = page_row(kt);
    fetch_keys(row);
  }
  for (; kt <= t_hi; kt += step) {
    const int key0 = kt * 16;
    if (kt + step <= t_hi) row_next = page_row(kt + step);
    // values of the keys 4 g + i; places that hold no key of this sequence's range give zeros
    f32x4 vf[4][VC];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kp = key0 + g * 4 + i;
      const bool there = kp >= lo && kp <= p_last;
      const float* p = a.v_pool + (row + g * 4 + i) * D + c * 4;
#pragma unroll
      for (int k = 0; k < VC; ++k) {
        vf[i][k] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (there) vf[i][k] = *reinterpret_cast<const f32x4*>(p + k * 64);
      }
    }
    f32x4 s0 = {0.f, 0.f, 0.f, 0.f}, s1 = s0, s2 = s0, s3 = s0;
#pragma unroll
    for (int k = 0; k < KC; ++k) {
      s0 = mfma(kf[k][0], qf[k][0], s0);
      s1 = mfma(kf[k][1], qf[k][1], s1);
      s2 = mfma(kf[k][2], qf[k][2], s2);
      s3 = mfma(kf[k][3], qf[k][3], s3);
    }
    if (kt + step <= t_hi) fetch_keys(row_next);
    const f32x4 sT = (s0 + s1) + (s2 + s3);
    float p[4], m_t = -INFINITY;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int kp = key0 + g * 4 + i;
      float v = sT[i] * a.scale;
      if (a.cap > 0.f) v = a.cap * tanh_full(v / a.cap);
      p[i] = valid && kp <= qpos && kp >= lo_q ? v : -INFINITY;
      m_t = fmaxf(m_t, p[i]);
    }
    m_t = fmaxf(m_t, __shfl_xor(m_t, 16, 64));
    m_t = fmaxf(m_t, __shfl_xor(m_t, 32, 64));
    const float m_new = fmaxf(m_run, m_t);
    const bool any = m_new > -INFINITY;
    const float corr = any ? expf(m_run - m_new) : 1.f;       // m_run = -inf gives 0
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      p[i] = any ? expf(p[i] - m_new) : (p[i] != p[i] ? p[i] : 0.f);      // (a maximum passes over what is no number: that stays)
      sum += p[i];
    }
    m_run = m_new;
    l_run = fmaf(l_run, corr, sum);
#pragma unroll
    for (int k = 0; k < D / 16; ++k) o[k] *= corr;
    // A value that is no finite number must reach the queries that see its key and no others: a weight of zero would
    // not keep it out.  Where some query of the tile does not see all 16 keys, look, and if there is one, go query by query.
    bool odd = false;
    if (key0 < lo_last || key0 + 15 > p_first) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < VC; ++k)
#pragma unroll
          for (int j = 0; j < 4; ++j) odd = odd || !(fabsf(vf[i][k][j]) < INFINITY);
    }
    if (__ballot(odd) == 0ull) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < VC; ++k)
#pragma unroll
          for (int j = 0; j < 4; ++j) o[k * 4 + j] = mfma(vf[i][k][j], p[i], o[k * 4 + j]);
    } else {
      for (int x = 0; x < nq; ++x) {
        const int xpos = p_first + x, xlo = a.window > 0 ? max(0, xpos + 1 - a.window) : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int kp = key0 + g * 4 + i;
          const bool sees = kp <= xpos && kp >= xlo;
          const float px = valid && qi == x ? p[i] : 0.f;
#pragma unroll
          for (int k = 0; k < VC; ++k)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              // the other queries' columns get 0 * value: their results so far are put back
              const f32x4 before = o[k * 4 + j];
              const f32x4 after = mfma(sees ? vf[i][k][j] : 0.f, px, before);
#pragma unroll
              for (int e = 0; e < 4; ++e) o[k * 4 + j][e] = valid && qi == x ? after[e] : before[e];
            }
        }
      }
    }
    row = row_next;
  }

  // the four waves meet: maximum, sum and output of every column
  float l_col = l_run;
  l_col += __shfl_xor(l_col, 16, 64);
  l_col += __shfl_xor(l_col, 32, 64);
  if (g == 0) {
    msh[wave][c] = m_run;
    lsh[wave][c] = l_col;
  }
  if (wave > 0) {
#pragma unroll
    for (int k = 0; k < D / 16; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e) osh[wave - 1][k * 4 + e][lane] = o[k][e];
  }
  __syncthreads();
  if (wave > 0) return;
  float M = msh[0][c], f[4], L = 0.f;
#pragma unroll
  for (int w = 1; w < 4; ++w) M = fmaxf(M, msh[w][c]);
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    f[w] = msh[w][c] > -INFINITY ? expf(msh[w][c] - M) : 0.f;
    L = fmaf(lsh[w][c], f[w], L);
  }
#pragma unroll
  for (int k = 0; k < D / 16; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = o[k][e] * f[0];
#pragma unroll
      for (int w = 1; w < 4; ++w) v = fmaf(osh[w - 1][k * 4 + e][lane], f[w], v);
      o[k][e] = v;
    }
  if (!valid) return;
  float* dst;
  float div = 1.f;
  if (a.splits > 1) {
    const size_t at = ((size_t)t * a.nH + h) * a.splits + split;
    if (g == 0) {
      a.part_ml[at * 2] = M;
      a.part_ml[at * 2 + 1] = L;
    }
    dst = a.part_o + at * D;
  } else {
    dst = a.out + ((size_t)t * a.nH + h) * D;
    div = L;
  }
#pragma unroll
  for (int k = 0; k < VC; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f32x4 v = {o[k * 4][e], o[k * 4 + 1][e], o[k * 4 + 2][e], o[k * 4 + 3][e]};
      if (a.splits == 1) v /= div;
      *reinterpret_cast<f32x4*>(dst + k * 64 + (g * 4 + e) * 4) = v;
    }
}

// The splits' results of one (token, head), merged in their order; a thread takes four dimensions.
__global__ void attn_f32_combine_kernel(const float* __restrict__ part_ml, const float* __restrict__ part_o, float* __restrict__ out,
                                        int S, int D) {
  const size_t row = blockIdx.x;
  const float* ml = part_ml + row * S * 2;
  const f32x4* po = reinterpret_cast<const f32x4*>(part_o + row * S * D) + threadIdx.x;
  float M = -INFINITY;
  for (int s = 0; s < S; ++s) M = fmaxf(M, ml[2 * s]);
  float L = 0.f;
  f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int s = 0; s < S; ++s) {
    const float f = ml[2 * s] > -INFINITY ? expf(ml[2 * s] - M) : 0.f;
    L = fmaf(ml[2 * s + 1], f, L);
    v += po[(size_t)s * (D / 4)] * f;
  }
  reinterpret_cast<f32x4*>(out + row * D)[threadIdx.x] = v / L;
}

}  // namespace

extern "C" int alice_attention_f32_supported(int nH, int nKV, int d, int page_size) {
  return nKV >= 1 && nH % nKV == 0 && nH / nKV <= 16 && nH <= 65535 && (d == 64 || d == 128 || d == 256) && page_size >= 16 && page_size % 16 == 0;
}

// Blocks that a tile's keys go to.  One where the tiles alone give every CU a block or there are few keys: a wave then
// walks its quarter of the keys, and no second launch is needed.  Else as many as fill the CUs, while every wave of a
// block still gets a tile of 16 keys.
extern "C" int alice_attention_f32_splits(int tiles, int nKV, int max_keys) {
  const int blocks = tiles * nKV;
  if (blocks < 1 || blocks >= 192 || max_keys <= 128) return 1;
  return max(1, min(min(ceil_div(256, blocks), max_keys / 64), 32));
}

// q, out: float32 [T, nH d]; pools: float32 [pages, nKV, page, d]; work: T nH splits (d + 2) floats where splits > 1.
// single_tokens: every sequence brings one token (T == n_seqs).
extern "C" int alice_attention_f32(const float* q, const float* k_pool, const float* v_pool, float* out, const int* positions,
                                   const int* cu_seqlens, const int* block_table, int bt_stride, int T, int n_seqs, int single_tokens,
                                   int nH, int nKV, int d, int page_size, float scale, float softcap, int window, int splits,
                                   float* work, hipStream_t stream) {
  ALICE_CHECK(alice_attention_f32_supported(nH, nKV, d, page_size), "attention: heads %d / %d of size %d on pages of %d are outside this kernel's range", nH, nKV, d, page_size);
  ALICE_CHECK(q && k_pool && v_pool && out && positions && cu_seqlens && block_table, "attention: a pointer is missing");
  ALICE_CHECK(T >= 0 && n_seqs >= 1 && bt_stride > 0 && softcap >= 0.f && window >= 0, "attention: bad sizes");
  ALICE_CHECK(!single_tokens || T == n_seqs, "attention: %d single tokens of %d sequences", T, n_seqs);
  ALICE_CHECK(splits >= 1 && splits <= 65535 && (splits == 1 || work), "attention: bad number of key splits %d", splits);
  ALICE_CHECK((((uintptr_t)q | (uintptr_t)k_pool | (uintptr_t)v_pool | (uintptr_t)out | (uintptr_t)work) & 15) == 0, "attention: operands are not aligned");
  if (T == 0) return 0;
  const size_t rows = (size_t)T * nH;
  float* part_o = work;                                       // the rows first: 16-byte aligned
  F32Args a{q, k_pool, v_pool, out, positions, single_tokens ? nullptr : cu_seqlens, block_table, bt_stride, n_seqs, nH, nKV, page_size,
            scale, softcap, window, splits, splits > 1 ? work + rows * splits * d : nullptr, part_o};
  const int qpt = 16 / (nH / nKV);
  dim3 grid(single_tokens ? T : ceil_div(T, qpt) + n_seqs, nKV, splits);
  if (d == 64) attn_f32_kernel<64><<<grid, 256, 0, stream>>>(a);
  else if (d == 128) attn_f32_kernel<128><<<grid, 256, 0, stream>>>(a);
  else attn_f32_kernel<256><<<grid, 256, 0, stream>>>(a);
  ALICE_LAUNCH_CHECK();
  if (splits > 1) {
    ALICE_CHECK(rows < (1ul << 31), "attention: too many rows for one launch");
    attn_f32_combine_kernel<<<(unsigned)rows, d / 4, 0, stream>>>(a.part_ml, a.part_o, out, splits, d);
    ALICE_LAUNCH_CHECK();
  }
  return 0;
}
