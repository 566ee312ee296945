// Matrix product y[M, N] = x[M, K] . W[N, K]^T for every combination of 32-bit and bfloat16
// operands, with 32-bit products and 32-bit accumulation: the kernels of the true 32-bit path, and
// the fallback of the bfloat16 path for matrices that stay in 32-bit.  (Of more than 16 tokens most products of 32-bit
// operands go to linear_thirds.hip, see in_thirds().)
//
// Weight layout and orientation as in the reference: row-major [out, in], y[r] = sum_c W[r,c] x[c]
// (gguf.rs:4063-4074, f32_matvec).  Epilogues: none; GeGLU gelu_tanh(gate) * up with W = [gate; up]
// stacked (llama3.rs:14519-14534); softcap cap * tanh(y / cap) (llama3.rs:14606-14611).
#include "common.h"
#include "alice_hip.h"
#include "linear_thirds.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Inner elements a stage; a row of a stage in LDS is eight 16-byte pieces, piece p of row r at p ^ (r / 2 % 8): the pieces that
// 16 lanes read (one of 16 neighbouring rows) or write (two whole rows) at a time lie in different banks.
constexpr int BK = 32;

// Four neighbouring elements of a row as float32.  VEC: in one load (rows start at multiples of four elements on memory
// aligned for them, K is a multiple of four); else one by one, none beyond the row's end.  Loads are unconditional: one
// behind a condition would be waited for where the ways join.
template <typename T> __device__ __forceinline__ f32x4 load4(const T* __restrict__ p);
template <> __device__ __forceinline__ f32x4 load4<float>(const float* __restrict__ p) { return *reinterpret_cast<const f32x4*>(p); }
template <> __device__ __forceinline__ f32x4 load4<bf16_t>(const bf16_t* __restrict__ p) {
  const uint2 w = *reinterpret_cast<const uint2*>(p);
  return f32x4{bf16_bits_to_f32(w.x & 0xffffu), bf16_bits_to_f32(w.x >> 16), bf16_bits_to_f32(w.y & 0xffffu), bf16_bits_to_f32(w.y >> 16)};
}
template <typename T, bool VEC>
__device__ __forceinline__ f32x4 load_row4(const T* __restrict__ row, int k, int end) {
  if constexpr (VEC) return load4<T>(row + min(k, end - 4));
  return f32x4{load_f32(row, min(k, end - 1)), load_f32(row, min(k + 1, end - 1)), load_f32(row, min(k + 2, end - 1)), load_f32(row, min(k + 3, end - 1))};
}

// More than 16 tokens of what linear_thirds.hip does not take (an operand in bfloat16, unaligned rows, or no time to gain there):
// the 32-bit matrix instruction (v_mfma_f32_16x16x4_f32: 32-bit products and sums, the rate of the vector unit's FMA at a quarter
// of its register reads).  A block of 2 x 2 waves takes 32 TM tokens by 32 TN rows of W, a
// wave 16 TM by 16 TN; both operands go through LDS 32 inner elements at a time in two buffers (one barrier a stage), the
// stage after the next on its way from memory meanwhile.  Every LDS and memory instruction stands behind a product of the
// same wave: with all of them ahead of a stage's products the waves of a SIMD fell into step and left the matrix unit idle
// a quarter of the time.  A lane reads 16-byte pieces: lane group g of a 16-element chunk holds the
// elements 4 g .. 4 g + 3 of its row, and product i of the chunk takes element i of every group, the same permutation of
// the inner dimension on both sides.  W is the first operand, so that a lane ends up with four neighbouring outputs of a
// token.  With GeGLU the first half of a wave's rows are gate rows, the second half the up rows of the same outputs.
// blockIdx: the tiles of one set of W rows are neighbours on one XCD, whose L2 then serves W's rows to all of them.
// split: slices of the inner dimension, slice z to Y + z M N (float32 sums that the residual add adds up).
//
// What bounds it: the matrix instruction (157 TFLOP/s at 256 CUs and 2.4 GHz, 141 at the 2.15 GHz that it runs at under this
// load; 512 tokens by 16,384 x 2,304 rows reach 129).  A product of 500 tokens with 18,432 x 2,304 rows and GeGLU takes
// 350 us (122 TFLOP/s), the down product of 2,304 x 9,216 176 us (120) in slices; 438 and 188 with the instructions of a
// stage ahead of its products, 1,576 and 1,444 with a 64 x 64 tile of scalar FMAs.
template <typename TA, typename TW, typename TO, int TM, int TN, bool VEC>
__global__ __launch_bounds__(256) void linear_mfma32_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TO* __restrict__ Y,
                                                            int M, int N, int K, int kslice, int mt, int nt, int epi, float param,
                                                            int full, int wide) {
  constexpr int BM = 32 * TM, BN = 32 * TN;
  constexpr int YROW = BN + 4;
  constexpr int STAGES = 2 * (BM + BN) * BK;
  __shared__ __align__(16) float lds[STAGES > BM * YROW ? STAGES : BM * YROW];
  auto As = reinterpret_cast<float (*)[BM][BK]>(lds);
  auto Bs = reinterpret_cast<float (*)[BN][BK]>(lds + 2 * BM * BK);
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;

  // tile of this block: neighbours in m first, a run of tiles an XCD (blocks go to the 8 XCDs in turn)
  const int total = mt * nt, per = (total + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile >= total) return;                                  // the whole block: no barrier is missed
  const int m0 = (tile % mt) * BM, nb = tile / mt;
  const bool geglu = epi == ALICE_EPI_GEGLU;
  const int n0 = nb * (geglu ? BN / 2 : BN);
  const int k_begin = blockIdx.y * kslice, k_end = min(K, k_begin + kslice);

  // loaders: 16-byte piece `id` of a stage is row id / 8, elements (id % 8) * 4; lw, sw: where it is written, what is read (see BK)
  const int lk = (tid & 7) * 4, lr = tid >> 3, lw = lk ^ (lr / 2 % 8 * 4), sw = c / 2 % 8 * 4;
  const TA* arow[TM];                                         // rows beyond the last are read as the last and not written
  const TW* wrow[TN];
#pragma unroll
  for (int j = 0; j < TM; ++j) arow[j] = A + (size_t)min(m0 + lr + 32 * j, M - 1) * K;
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int r = lr + 32 * j;
    int row = min(n0 + r, N - 1);
    if (geglu) {                                              // a wave's 16 TN rows: gate rows, then up rows of the same outputs
      const int w = r / (16 * TN), rr = r % (16 * TN), half = rr / (8 * TN);
      row = half * N + min(n0 + w * 8 * TN + rr % (8 * TN), N - 1);
    }
    wrow[j] = W + (size_t)row * K;
  }
  f32x4 pa[TM], pb[TN];                                       // the stage on its way from memory
  auto load = [&](int n, int k0) {                            // its n-th piece
    if (n < TM) pa[n] = load_row4<TA, VEC>(arow[n], k0 + lk, k_end);
    else pb[n - TM] = load_row4<TW, VEC>(wrow[n - TM], k0 + lk, k_end);
  };
  auto clear_beyond = [&](int k0) {                           // the last stage of a slice: nothing beyond its end
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = k0 + lk + e < k_end;
#pragma unroll
      for (int j = 0; j < TM; ++j) pa[j][e] = in ? pa[j][e] : 0.f;
#pragma unroll
      for (int j = 0; j < TN; ++j) pb[j][e] = in ? pb[j][e] : 0.f;
    }
  };
  auto write = [&](int n, int buf) {
    if (n < TM) *reinterpret_cast<f32x4*>(&As[buf][lr + 32 * n][lw]) = pa[n];
    else *reinterpret_cast<f32x4*>(&Bs[buf][lr + 32 * (n - TM)][lw]) = pb[n - TM];
  };
  f32x4 f0[TN + TM], f1[TN + TM];                             // operands of a stage's first and second 16 elements
  auto read = [&](f32x4 (&f)[TN + TM], int n, int buf, int ch) {
    if (n < TN) f[n] = *reinterpret_cast<const f32x4*>(&Bs[buf][(wn * TN + n) * 16 + c][(ch + g * 4) ^ sw]);
    else f[n] = *reinterpret_cast<const f32x4*>(&As[buf][(wm * TM + n - TN) * 16 + c][(ch + g * 4) ^ sw]);
  };
  f32x4 acc[TN][TM];
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The products of 16 elements with one other instruction behind each (op(0) .. op(ops - 1)): it is issued while the product
  // runs.
  constexpr int PRODUCTS = 4 * TM * TN, PIECES = TM + TN, READS = TN + TM;
  auto products = [&](const f32x4 (&f)[TN + TM], int ops, auto&& op) {
#pragma unroll
    for (int p = 0; p < PRODUCTS; ++p) {
      const int e = p / (TN * TM), i = p / TM % TN, j = p % TM;
      acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[i][e], f[TN + j][e], acc[i][j], 0, 0, 0);
      if (p < ops) op(p);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int p = PRODUCTS; p < ops; ++p) op(p);
  };

#pragma unroll
  for (int n = 0; n < PIECES; ++n) load(n, k_begin);
  if (k_begin + BK > k_end) clear_beyond(k_begin);
#pragma unroll
  for (int n = 0; n < PIECES; ++n) write(n, 0);
#pragma unroll
  for (int n = 0; n < PIECES; ++n) load(n, k_begin + BK);
  lds_barrier();
#pragma unroll
  for (int n = 0; n < READS; ++n) read(f0, n, 0, 0);
  // Behind the first half's products: the reads for the second half, the next stage into the other buffer (whose last reads
  // were ahead of the last barrier), the loads of the stage after it; behind the second half's: the next stage's first reads.
  int cur = 0;
  for (int k0 = k_begin; k0 < k_end; k0 += BK) {
    if (k0 + 2 * BK > k_end) clear_beyond(k0 + BK);
    products(f0, READS + 2 * PIECES, [&](int n) {
      if (n < READS) read(f1, n, cur, 16);
      else if (n < READS + PIECES) write(n - READS, cur ^ 1);
      else load(n - READS - PIECES, k0 + 2 * BK);
    });
    lds_barrier();
    products(f1, READS, [&](int n) { read(f0, n, cur ^ 1, 0); });
    cur ^= 1;
  }
  __syncthreads();

  // The outputs go through LDS (the last barrier has passed): 16-byte pieces of a token's row, and the epilogue's functions stand
  // in the code for four elements and not for a lane's 16 TM TN / 4 (which took 16,000 instructions).
  auto Ys = reinterpret_cast<float (*)[YROW]>(lds);
#pragma unroll
  for (int j = 0; j < TM; ++j)
#pragma unroll
    for (int i = 0; i < TN; ++i) *reinterpret_cast<f32x4*>(&Ys[(wm * TM + j) * 16 + c][(wn * TN + i) * 16 + g * 4]) = acc[i][j];
  __syncthreads();
  TO* __restrict__ y = Y + (size_t)blockIdx.y * M * N;
  const int pieces = geglu ? BN / 8 : BN / 4;                 // of a row
#pragma unroll 1
  for (int id = tid; id < BM * pieces; id += 256) {
    const int r = id / pieces, q = (id % pieces) * 4, m = m0 + r, n = n0 + q;
    if (m >= M || n >= N) continue;
    f32x4 v;
    if (geglu) {
      const float* p = &Ys[r][q / (8 * TN) * 16 * TN + q % (8 * TN)];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gated_act(p[e], p[8 * TN + e], param, full);
    } else {
      v = *reinterpret_cast<const f32x4*>(&Ys[r][q]);
      if (epi == ALICE_EPI_SOFTCAP) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = unary_act(v[e], param, full);
      }
    }
    TO* dst = y + (size_t)m * N + n;
    if constexpr (sizeof(TO) == 4) {
      if (wide) {                                             // rows of whole, aligned pieces
        *reinterpret_cast<f32x4*>(dst) = v;
        continue;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) store_f32(dst, e, v[e]);
  }
}

// Tile and number of slices for a product.  Estimated microseconds: 8, and for every block that a CU gets its products at a CU's
// rate (TFLOP/s, measured with 1 to 8 blocks a CU and K 576 and 2,304) and 1 more; not less than reading W takes; slices cost
// writing and reading their sums.  The rates are close, so what decides is how evenly the tiles fill the CUs: 500 tokens with
// GeGLU on 18,432 x 2,304 rows are 1,536 tiles of 64 x 96, six a CU, 350 us; 576 of 128 x 128, three for some, 504.  (A CU holds
// two blocks of 128 x 128: a third one runs alone.)
struct Tile {
  int bm, bn;
  float rate;
};
constexpr Tile TILES[] = {{128, 128, 0.510f}, {128, 64, 0.500f}, {64, 96, 0.492f}, {64, 64, 0.490f}, {32, 64, 0.460f}};
struct Plan {
  int tile, split;
  float us;
};
Plan plan_mfma32(int M, int N, int K, bool geglu, int min_split, int max_split) {
  Plan best{3, min_split, 1e30f};
  for (int i = 0; i < (int)(sizeof(TILES) / sizeof(TILES[0])); ++i) {
    const Tile& t = TILES[i];
    const int mt = ceil_div(M, t.bm), nt = ceil_div(N, geglu ? t.bn / 2 : t.bn);
    for (int s = min_split; s <= max_split; ++s) {
      const int ks = ceil_div(ceil_div(K, s), BK) * BK;
      if (s > 1 && (ks < 256 || (long)ks * (s - 1) >= K)) continue;      // no slice without elements
      const int blocks = ceil_div((long)mt * nt * s, 256);
      const float alone = i == 0 && blocks > 1 && blocks % 2 ? 0.5f : 0.f;
      float us = 8.f + (blocks + alone) * (2.f * t.bm * t.bn * (float)ks / (1e6f * t.rate) + 1.f);
      us = fmaxf(us, (geglu ? 2.f : 1.f) * N * (float)K * 4.f / 4.5e6f);
      if (s > 1) us += 2.f * s * (float)M * N * 4.f / 4.0e6f;
      if (us < best.us) best = Plan{i, s, us};
    }
  }
  return best;
}
constexpr int MAX_SPLIT = 8;
// The number of tokens that the slices are planned for.  Their number decides in which order the sums of an output are added, and an
// output must not depend on how a step is launched: steps of single tokens are captured with their number rounded up to a power of two
// up to 64 and to a multiple of 64 beyond, short prompts to a multiple of 16.  Any number of tokens here gives what either rounding of it
// gives.  (Numbers of tokens on two sides of a multiple of 64 may add in another order: rounding, no more.)
int planned_tokens(int M) { return M <= 32 ? 32 : ceil_div(M, 64) * 64; }
static_assert(THIRDS_BK == BK, "both ways cut the inner dimension into the same slices");
// Whether a product goes in thirds on the bfloat16 instruction: where that is estimated to be faster.  Both estimates are within a tenth of
// what measures, and where they are that close either way will do.  (2B shape, the 32-bit instruction and thirds: 500 tokens gate and up 356
// and 244 us, down 177 and 121, q, k, v 84 and 61, output 40 and 34; 128 tokens 105 and 75, 87 and 42, 32 and 38 (stays), 16 and 15; 32 tokens
// 48 and 46, 28 and 23, 31 and 30, 8 and 8.)
bool in_thirds(const ThirdsPlan& t, const Plan& p) { return t.us < p.us; }

// Elements a slice of up to 16 tokens' products.
int slice_of(int K, int split) { return ceil_div(ceil_div(K, split), 128) * 128; }

// 2 to 16 tokens: the tokens are the columns of the same matrix instruction, the rows of W its rows.  A block takes 16 R rows
// (with GeGLU 8 gate rows and the up rows of the same outputs: twice the blocks of 16 and 16, and the registers for more of
// them a CU), its NW waves every NW-th chunk of 32 inner elements of
// its slice; their sums meet in LDS.  W goes straight from memory into the instruction's operand, 128 bytes of a row a
// chunk, the next two chunks on their way while two are multiplied; the tokens' elements come through the L1.  A token's
// result depends on no other token, nor on how many there are.  (The rows that this kernel takes are those that few_by_fours() does not,
// whatever the number of tokens.)
// WHOLE: rows of whole, aligned units of eight elements.  Else (any K, any address) the same loads without an alignment, and the
// elements behind the last whole chunk one by one, by the wave whose turn it is: 2,304 rows by 2,305 at 4 tokens 9.0 us (by 2,304
// 9.1; on the tile of 64 tokens 71).
//
// What bounds it: reading W, in pieces of 128 bytes of a row.  With weights that no cache holds, at 4 tokens: 2,304 rows by 2,048 in eight
// slices 7.0 us; the rows that the kernels below take now: gate and up of the 2B shape (170 MB) 37.4, 4.5 TB/s, the output head (2.36 GB) 400, 5.9.
template <bool ALIGNED>
__device__ __forceinline__ f32x4 piece(const float* __restrict__ p) {
  struct __attribute__((packed, aligned(4))) Any { f32x4 v; };
  if constexpr (ALIGNED) return *reinterpret_cast<const f32x4*>(p);
  return reinterpret_cast<const Any*>(p)->v;
}
template <bool ALIGNED>
__device__ __forceinline__ void load8(const float* __restrict__ p, f32x4* v) {
  v[0] = piece<ALIGNED>(p);
  v[1] = piece<ALIGNED>(p + 4);
}
template <bool ALIGNED>
__device__ __forceinline__ void load8(const bf16_t* __restrict__ p, f32x4* v) {
  struct __attribute__((packed, aligned(2))) Any { uint4 v; };
  uint4 w;
  if constexpr (ALIGNED) w = *reinterpret_cast<const uint4*>(p);
  else w = reinterpret_cast<const Any*>(p)->v;
  v[0] = f32x4{bf16_bits_to_f32(w.x & 0xffffu), bf16_bits_to_f32(w.x >> 16), bf16_bits_to_f32(w.y & 0xffffu), bf16_bits_to_f32(w.y >> 16)};
  v[1] = f32x4{bf16_bits_to_f32(w.z & 0xffffu), bf16_bits_to_f32(w.z >> 16), bf16_bits_to_f32(w.w & 0xffffu), bf16_bits_to_f32(w.w >> 16)};
}

template <typename TA, typename TW, typename TO, int R, int NW, bool WHOLE>
__global__ __launch_bounds__(64 * NW) void linear_rows_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TO* __restrict__ Y, int M,
                                                              int N, int K, int kslice, int epi, float param, int full) {
  constexpr int U = 2, TURN = NW * 32;                        // chunks a step; elements from one of a wave's chunks to its next
  __shared__ __align__(16) f32x4 red[NW][R][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, c = lane & 15, g = lane >> 4;
  const bool geglu = R == 1 && epi == ALICE_EPI_GEGLU;
  const int n0 = blockIdx.x * (geglu ? 8 : 16 * R);
  const int k_begin = blockIdx.y * kslice, k_end = min(K, k_begin + kslice);
  const int k_chunks = WHOLE ? K : K & ~31, k_stop = min(k_end, k_chunks);       // what is read in units of eight
  const TW* wrow[R];                                          // rows and tokens beyond the last are read as the last and not written
#pragma unroll
  for (int r = 0; r < R; ++r) wrow[r] = W + (size_t)(geglu ? (c >> 3) * N + min(n0 + (c & 7), N - 1) : min(n0 + r * 16 + c, N - 1)) * K;
  const TA* arow = A + (size_t)min(c, M - 1) * K;

  f32x4 acc[R][2];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r][0] = acc[r][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 w[U][R][2], x[U][2], wn[U][R][2], xn[U][2];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(k0 + u * TURN + g * 8, k_chunks - 8);         // stays inside the row
#pragma unroll
      for (int r = 0; r < R; ++r) load8<WHOLE>(wrow[r] + k, wn[u][r]);
      load8<WHOLE>(arow + k, xn[u]);
    }
  };
  auto multiply = [&](int u) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[r][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[u][r][i][e], x[u][i][e], acc[r][e & 1], 0, 0, 0);
  };
  int k0 = k_begin + wave * 32;
  if (k0 < k_stop) fetch(k0);
  for (; k0 < k_stop; k0 += U * TURN) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // beyond the slice's end: zeros on both sides
      const bool in = k0 + u * TURN + g * 8 < k_stop;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int r = 0; r < R; ++r) w[u][r][i][e] = in ? wn[u][r][i][e] : 0.f;
          x[u][i][e] = in ? xn[u][i][e] : 0.f;
        }
      }
    }
    if (k0 + U * TURN < k_stop) fetch(k0 + U * TURN);
#pragma unroll
    for (int u = 0; u < U; ++u) multiply(u);
  }
  if constexpr (!WHOLE) {
    if (k_begin <= k_chunks && k_chunks < k_end && wave == (k_chunks - k_begin) / 32 % NW) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int k = k_chunks + g * 8 + i * 4 + e, kc = min(k, K - 1);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            const float v = load_f32(wrow[r], kc);
            w[0][r][i][e] = k < K ? v : 0.f;
          }
          const float v = load_f32(arow, kc);
          x[0][i][e] = k < K ? v : 0.f;
        }
      multiply(0);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) red[wave][r][lane] = acc[r][0] + acc[r][1];
  __syncthreads();
  if (wave >= R) return;
  f32x4 v = (red[0][wave][lane] + red[1][wave][lane]) + (red[2][wave][lane] + red[3][wave][lane]), up;
#pragma unroll
  for (int j = 4; j < NW; j += 4)
    v += (red[j][wave][lane] + red[j + 1][wave][lane]) + (red[j + 2][wave][lane] + red[j + 3][wave][lane]);
  if (geglu) {                                                // the up rows of lane group g are with lane group g + 2
#pragma unroll
    for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(v[e], 32, 64);
    if (g >= 2) return;
  }
  if (c >= M) return;
  const int n = n0 + wave * 16 + g * 4;
  TO* y = Y + (size_t)blockIdx.y * M * N + (size_t)c * N;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (n + e >= (geglu ? min(N, n0 + 8) : N)) continue;
    float o = v[e];
    if (geglu) o = gated_act(o, up[e], param, full);
    if (epi == ALICE_EPI_SOFTCAP) o = unary_act(o, param, full);
    store_f32(y, n + e, o);
  }
}

// Slices of the inner dimension for 2 to 16 tokens: three blocks a CU where the rows alone do not give them, slices of at
// least 256 elements, and rather a few more slices than uneven ones.  At 4 tokens, on this kernel, 2,304 rows by 9,216 take 38 us whole,
// 24.1 in four slices, 21.8 in six; by 2,048: 10.6, 8.1, 8.5 in six (uneven), 7.2 in eight; 4,096 rows by 2,304: 14.1, 12.4 in four, 10.8
// in three.  On the kernels below, with weights that no cache holds: by 9,216 22.8 whole, 18.4 in four, 16.6 in six, 17.6 in eight; by 2,048 7.0
// whole, 6.2 in three, 6.8 in four: the eight of 256 elements that this rule plans, here, are 7.0.
int rows_split(int N, int K) {
  const int most = max(1, min(K / 256, 8)), least = min(ceil_div(768, ceil_div(N, 16)), most);
  for (int s = least; s <= most; ++s)
    if (K % (128 * s) == 0) return s;
  return least;
}

// One token: a wave a row of W (with GeGLU the gate row and the up row of an output) on FMAs, four elements a lane a step; the lanes'
// sums meet in a fixed tree.  Any K, any address, any slices.  No column of the matrix instruction is idle.  With weights that no cache holds:
// 3,584 rows by 4,096 14.1 us, 8,192 by 2,304 15.0 (5 TB/s); beyond some 80 MB four rows a wave are the faster (below): 18,432 by 2,304 with
// GeGLU 33.5 us, 256,000 by 2,304 382.
template <typename TA, typename TW, typename TO, bool GEGLU>
__global__ __launch_bounds__(256) void linear_single_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TO* __restrict__ Y, int N,
                                                            int K, int kslice, int epi, float param, int full) {
  constexpr int NR = GEGLU ? 2 : 1;
  const int lane = threadIdx.x & 63, n = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (n >= N) return;
  const int k_begin = blockIdx.y * kslice, k_end = min(K, k_begin + kslice);       // (a slice begins at a multiple of 128)
  float acc[NR];
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = 0.f;
  const int K4 = k_end & ~3;
  for (int k = k_begin + lane * 4; k < K4; k += 256) {
    float w[NR][4];
#pragma unroll
    for (int r = 0; r < NR; ++r)
#pragma unroll
      for (int e = 0; e < 4; ++e) w[r][e] = load_f32(W, (size_t)(n + r * N) * K + k + e);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float x = load_f32(A, k + e);
#pragma unroll
      for (int r = 0; r < NR; ++r) acc[r] = fmaf(w[r][e], x, acc[r]);
    }
  }
  if (k_begin < k_end && lane < k_end - K4) {                 // up to three elements behind the last whole group of four
    const int k = K4 + lane;
    const float x = load_f32(A, k);
#pragma unroll
    for (int r = 0; r < NR; ++r) acc[r] = fmaf(load_f32(W, (size_t)(n + r * N) * K + k), x, acc[r]);
  }
#pragma unroll
  for (int r = 0; r < NR; ++r) acc[r] = wave_sum(acc[r]);
  if (lane) return;
  float o = acc[0];
  if (GEGLU) o = gated_act(acc[0], acc[NR - 1], param, full);
  if (epi == ALICE_EPI_SOFTCAP) o = unary_act(o, param, full);
  store_f32(Y, (size_t)blockIdx.y * N + n, o);
}

template <typename TA, typename TW, typename TO>
int launch_single(const void* x, const void* w, void* y, int N, int K, int epi, float epi_param, int full, int split, hipStream_t stream) {
  const int kslice = slice_of(K, split);
  const dim3 grid(ceil_div(N, 4), split);
#define GO(GEGLU) linear_single_kernel<TA, TW, TO, GEGLU><<<grid, 256, 0, stream>>>((const TA*)x, (const TW*)w, (TO*)y, N, K, kslice, epi, epi_param, full)
  if (epi == ALICE_EPI_GEGLU) GO(true); else GO(false);
#undef GO
  ALICE_LAUNCH_CHECK();
  return 0;
}

// Up to 4 tokens on FMAs, where rows are whole units of four elements at aligned addresses: a wave takes four rows of W (with GeGLU
// the gate and up rows of two outputs), its lanes 1 KB of a row at a time, and every element that it reads serves all tokens, whose
// elements wait in LDS.  The matrix instruction above leaves 12 or more of its 16 columns idle at so few, and its operand order
// reads W in pieces of 128 bytes of a row; here a load is a whole kilobyte, with the streaming hint (gate and up 35.4 -> 33.7 us,
// the output head 394 -> 357; the 128-byte pieces get slower by it), and two of every row are on their way while two
// are multiplied.  The tokens' elements are asked for ahead of W's first (33.7 -> 30.2 us: a block's start is what its CU waits for).
// What bounds it: reading W, at 6.6 TB/s where it is long.  4 tokens, 2B shape, weights that no cache holds, matrix instruction and
// this: q, k, v 12.4 and 8.7 us, gate and up 37.4 and 29.5, down (six slices) 21.6 and 16.6, head 400 and 355 (the output projection
// goes in slices that are too short for it); more tokens in one block gain nothing by it (eight: 42 us for gate and up, 468 for the head),
// but four a block do where there are few blocks.
// Which products a token's sum adds, and in which order, depends on K and the slices alone: a lane's elements in their order, then
// the lanes over the distances 32, 16 .. 1.  That is the order of the kernel for one token as well, and of those for 5 to 16 tokens below
// (the same bits).
constexpr int FEW_MT = 4, FEW_R = 4, FEW_SEG = 256, FEW_KC = 2560;       // tokens, rows a wave, elements a step, elements of a token that a block keeps (whole steps of two)

template <typename T> __device__ __forceinline__ f32x4 load_four(const T* p);
template <> __device__ __forceinline__ f32x4 load_four<float>(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
template <> __device__ __forceinline__ f32x4 load_four<bf16_t>(const bf16_t* p) {
  const uint2 v = *reinterpret_cast<const uint2*>(p);
  return f32x4{bf16_bits_to_f32(v.x & 0xffffu), bf16_bits_to_f32(v.x >> 16), bf16_bits_to_f32(v.y & 0xffffu), bf16_bits_to_f32(v.y >> 16)};
}

__device__ __forceinline__ f32x4 load_once(const float* p) { return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p)); }
__device__ __forceinline__ f32x4 load_once(const bf16_t* p) { return load_four(p); }

// V sums over the 64 lanes at once: a step over lane distance d adds the partner's value, and while several values are left each half of
// the lanes goes on with half of them.  Lane l ends with the sums of values first + 0 .. V / 8 - 1, first = V/2 (l / 32) + V/4 (l / 16 % 2)
// + V/8 (l / 8 % 2).
template <int V>
__device__ __forceinline__ int sums_by_lane(float (&v)[V], int lane) {
  static_assert(V >= 8, "three halvings");
  auto bits = [](float x) { return __float_as_uint(x); };
#pragma unroll
  for (int i = 0; i < V / 2; ++i) {
    auto p = __builtin_amdgcn_permlane32_swap(bits(v[i]), bits(v[i + V / 2]), false, false);
    v[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
#pragma unroll
  for (int i = 0; i < V / 4; ++i) {
    auto p = __builtin_amdgcn_permlane16_swap(bits(v[i]), bits(v[i + V / 4]), false, false);
    v[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
#pragma unroll
  for (int i = 0; i < V / 8; ++i) {
    const bool upper = lane & 8;
    const float give = upper ? v[i] : v[i + V / 8], keep = upper ? v[i + V / 8] : v[i];
    v[i] = keep + __uint_as_float(dpp_move<DPP_ROR8>(bits(give)));
  }
#pragma unroll
  for (int i = 0; i < V / 8; ++i) {
    v[i] += __uint_as_float(dpp_move<0x1B>(dpp_move<0x141>(bits(v[i]))));    // lane ^ 4: mirrored in its eight, then in its four
    v[i] += __uint_as_float(dpp_move<DPP_XOR2>(bits(v[i])));
    v[i] += __uint_as_float(dpp_move<DPP_XOR1>(bits(v[i])));
  }
  return (lane >> 5) * (V / 2) + ((lane >> 4) & 1) * (V / 4) + ((lane >> 3) & 1) * (V / 8);
}

template <typename TA, typename TW, typename TO, bool GEGLU>
__global__ __launch_bounds__(256) void linear_few_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TO* __restrict__ Y, int M, int N,
                                                         int K, int kslice, int kc, int epi, float param, int full) {
  constexpr int MT = FEW_MT, R = FEW_R, U = 2, P = (FEW_KC + 1023) / 1024;   // P: rounds of the block over a chunk's elements
  extern __shared__ __align__(16) float xs[];                 // [MT][kc]: the tokens' elements of a chunk, zeros behind the slice
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int m0 = blockIdx.z * MT;                             // this block's tokens are m0 .. m0 + MT - 1, as far as there are so many
  const int n0 = (blockIdx.x * 4 + wave) * (GEGLU ? R / 2 : R);
  const int k_begin = blockIdx.y * kslice, k_end = min(K, k_begin + kslice);
  const TW* wrow[R];                                          // rows beyond the last are read as the last and not written
#pragma unroll
  for (int r = 0; r < R; ++r) wrow[r] = W + (size_t)(GEGLU ? (r & 1) * N + min(n0 + (r >> 1), N - 1) : min(n0 + r, N - 1)) * K;
  float acc[MT * R];
#pragma unroll
  for (int i = 0; i < MT * R; ++i) acc[i] = 0.f;
  f32x4 w[U][R];
  auto fetch = [&](int k, f32x4 (&to)[R]) {                   // unconditional: behind the slice its last four elements
#pragma unroll
    for (int r = 0; r < R; ++r) to[r] = load_once(wrow[r] + min(k + lane * 4, k_end - 4));
  };
  // The tokens' elements of a chunk through registers into LDS: the first chunk's are asked for before W's first, which are on
  // their way while the block meets.
  f32x4 v[P][MT];
  auto load_x = [&](int c0) {
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int m = 0; m < MT; ++m) v[p][m] = load_four(A + (size_t)min(m0 + m, M - 1) * K + min(c0 + p * 1024 + tid * 4, k_end - 4));
  };
  load_x(k_begin);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) fetch(k_begin + u * FEW_SEG, w[u]);
  __builtin_amdgcn_sched_barrier(0);
  for (int c0 = k_begin; c0 < k_end; c0 += kc) {
    if (c0 > k_begin) {
      load_x(c0);
      lds_barrier();
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int k = p * 1024 + tid * 4;
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (k < kc) *reinterpret_cast<f32x4*>(xs + m * kc + k) = c0 + k < k_end ? v[p][m] : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    lds_barrier();
    const int stop = min(k_end - c0, kc);
    for (int s = 0; s < stop; s += U * FEW_SEG) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = s + u * FEW_SEG;
        if (k < stop) {                                       // (the same for the whole block)
          if (k + FEW_SEG > stop) {                           // what was read again behind the end: zeros
#pragma unroll
            for (int r = 0; r < R; ++r) w[u][r] = k + lane * 4 < stop ? w[u][r] : f32x4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(xs + m * kc + k + lane * 4);
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int r = 0; r < R; ++r) acc[m * R + r] = fmaf(w[u][r][e], x[e], acc[m * R + r]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch(c0 + k + U * FEW_SEG, w[u]);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  const int first = sums_by_lane<MT * R>(acc, lane);
  if (lane & 7) return;
  TO* y = Y + (size_t)blockIdx.y * M * N;
#pragma unroll
  for (int i = 0; i < MT * R / 8; i += GEGLU ? 2 : 1) {
    const int m = m0 + (first + i) / R, r = (first + i) % R, n = n0 + (GEGLU ? r >> 1 : r);
    if (m >= M || n >= N) continue;
    float o = acc[i];
    if (GEGLU) o = gated_act(acc[i], acc[i + 1], param, full);
    if (epi == ALICE_EPI_SOFTCAP) o = unary_act(o, param, full);
    store_f32(y, (size_t)m * N + n, o);
  }
}

template <typename TA, typename TW, typename TO>
int launch_few(const void* x, const void* w, void* y, int M, int N, int K, int epi, float epi_param, int full, int split, hipStream_t stream) {
  const int kslice = slice_of(K, split);
  const int kc = min(ceil_div(kslice, FEW_SEG) * FEW_SEG, FEW_KC);
  const dim3 grid(ceil_div(N, (epi == ALICE_EPI_GEGLU ? 2 : 4) * FEW_R), split, ceil_div(M, FEW_MT));
  const size_t lds = (size_t)FEW_MT * kc * sizeof(float);
#define GO(GEGLU) linear_few_kernel<TA, TW, TO, GEGLU><<<grid, 256, lds, stream>>>((const TA*)x, (const TW*)w, (TO*)y, M, N, K, kslice, kc, epi, epi_param, full)
  if (epi == ALICE_EPI_GEGLU) GO(true); else GO(false);
#undef GO
  ALICE_LAUNCH_CHECK();
  return 0;
}

// 5 to 16 tokens where the kernel above takes up to 4: the same sums, bit for bit, on the matrix instruction for 16 blocks of 4 rows by
// 4 tokens (v_mfma_f32_4x4x1_16b_f32: one 32-bit FMA an element a block, none of it idle).  So a token's result does not hang on how
// many others its step has, up to 16 of them, nor on the rounded size of a captured step.  A lane holds four elements of row lane % 4 for
// block lane / 4: block b of the 64 elements number a of every 256 adds what lane 16 a + b adds there.
// Two kernels share that, and where few blocks are all there is the kernel above takes four tokens a block (launch_more() chooses).
// Against the instruction for 16 columns, which adds in another order (rows x elements, slices; us at 8 and 16 tokens, before and after):
// 256,000 x 2,304: 402 -> 385 and 463 -> 457; 2,304 x 9,216, 6: 22.9 -> 18.9 and 27.4 -> 21.9; 28,672 x 3,584 with GeGLU 83 -> 76 and
// 101 -> 84; 18,432 x 2,304 with GeGLU 39.7 -> 38.7 and 47.9 -> 48.7; 4,096 x 2,304: 12.7 -> 10.2 and 12.9 -> 13.9; 2,048 x 2,048: 10.7 -> 6.7
// and 11.1 -> 8.7; 65,536 x 1,024: 53.2 -> 55.1 and 59.6 -> 62.5.  The error against 64 bits falls from 3e-7 to 1.3e-7 of the result.
template <typename T> struct Four;
template <> struct Four<float> { typedef f32x4 type; };
template <> struct Four<bf16_t> { typedef uint2 type; };
__device__ __forceinline__ f32x4 four_f32(const f32x4& v) { return v; }
__device__ __forceinline__ f32x4 four_f32(const uint2& v) {
  return f32x4{bf16_bits_to_f32(v.x & 0xffffu), bf16_bits_to_f32(v.x >> 16), bf16_bits_to_f32(v.y & 0xffffu), bf16_bits_to_f32(v.y >> 16)};
}
__device__ __forceinline__ f32x4 four_once(const float* p) { return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p)); }
__device__ __forceinline__ uint2 four_once(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }

// The sum of a tile over the accumulators a and blocks b, in the order of the kernel above (its lanes' distances 32 and 16: a; 8, 4, 2, 1: b), and
// its outputs: `v` holds rows n_first .. + 3 (with GeGLU the gate rows of outputs n_first and n_first + 1, then their up rows) of token
// m_first + lane % 4.
template <typename TO, bool GEGLU>
__device__ __forceinline__ void finish_tile(f32x4 v, TO* __restrict__ y, int m_first, int n_first, int M, int N, int epi, float param, int full, int lane) {
  auto bits = [](float f) { return __float_as_uint(f); };
  float h[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const auto p = __builtin_amdgcn_permlane32_swap(bits(v[i]), bits(v[i + 2]), false, false);
    h[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
  }
  const auto p = __builtin_amdgcn_permlane16_swap(bits(h[0]), bits(h[1]), false, false);
  float o = __uint_as_float(p[0]) + __uint_as_float(p[1]);                  // row lane / 16 of the four
  o += __uint_as_float(dpp_move<DPP_ROR8>(bits(o)));
  o += __uint_as_float(dpp_move<0x1B>(dpp_move<0x141>(bits(o))));           // lane ^ 4
  const int m = m_first + (lane & 3);
  int n = n_first + (lane >> 4);
  bool mine = (lane & 12) == 0 && m < M;
  if (GEGLU) {
    const auto q = __builtin_amdgcn_permlane32_swap(bits(o), bits(o), false, false);
    o = gated_act(o, __uint_as_float(q[1]), param, full);
    n = n_first + ((lane >> 4) & 1);
    mine = mine && lane < 32;
  }
  if (epi == ALICE_EPI_SOFTCAP) o = unary_act(o, param, full);
  if (mine && n < N) store_f32(y, (size_t)m * N + n, o);
}

// Many blocks: a wave takes 8 rows of W (with GeGLU the gate and up rows of 4 outputs), four steps of 64 elements on their way, an
// accumulator set for each a; the tokens' elements wait in LDS, four tokens' pieces side by side, the next chunk's in registers.
// What bounds it: reading W, in pieces of 256 bytes of four rows with neighbouring lanes in different rows (5.2 to 6.2 TB/s).
// NT threads a block: with 512 fewer blocks ask for the tokens' elements (256,000 x 2,304 at 16 tokens 473 -> 450).
constexpr int some_chunk(int MT) { return MT == 8 ? 768 : 512; }       // elements of a token that a block keeps

template <typename TA, typename TW, typename TO, bool GEGLU, int MT, int NT>
__global__ __launch_bounds__(NT, MT == 8 ? 3 : 2) void linear_some_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TO* __restrict__ Y, int M,
                                                                          int N, int K, int kslice, int epi, float param, int full) {
  constexpr int NX = MT / 4, R = 2, U = 4, SEG = 64, KC = some_chunk(MT), P = KC / NT;     // a round of the block: NT elements of four tokens
  static_assert(KC % NT == 0 && KC % (U * SEG) == 0, "whole rounds, whole turns");
  typedef typename Four<TA>::type X4;
  typedef typename Four<TW>::type W4;
  __shared__ __align__(16) f32x4 xs[NX * KC];                 // [token / 4][element / 4][token % 4]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, i4 = lane & 3, blk = lane >> 2;
  const int n0 = (blockIdx.x * (NT / 64) + wave) * (GEGLU ? 2 * R : 4 * R);
  const int k_begin = blockIdx.y * kslice, k_end = min(K, k_begin + kslice);
  const TW* wrow[R];                                          // rows beyond the last are read as the last and not written
#pragma unroll
  for (int r = 0; r < R; ++r)
    wrow[r] = W + (size_t)(GEGLU ? (i4 >> 1) * N + min(n0 + 2 * r + (i4 & 1), N - 1) : min(n0 + 4 * r + i4, N - 1)) * K;
  f32x4 acc[4][R][NX];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int x = 0; x < NX; ++x) acc[a][r][x] = f32x4{0.f, 0.f, 0.f, 0.f};
  W4 w[U][R];
  X4 v[NX][P];
  auto fetch = [&](int u, int k) {                            // unconditional: behind the slice its last four elements
    const int at = min(k + blk * 4, k_end - 4);
#pragma unroll
    for (int r = 0; r < R; ++r) w[u][r] = four_once(wrow[r] + at);
  };
  auto load_x = [&](int c0) {
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int p = 0; p < P; ++p)
        v[x][p] = *reinterpret_cast<const X4*>(A + (size_t)min(4 * x + (tid & 3), M - 1) * K + min(c0 + p * NT + (tid >> 2) * 4, k_end - 4));
  };
  load_x(k_begin);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < U; ++u) fetch(u, k_begin + u * SEG);
  __builtin_amdgcn_sched_barrier(0);
  for (int c0 = k_begin; c0 < k_end; c0 += KC) {
    if (c0 > k_begin) lds_barrier();
#pragma unroll
    for (int x = 0; x < NX; ++x)
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int k = p * NT + (tid >> 2) * 4;
        xs[x * KC + k + (tid & 3)] = c0 + k < k_end ? four_f32(v[x][p]) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
    if (c0 + KC < k_end) load_x(c0 + KC);
    lds_barrier();
    const int stop = min(k_end - c0, KC);
    for (int s = 0; s < stop; s += U * SEG) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = s + u * SEG;
        if (k < stop) {                                       // (the same for the whole block)
          f32x4 wf[R];
#pragma unroll
          for (int r = 0; r < R; ++r) wf[r] = four_f32(w[u][r]);
          if (k + SEG > stop) {                               // what was read again behind the end: zeros
#pragma unroll
            for (int r = 0; r < R; ++r) wf[r] = k + blk * 4 < stop ? wf[r] : f32x4{0.f, 0.f, 0.f, 0.f};
          }
#pragma unroll
          for (int x = 0; x < NX; ++x) {
            const f32x4 xv = xs[x * KC + k + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int r = 0; r < R; ++r) acc[u][r][x] = __builtin_amdgcn_mfma_f32_4x4x1f32(wf[r][e], xv[e], acc[u][r][x], 0, 0, 0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch(u, c0 + k + U * SEG);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  TO* y = Y + (size_t)blockIdx.y * M * N;
#pragma unroll
  for (int x = 0; x < NX; ++x)
#pragma unroll
    for (int r = 0; r < R; ++r)
      finish_tile<TO, GEGLU>((acc[0][r][x] + acc[2][r][x]) + (acc[1][r][x] + acc[3][r][x]), y, 4 * x, n0 + (GEGLU ? 2 : 4) * r, M, N, epi, param, full, lane);
}

// Fewer blocks: the four waves share 16 rows of W (with GeGLU the gate and up rows of 8 outputs), a wave the 64 elements number a of every
// 256; W and the tokens' elements come straight from memory, two steps of each, and the accumulators meet in LDS.  4,096 x 2,304 at 8 and 16 tokens
// 10.2 and 13.7 us, 13.7 and 17.1 by the kernel above; 2,304 x 9,216 whole 27 and 36 (44 and 54); with three blocks a CU and more it is the slower.
template <typename TA, typename TW, typename TO, bool GEGLU, int MT>
__global__ __launch_bounds__(256, MT == 8 ? 4 : 3) void linear_quarters_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TO* __restrict__ Y, int M,
                                                                               int N, int K, int kslice, int epi, float param, int full) {
  constexpr int NX = MT / 4, R = 4, U = 2, TURN = 8;          // TURN: tiles that meet at a time
  static_assert(R * NX % TURN == 0, "whole turns");
  typedef typename Four<TA>::type X4;
  typedef typename Four<TW>::type W4;
  __shared__ __align__(16) f32x4 red[4][TURN][64];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), i4 = lane & 3, blk = lane >> 2;
  const int n0 = blockIdx.x * (GEGLU ? 2 * R : 4 * R);
  const int k_begin = blockIdx.y * kslice, k_end = min(K, k_begin + kslice);
  const TW* wrow[R];                                          // rows and tokens beyond the last are read as the last and not written
#pragma unroll
  for (int r = 0; r < R; ++r)
    wrow[r] = W + (size_t)(GEGLU ? (i4 >> 1) * N + min(n0 + 2 * r + (i4 & 1), N - 1) : min(n0 + 4 * r + i4, N - 1)) * K;
  const TA* xrow[NX];
#pragma unroll
  for (int x = 0; x < NX; ++x) xrow[x] = A + (size_t)min(4 * x + i4, M - 1) * K;
  f32x4 acc[R][NX];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int x = 0; x < NX; ++x) acc[r][x] = f32x4{0.f, 0.f, 0.f, 0.f};
  W4 w[U][R];
  X4 v[U][NX];
  auto fetch = [&](int u, int k) {                            // unconditional: behind the slice its last four elements
    const int at = min(k + blk * 4, k_end - 4);
#pragma unroll
    for (int x = 0; x < NX; ++x) v[u][x] = *reinterpret_cast<const X4*>(xrow[x] + at);
#pragma unroll
    for (int r = 0; r < R; ++r) w[u][r] = four_once(wrow[r] + at);
  };
  const int k0 = k_begin + wave * 64;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    fetch(u, k0 + u * 256);
    __builtin_amdgcn_sched_barrier(0);
  }
  for (int s = k0; s < k_end; s += U * 256) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = s + u * 256;
      if (k < k_end) {                                        // (the same for the whole wave)
        f32x4 wf[R], xf[NX];
#pragma unroll
        for (int r = 0; r < R; ++r) wf[r] = four_f32(w[u][r]);
#pragma unroll
        for (int x = 0; x < NX; ++x) xf[x] = four_f32(v[u][x]);
        if (k + 64 > k_end) {                                 // what was read again behind the end: zeros on both sides
          const bool in = k + blk * 4 < k_end;
#pragma unroll
          for (int r = 0; r < R; ++r) wf[r] = in ? wf[r] : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int x = 0; x < NX; ++x) xf[x] = in ? xf[x] : f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int x = 0; x < NX; ++x)
#pragma unroll
            for (int r = 0; r < R; ++r) acc[r][x] = __builtin_amdgcn_mfma_f32_4x4x1f32(wf[r][e], xf[x][e], acc[r][x], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      fetch(u, k + U * 256);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  TO* y = Y + (size_t)blockIdx.y * M * N;
#pragma unroll
  for (int t0 = 0; t0 < R * NX; t0 += TURN) {
    if (t0 > 0) lds_barrier();
#pragma unroll
    for (int t = 0; t < TURN; ++t) red[wave][t][lane] = acc[(t0 + t) / NX][(t0 + t) % NX];
    lds_barrier();
    for (int t = wave; t < TURN; t += 4)
      finish_tile<TO, GEGLU>((red[0][t][lane] + red[2][t][lane]) + (red[1][t][lane] + red[3][t][lane]), y, (t0 + t) % NX * 4,
                             n0 + (GEGLU ? 2 : 4) * ((t0 + t) / NX), M, N, epi, param, full, lane);
  }
}

// The three ways give the same bits, so the rule may look at the number of tokens.  Blocks of 16 rows and four tokens that find a CU
// each, or two and a short way, go as up to four tokens do (1,024 x 2,048 at 16 tokens 6.2 us, 14.2 with 8 rows a wave; 2,048 x 2,048 at 16 8.7
// and 11.4 in quarters); up to 256 blocks of 16 rows in quarters; more with 8 rows a wave.  There, beyond 8 tokens, eight waves a block
// where their blocks fill one round of the CUs (216 blocks: 22.6 -> 21.5) or many with a long way (448: 87.6 -> 83.6; 151,936 x 1,024: 138.6, and 149.8
// with eight); not with a second round that is nearly empty (288: 48.7 -> 55.8), nor where half the CUs get none (108: 8.5 -> 12.3).
template <typename TA, typename TW, typename TO>
int launch_more(const void* x, const void* w, void* y, int M, int N, int K, int epi, float epi_param, int full, int split, hipStream_t stream) {
  const int kslice = slice_of(K, split), rows = epi == ALICE_EPI_GEGLU ? 2 * N : N;
  const int blocks16 = ceil_div(rows, 16) * split, by_four = blocks16 * ceil_div(M, FEW_MT), blocks64 = ceil_div(rows, 64) * split;
  if (by_four <= 256 || (by_four <= 512 && kslice <= 2048)) return launch_few<TA, TW, TO>(x, w, y, M, N, K, epi, epi_param, full, split, stream);
  const bool quarters = blocks16 <= 256, wide = M > 8 && ((blocks64 > 160 && blocks64 <= 256) || (blocks64 >= 400 && kslice >= 2048));
  const dim3 grid(ceil_div(rows, quarters ? 16 : wide ? 64 : 32), split);
#define GO3(NAME, THREADS, ...) NAME<TA, TW, TO, __VA_ARGS__><<<grid, THREADS, 0, stream>>>((const TA*)x, (const TW*)w, (TO*)y, M, N, K, kslice, epi, epi_param, full)
#define GO2(GEGLU)                                                           \
  do {                                                                       \
    if (quarters && M <= 8) GO3(linear_quarters_kernel, 256, GEGLU, 8);      \
    else if (quarters) GO3(linear_quarters_kernel, 256, GEGLU, 16);          \
    else if (M <= 8) GO3(linear_some_kernel, 256, GEGLU, 8, 256);            \
    else if (M <= 12 && !wide) GO3(linear_some_kernel, 256, GEGLU, 12, 256); \
    else if (M <= 12) GO3(linear_some_kernel, 512, GEGLU, 12, 512);          \
    else if (!wide) GO3(linear_some_kernel, 256, GEGLU, 16, 256);            \
    else GO3(linear_some_kernel, 512, GEGLU, 16, 512);                       \
  } while (0)
  if (epi == ALICE_EPI_GEGLU) GO2(true); else GO2(false);
#undef GO2
#undef GO3
  ALICE_LAUNCH_CHECK();
  return 0;
}

template <typename TA, typename TW, typename TO>
int launch_rows(const void* x, const void* w, void* y, int M, int N, int K, int epi, float epi_param, int full, int split,
                hipStream_t stream) {
  const int kslice = slice_of(K, split);
  const bool whole = K % 8 == 0 && K >= 32 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0;
  const int by = epi == ALICE_EPI_GEGLU ? 8 : (N >= 16384 ? 32 : 16);      // many rows: a token's elements serve 32 of them
  const dim3 grid(ceil_div(N, by), split);
  // Four waves a block, eight where there are few blocks with long rows (2,304 rows by 9,216 in one slice, 2 tokens: 23.5 us, 29.0 with
  // four; by 2,304 four are the better: 8.3 and 9.0).  A rule without the number of tokens: the sums are the same for all of them.
  const bool eight = by != 32 && (long)grid.x * split <= 256 && kslice >= 4096;
#define GO2(R, NW, WHOLE) linear_rows_kernel<TA, TW, TO, R, NW, WHOLE><<<grid, 64 * NW, 0, stream>>>((const TA*)x, (const TW*)w, (TO*)y, M, N, K, kslice, epi, epi_param, full)
#define GO(R, NW)                  \
  do {                             \
    if (whole) GO2(R, NW, true);   \
    else GO2(R, NW, false);        \
  } while (0)
  if (by == 32) GO(2, 4);
  else if (eight) GO(1, 8);
  else GO(1, 4);
#undef GO
#undef GO2
  ALICE_LAUNCH_CHECK();
  return 0;
}

template <typename TA, typename TW, typename TO>
int launch_tiled(const void* x, const void* w, void* y, int M, int N, int K, int epi, float epi_param, int full, int split,
                 hipStream_t stream) {
  const bool geglu = epi == ALICE_EPI_GEGLU;
  const int vec = K % 4 == 0 && ((uintptr_t)x & (4 * sizeof(TA) - 1)) == 0 && ((uintptr_t)w & (4 * sizeof(TW) - 1)) == 0;
  Plan p = plan_mfma32(planned_tokens(M), N, K, geglu, split, split);         // the tile that goes best with this many slices
  if constexpr (sizeof(TA) == 4 && sizeof(TW) == 4 && sizeof(TO) == 4) {
    const ThirdsPlan t = alice_linear_thirds_plan(planned_tokens(M), N, K, geglu, split, split);
    if (vec && in_thirds(t, p))
      return alice_linear_thirds((const float*)x, (const float*)w, (float*)y, M, N, K, epi, epi_param, full, t, stream);
  }
  if (split == 1) p = plan_mfma32(M, N, K, geglu, 1, 1);      // (no tile changes the order of the sums)
  if (!vec) p.tile = 3;                                       // one tile for rows that are no multiples of four elements
  const int kslice = ceil_div(ceil_div(K, split), BK) * BK;
  const int BM = TILES[p.tile].bm, cols = geglu ? TILES[p.tile].bn / 2 : TILES[p.tile].bn;
  const int mt = ceil_div(M, BM), nt = ceil_div(N, cols);
  ALICE_CHECK((long)mt * nt < (1l << 30), "linear: too many tiles for one launch");
  const int wide = N % 4 == 0 && ((uintptr_t)y & 15) == 0;
  dim3 grid(8 * ceil_div((long)mt * nt, 8), split);
#define GO(TM, TN, VEC) linear_mfma32_kernel<TA, TW, TO, TM, TN, VEC><<<grid, 256, 0, stream>>>((const TA*)x, (const TW*)w, (TO*)y, M, N, K, kslice, mt, nt, epi, epi_param, full, wide)
  if (!vec) GO(2, 2, false);
  else if (p.tile == 0) GO(4, 4, true);
  else if (p.tile == 1) GO(4, 2, true);
  else if (p.tile == 2) GO(2, 3, true);
  else if (p.tile == 3) GO(2, 2, true);
  else GO(1, 2, true);
#undef GO
  ALICE_LAUNCH_CHECK();
  return 0;
}

}  // namespace

// Whether up to 4 tokens go on FMAs (and up to 16 as those do), by the inner dimension: rows of whole units of four elements, long enough that the
// block's start does not outweigh them (65,536 rows by 256: 22.7 us, 16.2 on the matrix instruction; by 1,024 and more it is faster), and
// slices that are (of 256 elements: 8.2 us, 7.2 on the matrix instruction).  The rule of the slices and that of the launch ask here.
static bool few_by_length(int K, int split) { return K % 4 == 0 && K >= 1024 && (split == 1 || slice_of(K, split) >= 512); }
// And by the operands: at addresses of such units.
static bool few_by_fours(const void* x, int x_dtype, const void* w, int w_dtype, int K, int split) {
  auto unit = [](int dtype) { return dtype == DT_F32 ? 15u : 7u; };
  return few_by_length(K, split) && ((uintptr_t)x & unit(x_dtype)) == 0 && ((uintptr_t)w & unit(w_dtype)) == 0;
}

// Slices for one token: W is read at 6.6 TB/s with three blocks a CU, at three quarters of that with few; the busiest CU reads
// its blocks' rows at 40 GB/s or less; a slice more costs the add behind it 0.2 us.  (Planned and measured, weights that no cache holds:
// 2,304 rows by 2,048 whole, 7.2 us, 6.2 and 0.6 for the add in three; by 9,216 in 6, 16.8, 24.5 whole; 3,584 by 14,336 in 4, 35.3, 39.2 whole;
// 8,192 by 3,584 in 2, 21.8, 20.7 whole.)
static int single_split(int N, int K) {
  const int blocks = ceil_div(N, 4 * FEW_R);
  int best = 1;
  float best_us = 1e30f;
  for (int s = 1; s <= MAX_SPLIT; ++s) {
    const int ks = slice_of(K, s);
    if (s > 1 && (!few_by_length(K, s) || (long)ks * (s - 1) >= K)) continue;
    const float full = fminf(1.f, 0.75f + 0.25f * blocks * s / 768.f);
    const float us = fmaxf((float)N * K * 4e-6f / (6.6f * full), ceil_div((long)blocks * s, 256) * (float)ks * 64.f / 40e3f) + 0.2f * s;
    if (us < best_us) { best_us = us; best = s; }
  }
  return best;
}

// Into how many slices of the inner dimension a product without an epilogue is best cut (for 2 to 16 tokens one
// number, whatever captured steps round theirs to).
// floats: both operands are float32.  Where one is bfloat16 or starts on no 16 bytes the product stays with the 32-bit instruction, and
// with the slices of its own plan, except that the plan's cost is too low for blocks that are alone on a CU: up to 128 tokens, and where
// it would take one slice, the thirds' number is the better one.  (Product and the norm that reads the slices, thirds' against own number,
// float32 tokens by bfloat16 weights, 18 shapes of 2,048 x 2,048 to 3,584 x 14,336 at 17 to 2,000 tokens: 17 tokens by 3,584 x 14,336 62 and
// 94 us, 128 by 4,096 x 2,304 40 and 70, 256 by 4,096 x 2,304 in 4 and 1 slices 68 and 93, on the whole 1.24 times, at worst 6 % slower;
// the others 140 and 103 at 256 by 4,608 x 4,096, 224 and 210 at 500 by 2,304 x 9,216.  Bfloat16 tokens by float32 weights: 1.22 times.)
int alice_linear_split_hint_generic(int M, int N, int K, bool floats, bool aligned) {
  if (M == 1) return few_by_length(K, 1) ? single_split(N, K) : 1;
  if (M <= 16) return rows_split(N, K);
  const Plan p = plan_mfma32(planned_tokens(M), N, K, false, 1, MAX_SPLIT);
  if (!aligned || K % 4 != 0 || (!floats && planned_tokens(M) > 128 && p.split > 1)) return p.split;
  const ThirdsPlan t = alice_linear_thirds_plan(planned_tokens(M), N, K, false, 1, MAX_SPLIT);
  return in_thirds(t, p) ? t.split : p.split;
}

// The tile of a product of more than 16 tokens that goes in thirds, -1 if it goes on the 32-bit instruction (float32 and aligned operands).
extern "C" int alice_linear_thirds_tile(int M, int N, int K, int geglu, int split) {
  const ThirdsPlan t = alice_linear_thirds_plan(planned_tokens(M), N, K, geglu != 0, split, split);
  return M > 16 && K % 4 == 0 && in_thirds(t, plan_mfma32(planned_tokens(M), N, K, geglu != 0, split, split)) ? t.tile : -1;
}

int alice_linear_generic(const void* x, int x_dtype, const void* w, int w_dtype, void* y, int y_dtype,
                         int M, int N, int K, int epi, float epi_param, int split_k, int full_precision,
                         hipStream_t stream) {
  ALICE_CHECK(dtype_ok(x_dtype) && dtype_ok(w_dtype) && dtype_ok(y_dtype), "linear: unknown dtype");
  ALICE_CHECK(M >= 0 && N > 0 && K > 0, "linear: bad sizes M=%d N=%d K=%d", M, N, K);
  ALICE_CHECK(epi == ALICE_EPI_NONE || epi == ALICE_EPI_GEGLU || epi == ALICE_EPI_SOFTCAP,
              "linear: unknown epilogue %d", epi);
  ALICE_CHECK(epi != ALICE_EPI_SOFTCAP || epi_param > 0.f || epi_param == ALICE_UNARY_RELU2 || epi_param == ALICE_UNARY_SILU, "linear: softcap must be positive");
  ALICE_CHECK(split_k == 1 || (epi == ALICE_EPI_NONE && y_dtype == DT_F32), "linear: partial sums are float32 and take no epilogue");
  ALICE_CHECK(split_k >= 1 && split_k <= MAX_SPLIT, "linear: %d slices of the inner dimension are outside 1..%d", split_k, MAX_SPLIT);
  if (M == 0) return 0;
  int rc = 0;
  DISPATCH_DTYPE(x_dtype, TA, DISPATCH_DTYPE(w_dtype, TW, DISPATCH_DTYPE(y_dtype, TO, {
    const bool few = M <= 16 && few_by_fours(x, x_dtype, w, w_dtype, K, split_k);
    // One token: the same sums either way; a wave a row is the faster start (weights that no cache holds: 1,000 x 1,024 4.0 and 4.4 us, 3,584 x
    // 4,096 14.1 and 14.8), four rows a wave read longer matrices faster (8,192 x 3,584: 21.8 and 21.0, 12,288 x 2,304 23.0 and 20.1, gate and
    // up of the 2B shape 33.5 and 29.4); between 50 and 80 MB it goes either way by 4 %.
    const bool large = (size_t)N * K * sizeof(TW) * (epi == ALICE_EPI_GEGLU ? 2 : 1) >= ((size_t)80 << 20);
    // (In slices, which are planned for four rows a wave, a wave a row takes what that does not: operands at any address.)
    if (M == 1 && !(few && (large || split_k > 1))) rc = launch_single<TA, TW, TO>(x, w, y, N, K, epi, epi_param, full_precision, split_k, stream);
    else if (few && M <= FEW_MT) rc = launch_few<TA, TW, TO>(x, w, y, M, N, K, epi, epi_param, full_precision, split_k, stream);
    else if (few) rc = launch_more<TA, TW, TO>(x, w, y, M, N, K, epi, epi_param, full_precision, split_k, stream);
    else rc = M <= 16 ? launch_rows<TA, TW, TO>(x, w, y, M, N, K, epi, epi_param, full_precision, split_k, stream)
                      : launch_tiled<TA, TW, TO>(x, w, y, M, N, K, epi, epi_param, full_precision, split_k, stream);
  })));
  return rc;
}
