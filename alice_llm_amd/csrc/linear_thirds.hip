// 32-bit products of more than 16 tokens on the bfloat16 matrix instruction: y[M, N] = x[M, K] . W[N, K]^T, all float32
// (gguf.rs:4063-4074; GeGLU llama3.rs:14519-14534, softcap llama3.rs:14606-14611), with 32-bit sums and the precision of 32-bit
// products.
//
// A float32 is the sum of three bfloat16 numbers: each takes the next eight bits of the mantissa, rounded to nearest, and what it
// leaves is exact.  Of the nine products of two such sums the six largest are taken, every one of them exact in 32 bits; the three
// left out are at most 2^-24 of the whole product and of either sign.  The largest of the six goes into one float32 accumulator, the
// other five, 2^-6.5 of it at most, into a second one, and the two are added at the end: the largest product has 16 bits, which an
// accumulator of 24 takes without rounding until it is some hundred times the product, and what the second accumulator rounds is
// that much less.  Against 64 bits the error is 0.23 to 0.33 of the 32-bit instruction's (normal numbers, K 64 / 2,304 / 9,216 in three
// slices / 16,384: 0.48, 2.0, 2.3 and 5.7e-7 of the result's norm; 1.44, 8.6, 9.9 and 22.9), that of the 2B shape's logits after a
// prompt of 500 tokens 0.76e-6 instead of 2.8e-6.  With all six in one accumulator (in the same time) it was 0.46, 5.1, 6.0, 13.8 and
// 1.6e-6, and tokens of few elements, up to some 500 of 2,304, were up to 1.5 times as far off as on the 32-bit instruction, which
// rounds nothing where a product is zero: they have 1.03 of its error now with one to three elements, 0.54 with 16, 0.28 with 256.
#include "common.h"
#include "alice_hip.h"
#include "linear_thirds.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int BK = THIRDS_BK;                                 // inner elements a stage: one product's

__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// Eight elements of a row, times `sign` (1 or -1, with SIGNED), as three times eight bfloat16 numbers.
// top: the largest size met so far (of numbers: what is none leaves it, and every sum that it enters tells).
template <bool SIGNED>
__device__ __forceinline__ void thirds(const f32x4 (&v)[2], u32x4 (&p)[3], float& top, float sign = 1.f) {
  const uint32_t flip = (__float_as_uint(sign) >> 31) * 0x80008000u;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float x = v[i >> 1][(i & 1) * 2], y = v[i >> 1][(i & 1) * 2 + 1];
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(top) : "v"(x), "v"(y));      // (fmaxf quiets every operand first: three times the instructions)
#pragma unroll
    for (int t = 0; t < 3; ++t) {
      const uint32_t h = SIGNED && t == 0 ? pack_bf16x2(x, y) ^ flip : pack_bf16x2(x, y);
      p[t][i] = h;
      const float hx = __uint_as_float(h << 16), hy = __uint_as_float(h & 0xffff0000u);
      x = SIGNED && t == 0 ? fmaf(x, sign, -hx) : x - hx;
      y = SIGNED && t == 0 ? fmaf(y, sign, -hy) : y - hy;
    }
  }
}

// A block takes 16 TM tokens by 64 TN rows of W; its waves are two groups of four that share the inner dimension of the block's
// slice, first half and second half, 32 elements a stage each.  A wave takes all the tokens by 16 TN rows: its rows go from memory
// to its own registers and into thirds there, no other wave needs them; a group's tokens are split once, on their way into LDS, in
// the order in which the instruction takes them (every access one contiguous kilobyte of a wave), in two buffers with one barrier a
// stage.  A lane's eight elements of a stage are 4 g .. 4 g + 3 and 16 + 4 g .. 16 + 4 g + 3 on both sides (whole 64-byte pieces of
// a row a load).  The second group multiplies by the tokens' negative: the instruction adds by cutting off (towards minus infinity),
// and that would move every output of every token the same way (with one accumulator a third of the error of a product of 9,216
// elements was one vector common to all tokens, which no average over keys or layers removes: logits after prompts of 1,852 tokens
// were off by 2.6e-6 of their norm instead of 1.9e-6); the two groups' shifts cancel.  W is the first operand, so that a lane ends
// up with four neighbouring outputs of a token.  The groups' sums meet in LDS, on the way the outputs take to leave as 16-byte
// pieces of a token's row.  With GeGLU the first half of the block's rows are
// gate rows, the second half the up rows of the same outputs.  split: slices of the inner dimension, slice z to Y + z M N.
//
// What bounds it: the matrix instruction at the clock it runs at under this load.  500 tokens by 18,432 x 2,304 with GeGLU:
// 246 us (173 TFLOP/s of 32-bit products; 1.03 PFLOP/s of bfloat16 ones, where large library products reach 1.07 to 1.14), 183 with
// neither loads nor LDS nor splitting (with one accumulator); 356 on the 32-bit instruction.  Both operands through LDS, 128 x 128 to
// 256 x 144 a block: 247 to 330 us; products, splitting and loads interleaved by hand with the next stage's tokens read ahead: the
// same 275 as without for 64 x 128 a block; one group of four waves: 278.
template <int TM, int TN>
__global__ __launch_bounds__(512, 2) void linear_thirds_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ Y,
                                                               int M, int N, int K, int kslice, int split, int mt, int nt, int epi, float param,
                                                               int full, int wide) {
  constexpr int NW = 4, KG = 2, THREADS = 64 * NW * KG, BM = 16 * TM, BN = 16 * TN * NW, XJ = (TM + NW - 1) / NW;
  constexpr int YROW = BN + 4;
  constexpr int STAGE = 3 * TM * 64;                          // in units of 16 bytes
  extern __shared__ __align__(16) u32x4 lds[];
  __shared__ int again;
  __shared__ uint32_t xmask[KG][TM];                          // a token tile's tokens that marks() marks, a bit each
  const int tid = threadIdx.x, lane = tid & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6) % NW, group = __builtin_amdgcn_readfirstlane(tid >> 6) / NW;
  auto plane = [&](int buf, int t, int tile) { return lds + (group * 2 + buf) * STAGE + (t * TM + tile) * 64; };

  // tile and slice of this block: neighbours in m first, then in n, a run an XCD (blocks go to the 8 XCDs in turn)
  const int per = (mt * nt * split + 7) >> 3, item = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (item >= mt * nt * split) return;                        // the whole block: no barrier is missed
  const int slice = item / (mt * nt), tile = item % (mt * nt);
  const int m0 = (tile % mt) * BM, nb = tile / mt;
  const bool geglu = epi == ALICE_EPI_GEGLU;
  const int n0 = nb * (geglu ? BN / 2 : BN);
  const int s_begin = slice * kslice, s_end = min(K, s_begin + kslice);
  // a group's share of the slice; the groups take equally many stages, the last ones of zeros alone if need be
  const int span = ((s_end - s_begin + KG - 1) / KG + BK - 1) / BK * BK;
  const int k_begin = s_begin + group * span, k_stop = k_begin + span, k_end = min(s_end, k_stop);

  // rows and tokens beyond the last are read as the last and not written
  const float* wsrc[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    const int r = (wave * TN + i) * 16 + c;
    int row = min(n0 + r, N - 1);
    if (geglu) row = (r >= BN / 2) * N + min(n0 + r % (BN / 2), N - 1);
    wsrc[i] = W + (size_t)row * K;
  }
  const float* xsrc[XJ];
#pragma unroll
  for (int j = 0; j < XJ; ++j) xsrc[j] = A + (size_t)min(m0 + (wave + NW * j) * 16 + c, M - 1) * K;
  f32x4 wr[TN][2], xr[XJ][2];                                 // the stage on its way from memory
  auto load = [&](const float* p, f32x4 (&v)[2], int k0) {
    v[0] = *reinterpret_cast<const f32x4*>(p + min(k0 + g * 4, s_end - 4));
    v[1] = *reinterpret_cast<const f32x4*>(p + min(k0 + 16 + g * 4, s_end - 4));
  };
  auto clear_beyond = [&](f32x4 (&v)[2], int k0) {            // the last stage of a slice: nothing beyond its end
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const bool in = k0 + g * 4 + h * 16 < k_end;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[h][e] = in ? v[h][e] : 0.f;
    }
  };
  f32x4 acc[TN][TM], rest[TN][TM];                            // the sums of the largest of the six products, and of the other five
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = rest[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (tid == 0) again = 0;
  const float sign = group ? -1.f : 1.f;
  float xtop[XJ] = {}, wtop[TN] = {};                         // the largest sizes among the numbers of a row that this lane splits
  auto put = [&](int j, int buf) {
    u32x4 p[3];
    thirds<true>(xr[j], p, xtop[j], sign);
#pragma unroll
    for (int t = 0; t < 3; ++t) plane(buf, t, wave + NW * j)[lane] = p[t];
  };
  auto mine = [&](int j) { return TM % NW == 0 || wave + NW * j < TM; };
#pragma unroll
  for (int j = 0; j < XJ; ++j) load(xsrc[j], xr[j], k_begin);
#pragma unroll
  for (int i = 0; i < TN; ++i) load(wsrc[i], wr[i], k_begin);
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    clear_beyond(xr[j], k_begin);
    if (mine(j)) put(j, 0);
    load(xsrc[j], xr[j], k_begin + BK);
  }
  lds_barrier();
  int cur = 0;
  auto stage = [&](int k0, bool last) {
    u32x4 w[TN][3];
    auto split = [&](int i) {
      if (k0 + BK > k_end) clear_beyond(wr[i], k0);
      thirds<false>(wr[i], w[i], wtop[i]);
      if (!last) load(wsrc[i], wr[i], k0 + BK);
    };
    auto products = [&](int i, int wt, const u32x4 (&x)[TM], f32x4 (&sum)[TM]) {
#pragma unroll
      for (int j = 0; j < TM; ++j) sum[j] = mfma(w[i][wt], x[j], sum[j]);
    };
    u32x4 x[3][TM];
    auto fetch = [&](int t) {
#pragma unroll
      for (int j = 0; j < TM; ++j) x[t][j] = plane(cur, t, j)[lane];
    };
    // Blocks of 128 tokens take a part of the tokens at a time, or two accumulators do not fit beside them (245 registers, no time lost
    // at two row tiles a wave); the others all three, a row tile after the other (64 x 192 by parts: 246 to 262 us).
    if constexpr (TM < 8) {
#pragma unroll
      for (int t = 0; t < 3; ++t) fetch(t);
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        split(i);
        products(i, 2, x[0], rest[i]);
        products(i, 0, x[2], rest[i]);
        products(i, 1, x[1], rest[i]);
        products(i, 1, x[0], rest[i]);
        products(i, 0, x[1], rest[i]);
        products(i, 0, x[0], acc[i]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int t = 2; t >= 0; --t) {
        fetch(t);
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          if (t == 2) split(i);
#pragma unroll
          for (int wt = 2 - t; wt >= 0; --wt) products(i, wt, x[t], t + wt == 0 ? acc[i] : rest[i]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if (!last) {
#pragma unroll
      for (int j = 0; j < XJ; ++j) {
        if (k0 + 2 * BK > k_end) clear_beyond(xr[j], k0 + BK);
        if (mine(j)) put(j, cur ^ 1);
        load(xsrc[j], xr[j], k0 + 2 * BK);
      }
      lds_barrier();
      cur ^= 1;
    }
  };
  int k0 = k_begin;
  for (; k0 + BK < k_stop; k0 += BK) stage(k0, false);
  stage(k0, true);
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] += rest[i][j];

  // A number that is not finite, or that rounds to no finite bfloat16, has a remainder that is none, and every sum that it enters
  // is then none either.  What of a number is below the smallest normal bfloat16, 2^-126, may be lost: with 16,384 others of at most
  // 2^20 that is 2^-92 of a sum, less than its own rounding from 2^-64 on.  Smaller sums, those that are no finite numbers, and all
  // of a token or a row of W with a number larger than 2^20, are taken again by 32-bit products, and no others: what a token gets
  // hangs on its own numbers and W's, not on the tokens beside it.  Below 2^-134 all of a number is lost, and a sum of exactly zero
  // tells nothing (they come by chance too, one of some millions): tokens and rows of which all numbers are below 2^-102, but not all
  // zero, are taken again as well.  What stays is a zero instead of a sum below 2^-100, where a token's larger numbers meet nothing but
  // zeros of the row and what is left of it is all below 2^-134.
  // Marks of 16 rows, a bit each; lanes c + 16 g hold row c.
  auto marks = [](float top) {
    auto rows = [](uint64_t lanes) { return (uint32_t)(lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffffu; };
    return rows(__ballot(top > 0x1p20f)) | (rows(__ballot(top != 0.f)) & ~rows(__ballot(top >= 0x1p-102f)));
  };
  auto odd = [](float sum) {
    const float v = fabsf(sum);
    return (!(v >= 0x1p-64f) & (v != 0.f)) | !(v < INFINITY);
  };
  bool any = false;
#pragma unroll
  for (int j = 0; j < XJ; ++j) {
    const uint32_t mask = marks(xtop[j]);
    any = any | (mask != 0);
    if (mine(j) && lane == 0) xmask[group][wave + NW * j] = mask;
  }
  uint32_t wmask[TN];
#pragma unroll
  for (int i = 0; i < TN; ++i) {
    wmask[i] = marks(wtop[i]);
    any = any | (wmask[i] != 0);
#pragma unroll
    for (int j = 0; j < TM; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) any = any | odd(acc[i][j][e]);
  }
  if (__ballot(any) != 0 && lane == 0) again = 1;             // any of them: the same value
  __syncthreads();
  if (again) {
    f32x4 sum[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k0 = k_begin; k0 < k_stop; k0 += BK) {
      __syncthreads();
#pragma unroll
      for (int j = 0; j < XJ; ++j) {
        load(xsrc[j], xr[j], k0);
        clear_beyond(xr[j], k0);
#pragma unroll
        for (int h = 0; h < 2; ++h) if (mine(j)) plane(0, h, wave + NW * j)[lane] = __builtin_bit_cast(u32x4, xr[j][h] * sign);
      }
#pragma unroll
      for (int i = 0; i < TN; ++i) {
        load(wsrc[i], wr[i], k0);
        clear_beyond(wr[i], k0);
      }
      __syncthreads();
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < TM; ++j) {
          const f32x4 x = __builtin_bit_cast(f32x4, plane(0, h, j)[lane]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < TN; ++i) sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wr[i][h][e], x[e], sum[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < TN; ++i)
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)                           // output 4 g + e of row tile i, token c of token tile j
          if (((wmask[i] >> (g * 4 + e) | xmask[group][j] >> c) & 1) || odd(acc[i][j][e])) acc[i][j][e] = sum[i][j][e];
    __syncthreads();
  }

  // The outputs go through LDS: 16-byte pieces of a token's row, and the epilogue's functions stand in the code for four elements.
  auto Ys = reinterpret_cast<float (*)[YROW]>(lds);
  // the second group's negative sums first, which the first group then takes from its own
#pragma unroll
  for (int gr = KG - 1; gr >= 0; --gr) {
    if (gr == group) {
#pragma unroll
      for (int j = 0; j < TM; ++j)
#pragma unroll
        for (int i = 0; i < TN; ++i) {
          f32x4* p = reinterpret_cast<f32x4*>(&Ys[j * 16 + c][(wave * TN + i) * 16 + g * 4]);
          *p = gr == KG - 1 ? acc[i][j] : acc[i][j] - *p;
        }
    }
    __syncthreads();
  }
  float* __restrict__ y = Y + (size_t)slice * M * N;
  const int pieces = geglu ? BN / 8 : BN / 4;                 // of a row
#pragma unroll 1
  for (int id = tid; id < BM * pieces; id += THREADS) {
    const int r = id / pieces, q = (id % pieces) * 4, m = m0 + r, n = n0 + q;
    if (m >= M || n >= N) continue;
    f32x4 v;
    if (geglu) {
      const float* p = &Ys[r][q];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gated_act(p[e], p[BN / 2 + e], param, full);
    } else {
      v = *reinterpret_cast<const f32x4*>(&Ys[r][q]);
      if (epi == ALICE_EPI_SOFTCAP) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = unary_act(v[e], param, full);
      }
    }
    float* dst = y + (size_t)m * N + n;
    if (wide) {                                               // rows of whole, aligned pieces
      *reinterpret_cast<f32x4*>(dst) = v;
      continue;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < N) dst[e] = v[e];
  }
}

template <int TM, int TN>
int launch(const float* x, const float* w, float* y, int M, int N, int K, int epi, float param, int full, int split, hipStream_t stream) {
  constexpr int BM = 16 * TM, BN = 64 * TN;
  constexpr int STAGES = 2 * 2 * 3 * TM * 1024, OUT = BM * (BN + 4) * 4, LDS = STAGES > OUT ? STAGES : OUT;
  const int mt = ceil_div(M, BM), nt = ceil_div(N, epi == ALICE_EPI_GEGLU ? BN / 2 : BN);
  ALICE_CHECK((long)mt * nt * split < (1l << 30), "linear: too many tiles for one launch");
  const int kslice = ceil_div(ceil_div(K, split), BK) * BK;
  const int wide = N % 4 == 0 && ((uintptr_t)y & 15) == 0;
  const int grid = 8 * ceil_div((long)mt * nt * split, 8);
  auto kern = linear_thirds_kernel<TM, TN>;
  static std::atomic<uint64_t> told{0};
  ALICE_CHECK(LDS <= 48 * 1024 || lds_granted((const void*)kern, LDS, told), "linear: the device does not give a block %d bytes of LDS", LDS);
  kern<<<grid, 512, LDS, stream>>>(x, w, y, M, N, K, kslice, split, mt, nt, epi, param, full, wide);
  ALICE_LAUNCH_CHECK();
  return 0;
}

// Microseconds that a block takes for a stage of each of its groups with the chip full.
struct Tile {
  int bm, bn;
  float stage;
};
constexpr Tile TILES[] = {{128, 128, 2.5f}, {64, 192, 2.1f}, {64, 128, 1.5f}, {64, 64, 1.0f}, {32, 128, 1.35f}, {32, 64, 0.95f}};

}  // namespace

// The tile, and between min_split and max_split slices the number of them, by estimated microseconds: a CU's blocks one after the
// other; slices cost writing and reading their sums.  (Planned and measured, by weights that no cache holds: 512 tokens by 18,432 x
// 2,304 with GeGLU in 64 x 192, three blocks a CU, 233 and 246; 4,096 x 2,304 in two slices of 128 x 128 58 and 54; 2,304 x 9,216 in seven 127
// and 123, 2,304 x 2,048 in three 39 and 34; 128 tokens 80 and 78, 22 and 21, 40 and 41 in 64 x 192 and 64 x 128; 33 tokens by 2,304 x 9,216
// in 64 x 64 28 and 27; 17 by 28,672 x 2,304 with GeGLU in 32 x 128 53 and 54.)
ThirdsPlan alice_linear_thirds_plan(int M, int N, int K, bool geglu, int min_split, int max_split) {
  ThirdsPlan best{-1, 1, 1e30f};
  for (int i = 0; i < (int)(sizeof(TILES) / sizeof(TILES[0])); ++i) {
    const Tile& t = TILES[i];
    const int mt = ceil_div(M, t.bm), nt = ceil_div(N, geglu ? t.bn / 2 : t.bn);
    for (int s = min_split; s <= max_split; ++s) {
      const int ks = ceil_div(ceil_div(K, s), BK) * BK;
      if (s > 1 && (ks < 256 || (long)ks * (s - 1) >= K)) continue;          // no slice without elements
      const float us = 4.f + ceil_div(ceil_div((long)mt * nt * s, 8), 32) * (ceil_div(ks, 2 * BK) * t.stage + 0.7f) + (s > 1 ? 2.f * s * (float)M * N * 4.f / 4.0e6f : 0.f);
      if (us < best.us) best = ThirdsPlan{i, s, us};
    }
  }
  return best;
}

int alice_linear_thirds(const float* x, const float* w, float* y, int M, int N, int K, int epi, float param, int full, const ThirdsPlan& p,
                        hipStream_t stream) {
  ALICE_CHECK(K % 4 == 0 && ((uintptr_t)x & 15) == 0 && ((uintptr_t)w & 15) == 0 && p.split >= 1, "linear: operands for the products in thirds are not aligned");
#define GO(TM, TN) return launch<TM, TN>(x, w, y, M, N, K, epi, param, full, p.split, stream)
  switch (p.tile) {
    case 0: GO(8, 2);
    case 1: GO(4, 3);
    case 2: GO(4, 2);
    case 3: GO(4, 1);
    case 4: GO(2, 2);
    case 5: GO(2, 1);
  }
#undef GO
  alice_set_error("linear: no tile %d for the products in thirds", p.tile);
  return 1;
}
