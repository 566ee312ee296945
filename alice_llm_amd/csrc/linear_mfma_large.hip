// The matrix product of long prompts: tiles of 256 tokens by 256, 192 or 128 features, one block a CU, both operands staged
// straight from memory into LDS.  The layouts and the operand roles are described in linear_mfma.h; the tiled kernel
// (linear_mfma_tiled.h) takes everything that this one does not.  y[r] = sum_c W[r,c] x[c] (gguf.rs:4063-4074) with the gated
// epilogue (llama3.rs:14519-14534).
#include <type_traits>
#include "linear_mfma.h"

namespace {

constexpr int LARGE_XT = 16;            // token tiles of a block: 256 tokens
constexpr int LARGE_SLOTS = 5;          // k-tiles that LDS holds: 160, 140 or 120 KB

// One tile of 1 KB from memory into LDS, lane l's 16 bytes to place `lds` + `AT` KB + 16 l of the block's memory.  The instruction
// has no register for its result; what it counts on (vmcnt) is waited for ahead of the barriers below.  m0, which names the place, is an
// operand, so that the compiler knows what it holds; after a write of it the instruction needs one wait state.
template <int AT>
__device__ __forceinline__ void tile_to_lds(const bf16_t* src, unsigned off, uint32_t lds) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(src), "{m0}"(lds + AT * 1024) : "memory");
}

enum { GATE_GELU, GATE_SILU };

struct LargeShape {
  int M, KT, NT, gx, gy, tiles, items, per;   // k-tiles in all; tiles of the output; tiles times slices; k-tiles a slice
};

// Four waves, two by two, each 128 tokens by 8 FT features (FT: 16-feature tiles of a block): up to 256 accumulators a lane, which
// stay in the matrix registers (`pin` says so; left alone the compiler moves them to and fro, 400 moves for 128 products), and
// two sets of fragments, the k-tile that is multiplied and the next one.  A k-tile asks the CU's path to the L2 for
// (16 + FT) KB per 64 FT products, 32 KB with the widest tile, where two blocks of the tiled kernel ask for 48, and it is this path, the
// instructions beside the products and, with all CUs at it, the card's power that bound these products (on zeros, which take a third less power,
// 1.7 PFLOP/s where 1.4 are reached on numbers).
//
// LDS is a ring of five k-tiles.  While k-tile s is multiplied the fragments of s + 1 are read and s + 4 is staged, one
// read behind every fourth product and one tile behind every eighth, so that each is issued while a product runs.  Every
// second k-tile (the odd ones) begins with the one barrier there is: each wave has by then
//   - read all of k-tile s (it waits for its reads), so that the places of s - 1 and s may be staged anew: s + 4 into that of s - 1
//     behind this barrier, s + 5 into that of s behind it as well;
//   - waited for its own share of the staging of s + 1 and s + 2 (all but the last k-tile that it asked for), which are what is read
//     until the next barrier.
// A block goes through its tiles of the output in one run: behind a tile's last k-tiles the next tile's first ones are staged,
// so that only the epilogue stands between two tiles.  K-tiles come in pairs: a slice has an even number of them, four at least.
// GATE: which gated form (a choice at run time, made once an output, took the epilogue of GELU from 5 to 8 us a tile).  The gated
// instances of 256 features keep one to three registers in scratch, written and read outside the loops over k-tiles.
template <int EPI, typename TO, int FT, int GATE>
__global__ __launch_bounds__(256, 1) void linear_large_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ wf, LargeShape sh,
                                                           TO* __restrict__ y, int N, int y_frag) {
  constexpr int XT = LARGE_XT, HX = XT / 2, HW = FT / 2;   // token and feature tiles: a block's, a wave's
  constexpr int STAGE = (XT + FT) * 1024, RING = LARGE_SLOTS * STAGE;
  constexpr int PER = (XT + FT) / 4;                       // tiles that a wave stages a k-tile
  extern __shared__ __align__(16) char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  // Blocks go to the XCDs round robin by index; XCD c works through the c-th eighth of the items (tiles of a slice, the slices one
  // after the other), in bands of 1,024 tokens, a band column by column: the 32 blocks of an XCD are 4 by 8 tiles at a time, whose
  // operands its L2 reads once.  (14,494 tokens by 8,192 x 3,584: 664 us, in bands of 2,048 tokens 705, of 4,096 783.)
  const int xcd = blockIdx.x & 7, of_xcd = gridDim.x >> 3, share = (sh.items + 7) >> 3;
  const int end_item = min((xcd + 1) * share, sh.items);
  int item = xcd * share + (blockIdx.x >> 3);
  if (item >= end_item) return;
  constexpr int BAND = 4;
  auto place = [&](int it, int& slice, int& bx, int& by) {
    slice = it / sh.tiles;
    const int t = it - slice * sh.tiles, band = t / (BAND * sh.gx), in = t - band * BAND * sh.gx, high = min(BAND, sh.gy - band * BAND);
    bx = in / high;
    by = band * BAND + in - bx * high;
  };
  auto k_tiles = [&](int slice) { return min(sh.per, sh.KT - slice * sh.per); };

  // ---- staging: the sources of the wave's tiles, the lane's place behind them at the k-tile to stage, the ring's place for it
  const unsigned place16 = lane * 16;
  const bf16_t* src[PER];
  unsigned off = 0;
  uint32_t slot = wave * PER * 1024;
  auto sources = [&](int it) {
    int slice, bx, by;
    place(it, slice, bx, by);
    off = place16;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int t = wave * PER + i, f = t - XT;
      int w = bx * FT + f;
      if (EPI == ALICE_EPI_GEGLU) {                        // gate and up tiles in turn
        const int pair = bx * (FT / 2) + (f >> 1);
        w = pair < sh.NT / 2 ? ((f & 1) ? sh.NT / 2 + pair : pair) : sh.NT;
      }
      // (tiles beyond the matrix or the tokens: the last one's, results unused)
      src[i] = (t < XT ? x + (size_t)min(by * XT + t, (sh.M - 1) >> 4) * sh.KT * 512 : wf + (size_t)min(w, sh.NT - 1) * sh.KT * 512) +
               (size_t)slice * sh.per * 512;
    }
  };
  auto stage = [&](int i) {
    if (i == 0) tile_to_lds<0>(src[0], off, slot);
    if (i == 1) tile_to_lds<1>(src[1], off, slot);
    if (i == 2) tile_to_lds<2>(src[2], off, slot);
    if (i == 3) tile_to_lds<3>(src[3], off, slot);
    if (i == 4) tile_to_lds<4>(src[4], off, slot);
    if (i == 5) tile_to_lds<5>(src[5], off, slot);
    if constexpr (PER > 6) if (i == 6) tile_to_lds<6>(src[6], off, slot);
    if constexpr (PER > 7) if (i == 7) tile_to_lds<7>(src[7], off, slot);
  };
  static_assert(PER >= 6 && PER <= 8, "the tiles that a wave stages");
  auto staged = [&]() {
    off += 1024;
    slot = slot + STAGE >= RING ? slot + STAGE - RING : slot + STAGE;
  };

  f32x4 acc[HW][HX];
  auto pin = [&]() {
#pragma unroll
    for (int i = 0; i < HW; ++i)
#pragma unroll
      for (int j = 0; j < HX; ++j) asm volatile("" : "+a"(acc[i][j]));
  };
  u32x4 xf[2][HX], wk[2][HW];
  uint32_t from = 0;                                       // the ring's place that fragments are read from
  const char* w_lds = lds + (XT + wn * HW) * 1024 + place16;
  const char* x_lds = lds + wm * HX * 1024 + place16;
  auto read_w = [&](int i) { return *reinterpret_cast<const u32x4*>(w_lds + from + i * 1024); };
  auto read_x = [&](int j) { return *reinterpret_cast<const u32x4*>(x_lds + from + j * 1024); };

  // One k-tile: its products, the reads of the next one's fragments, the staging of the one four on.
  auto k_tile = [&](auto meet, u32x4 (&w0)[HW], u32x4 (&x0)[HX], u32x4 (&w1)[HW], u32x4 (&x1)[HX]) {
    if constexpr (decltype(meet)::value) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(PER) : "memory");
    from = from + STAGE >= RING ? 0 : from + STAGE;
    constexpr int PRODUCTS = HW * HX, READS = HW + HX, SPAN = PRODUCTS - 8;      // (the last read has eight products to arrive in)
#pragma unroll
    for (int j = 0; j < HX; ++j) {
#pragma unroll
      for (int i = 0; i < HW; ++i) {
        acc[i][j] = mfma16(w0[i], x0[j], acc[i][j]);
        const int n = j * HW + i, rd = n * READS / SPAN, st = n * PER / PRODUCTS;
        if (rd < READS && (n + 1) * READS / SPAN > rd) {
          __builtin_amdgcn_sched_barrier(0);
          if (rd < HW) w1[rd] = read_w(rd);
          else x1[rd - HW] = read_x(rd - HW);
          __builtin_amdgcn_sched_barrier(0);
        }
        if ((n + 1) * PER / PRODUCTS > st) {
          __builtin_amdgcn_sched_barrier(0);
          stage(st);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    staged();
  };

  sources(item);
#pragma unroll 1
  for (int s = 0; s < LARGE_SLOTS - 1; ++s) {
#pragma unroll
    for (int i = 0; i < PER; ++i) stage(i);
    staged();
  }
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((LARGE_SLOTS - 3) * PER) : "memory");      // k-tiles 0 and 1 are there
#pragma unroll
  for (int i = 0; i < HW; ++i) wk[0][i] = read_w(i);
#pragma unroll
  for (int j = 0; j < HX; ++j) xf[0][j] = read_x(j);

#pragma unroll 1
  for (; item < end_item; item += of_xcd) {
    int slice, bx, by;
    place(item, slice, bx, by);
    const int kts = k_tiles(slice);
#pragma unroll
    for (int i = 0; i < HW; ++i)
#pragma unroll
      for (int j = 0; j < HX; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    pin();
    // the last four k-tiles stage the first four of the block's next item (behind its last item: that one's again, never read)
    int s = 0;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {
      if (part) sources(min(item + of_xcd, end_item - 1));
      const int end = part ? kts : kts - (LARGE_SLOTS - 1);
#pragma unroll 1
      for (; s < end; s += 2) {
        k_tile(std::false_type{}, wk[0], xf[0], wk[1], xf[1]);
        k_tile(std::true_type{}, wk[1], xf[1], wk[0], xf[0]);
        pin();
      }
    }
    int lane_e = lane;
    asm volatile("" : "+v"(lane_e));                       // (so that none of the epilogue's addresses is kept in registers through the products)
    const int r = lane_e & 15, g = lane_e >> 4;
    TO* ys = y + (size_t)slice * sh.M * N;                 // the slice's own partial result
#pragma unroll
    for (int j = 0; j < HX; ++j) {
      const int m = (by * XT + wm * HX + j) * 16 + r;
      __builtin_amdgcn_sched_barrier(0);
      if (m >= sh.M) continue;
      if constexpr (EPI == ALICE_EPI_GEGLU) {
#pragma unroll
        for (int p = 0; p < HW / 2; ++p) {
          const int pair = bx * (FT / 2) + wn * (HW / 2) + p, n = pair * 16 + g * 4;
          if (pair >= sh.NT / 2) continue;
          f32x4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) 
            o[e] = (GATE == GATE_GELU ? gelu_tanh_f(acc[2 * p][j][e], false) : silu_f(acc[2 * p][j][e], false)) * acc[2 * p + 1][j][e];
          if (y_frag) store4_frag((bf16_t*)ys, m, n, N, o);
          else *reinterpret_cast<uint2*>((bf16_t*)ys + (size_t)m * N + n) = uint2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])};
        }
      } else {
#pragma unroll
        for (int i = 0; i < HW; ++i) {
          const int tile = bx * FT + wn * HW + i;
          if (tile < sh.NT) *reinterpret_cast<f32x4*>((float*)ys + (size_t)m * N + tile * 16 + g * 4) = acc[i][j];
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // no staging is on its way when the block gives its LDS back
}

template <int EPI, typename TO, int FT, int GATE>
int launch_large(const void* x, const void* w, void* y, const LargeShape& sh, int N, int y_frag, hipStream_t s) {
  auto kern = linear_large_kernel<EPI, TO, FT, GATE>;
  constexpr int lds = LARGE_SLOTS * (LARGE_XT + FT) * 1024;
  static std::atomic<uint64_t> told{0};
  ALICE_CHECK(lds_granted((const void*)kern, lds, told), "linear: the device does not give a block %d bytes of LDS", lds);
  const int blocks = sh.items < 256 ? 8 * ceil_div(sh.items, 8) : 256;
  kern<<<blocks, 256, lds, s>>>((const bf16_t*)x, (const bf16_t*)w, sh, (TO*)y, N, y_frag);
  ALICE_LAUNCH_CHECK();
  return 0;
}

}  // namespace

// Whether the kernel takes a product cut into `split` slices: whole output tiles, k-tiles in pairs, two pairs a slice at least.
bool alice_mfma_large_takes(int M, int N, int K, int epi, float epi_param, int y_dtype, int split) {
  if (M < 1 || K % 64 != 0 || N % 16 != 0 || split < 1) return false;
  if (!(epi == ALICE_EPI_NONE && y_dtype == DT_F32) && !(epi == ALICE_EPI_GEGLU && epi_param <= 0.f && y_dtype == DT_BF16 && split == 1)) return false;
  const int KT = K / 32, per = ceil_div(KT, split), last = KT - per * (split - 1);
  return per % 2 == 0 && last >= 4 && last <= per;
}

// Microseconds of a product by this kernel and by the tiled one with its widest tile.  A block of this kernel takes 0.64, 0.52 or 0.42 us a
// k-tile and 4 to 11 us a tile beside them; the last round of blocks, with part of the chip idle, runs faster for the power that these
// leave.  Every slice is a partial result that the add and norm behind it reads.
// Sums without an epilogue: fitted to 170 products, ten matrices of the 2B, 9B and 27B widths and of 2,048 and 2,560 at 450 to 8,192 tokens,
// with weights that no cache holds, as a model's layers find them (to 4 % either kernel's; the choices that follow are 1.08 times as fast as
// the tiled kernel, 1.4 % behind the best measured ones on average, and none is more than 2 % slower than the tiled kernel.  Costs
// fitted to weights that a cache held took 128 features too cheaply: 39 of the 170 lost 2 to 12 %, 1,024 tokens by 2,304 x 2,048 for one).
// Gated products: fitted to 34 of them at 512 to 8,192 tokens, of weights that a cache held; of 68 with cold weights one is 1.8 % slower than
// the tiled kernel (2,048 wide at 505 tokens) and two that could gain an eighth stay with it (2B and 2,048 wide at 600).
static float large_cost(int M, int N, int K, int epi, int ft, int split) {
  const bool gated = epi == ALICE_EPI_GEGLU;
  const float k_tile = gated ? (ft == 16 ? 0.66f : ft == 12 ? 0.49f : 0.37f) : (ft == 16 ? 0.64f : ft == 12 ? 0.516f : 0.42f);
  const float tile = gated ? (ft == 16 ? 7.f : ft == 12 ? 5.9f : 3.9f) : (ft == 16 ? 10.6f : ft == 12 ? 7.9f : 5.f);
  const float part = gated ? 0.68f : ft == 16 ? 0.726f : ft == 12 ? 0.759f : 0.825f;     // a round's time with hardly a block in it
  const int items = ceil_div(N / 16 * (gated ? 2 : 1), ft) * ceil_div(M, 16 * LARGE_XT) * split, rounds = ceil_div(items, 256);
  const float busy = rounds - 1 + part + (1.f - part) * (items / 256.f - (rounds - 1));
  return 3.5f + busy * (ceil_div(K / 32, split) * k_tile + tile) + 0.99e-6f * (split - 1) * M * N;
}
static float tiled_wide_cost(int M, int N, int K, int epi, int split) {
  const bool gated = epi == ALICE_EPI_GEGLU;
  const float rounds = (float)ceil_div(N * (gated ? 2 : 1), 256) * ceil_div(M, 128) * split / 256.f;
  const int pairs = (ceil_div((long)ceil_div(N * (gated ? 2 : 1), 256) * ceil_div(M, 128) * split, 256) - 1) / 2;
  const float rest = rounds - 2 * pairs;                   // two blocks a CU in 1.79 times the time of one
  const float busy = 1.79f * pairs + (rest <= 1.f ? 0.6f + 0.4f * rest : 1.f + 0.79f * (0.57f + 0.43f * (rest - 1.f)));
  return 4.3f + busy * (ceil_div(K / 32, split) * 0.435f + (gated ? 1.6f : 4.f)) + 0.85e-6f * (split - 1) * M * N;
}

// The tile for a product that the tiled kernel would take as `tiled` says, ft 0: that one.  split 0: the slices are chosen too.  From 448
// tokens on: below, sums in one round of blocks that wait for memory are better off in the tiled kernel's tiles (this kernel
// gains at a few gated products of 320 to 447 tokens, 9B at 384 101 -> 83 us, for which the costs are not fitted).  Where the tiled kernel has a
// narrow tile for the sums of a few hundred tokens the cost above is its widest tile's and this kernel must promise a quarter less; where it has
// low blocks of long slices, two on some CUs, it takes a fifth longer than the cost says (4,096 inner elements, 342 blocks: 74 us for 57).
// Elsewhere sums must promise 2 % and gated products 3: nearer than that (2,048 tokens by 2,048 x 8,192: 60.5 and 61.4 us in one run, 63.1 and
// 60.3 in another) a model was faster with the tiled kernel.
// With weights that no cache holds, 2B down at 2,048 tokens 87 -> 72 us, 9B output at 3,072 92 -> 76, 27B down at 1,024 307 -> 241; gated
// ones, with weights from a cache, 2B at 2,048 tokens 147 -> 130, 9B at 8,192 1,249 -> 1,140.
LargePlan alice_mfma_large_plan(int M, int N, int K, int epi, float epi_param, int y_dtype, int split, const TiledPlan& tiled) {
  LargePlan best{0, tiled.split};
  if (M < LARGE_FROM || !alice_frag16_supported(N * (epi == ALICE_EPI_GEGLU ? 2 : 1), K, epi)) return best;
  const int slices = split > 0 ? split : tiled.split;
  float least = tiled_wide_cost(M, N, K, epi, slices);
  if (epi == ALICE_EPI_GEGLU) least *= 0.97f;
  else if (tiled.wn < 4) least *= 0.74f;
  else if (tiled.tm == 4 && (long)ceil_div(N, 256) * ceil_div(M, 64) * slices > 256 && ceil_div(K / 32, slices) >= 64) least *= 1.19f;
  else least *= 0.98f;
  for (int sp = split > 0 ? split : 1; sp <= (split > 0 ? split : 4); ++sp) {
    if (!alice_mfma_large_takes(M, N, K, epi, epi_param, y_dtype, sp) || (sp > 1 && split == 0 && K / 32 / sp < 16)) continue;
    for (int ft = 16; ft >= 8; ft -= 4) {
      const float cost = large_cost(M, N, K, epi, ft, sp);
      if (cost < least) { least = cost; best = LargePlan{ft, sp}; }
    }
  }
  return best;
}

// (A plan weighs both kernels at their own numbers of slices.  Weighed again at the number that was chosen, the other kernel may win: 2 slices
// of 1,100 tokens by 2,304 x 2,048 are proposed for this one, where the tiled kernel would like 3 and take 2 a little faster.)
LargePlan alice_mfma_large_choice(int M, int N, int K, int epi, float epi_param, int y_dtype, int split) {
  if (epi == ALICE_EPI_NONE && y_dtype == DT_F32) {
    const LargePlan proposed = alice_mfma_large_plan(M, N, K, epi, epi_param, y_dtype, 0, alice_mfma_tiled_plan(M, N, K, epi, y_dtype, 0, 1));
    if (proposed.split == split) return proposed;
  }
  return alice_mfma_large_plan(M, N, K, epi, epi_param, y_dtype, split, alice_mfma_tiled_plan(M, N, K, epi, y_dtype, split, 1));
}
extern "C" int alice_linear_large_tile(int M, int N, int K, int epilogue, float epi_param, int y_dtype, int split_k) {
  return M >= LARGE_FROM ? 16 * alice_mfma_large_choice(M, N, K, epilogue, epi_param, y_dtype, split_k).ft : 0;
}

int alice_mfma_large(const void* x, const void* w, void* y, int M, int N, int K, int epi, float epi_param, int split, int ft, int y_frag,
                     hipStream_t s) {
  const int NT = N / 16 * (epi == ALICE_EPI_GEGLU ? 2 : 1), gx = ceil_div(NT, ft), gy = ceil_div(M, 16 * LARGE_XT);
  ALICE_CHECK((long)gx * gy * split < (1l << 26), "linear: too many tiles for one launch");
  const LargeShape sh{M, K / 32, NT, gx, gy, gx * gy, gx * gy * split, ceil_div(K / 32, split)};
#define GO(FT)                                                                                                        \
  do {                                                                                                                \
    if (epi == ALICE_EPI_GEGLU && epi_param == 0.f) return launch_large<ALICE_EPI_GEGLU, bf16_t, FT, GATE_GELU>(x, w, y, sh, N, y_frag, s);  \
    if (epi == ALICE_EPI_GEGLU) return launch_large<ALICE_EPI_GEGLU, bf16_t, FT, GATE_SILU>(x, w, y, sh, N, y_frag, s);  \
    return launch_large<ALICE_EPI_NONE, float, FT, GATE_GELU>(x, w, y, sh, N, 0, s);                                  \
  } while (0)
  if (ft == 16) GO(16);
  if (ft == 12) GO(12);
  ALICE_CHECK(ft == 8, "linear: no tile of 256 tokens by %d features", 16 * ft);
  GO(8);
#undef GO
}
