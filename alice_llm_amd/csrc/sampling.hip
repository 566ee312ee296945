// Choosing the next token from float32 logits [B, V] on the device: argmax, and
// temperature -> top-k -> top-p -> softmax -> inverse CDF with a given uniform number per row.
//
// Semantics of the reference's host functions (src/sampling.rs:10-123): temperature multiplies the
// logits by 1/T; top-k keeps the k largest, ties at the threshold kept (25-41); top-p keeps the
// shortest descending prefix whose cumulative probability exceeds p (45-74; here all values tied
// with the last kept one are kept as well); softmax subtracts the maximum (77-92); the draw is the
// first index whose cumulative probability exceeds u (114-123).  Argmax returns the lowest index
// among equal maxima (llama3.rs:18862-18872).  One block per row; every reduction has a fixed
// order, so a row's result depends on nothing but the row, u and the options.
#include "common.h"
#include "alice_hip.h"

namespace {

constexpr int ST = 1024;     // threads per row

__device__ __forceinline__ uint32_t order_key(float x) {
  uint32_t b = __float_as_uint(x);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// Stage 1 (chunks > 1): block (row, chunk) scans its slice of the row and writes (value, index) to `part`;
// stage 2 runs the same kernel over the partial results.  The lowest index wins among equal values at
// both stages, so the result does not depend on the number of chunks.
__global__ __launch_bounds__(ST) void argmax_kernel(const float* __restrict__ vals, const int* __restrict__ idxs,
                                                    int* __restrict__ out, float* __restrict__ part_v,
                                                    int* __restrict__ part_i, int V, int chunks) {
  __shared__ float bv[ST / 64];
  __shared__ int bi[ST / 64];
  const float* row = vals + (size_t)blockIdx.x * V;
  const int* irow = idxs ? idxs + (size_t)blockIdx.x * V : nullptr;
  const int per = (V + chunks - 1) / chunks;
  const int lo = blockIdx.y * per, hi = min(V, lo + per);
  float best = -INFINITY;
  int idx = 0x7fffffff;
  for (int i = lo + threadIdx.x; i < hi; i += ST) {
    float v = row[i];
    int id = irow ? irow[i] : i;
    if (v > best || (v == best && id < idx)) { best = v; idx = id; }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    float ov = __shfl_xor(best, o, 64);
    int oi = __shfl_xor(idx, o, 64);
    if (ov > best || (ov == best && oi < idx)) { best = ov; idx = oi; }
  }
  if ((threadIdx.x & 63) == 0) { bv[threadIdx.x >> 6] = best; bi[threadIdx.x >> 6] = idx; }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < ST / 64; ++w)
      if (bv[w] > best || (bv[w] == best && bi[w] < idx)) { best = bv[w]; idx = bi[w]; }
    if (chunks > 1) {
      part_v[(size_t)blockIdx.x * chunks + blockIdx.y] = best;
      part_i[(size_t)blockIdx.x * chunks + blockIdx.y] = idx;
    } else {
      out[blockIdx.x] = idx == 0x7fffffff ? 0 : idx;
    }
  }
}

__device__ __forceinline__ int block_count(int v, int* ired) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  v = wave_reduce(v, [](int a, int b) { return a + b; });
  __syncthreads();
  if (lane == 0) ired[wid] = v;
  __syncthreads();
  int t = 0;
  for (int w = 0; w < ST / 64; ++w) t += ired[w];
  return t;
}

// Inclusive prefix sum over a block of ST in thread order; `excl` gets the previous thread's inclusive sum (bit for bit).
__device__ __forceinline__ float block_inclusive_scan(float v, float* wred, float* excl) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    float n = __shfl_up(v, o, 64);
    if (lane >= o) v += n;
  }
  float prev = __shfl_up(v, 1, 64);
  __syncthreads();
  if (lane == 63) wred[wid] = v;
  __syncthreads();
  float before = 0.f;                                      // (all the waves' sums at once: what is not before this wave adds zero)
#pragma unroll
  for (int w = 0; w < ST / 64 - 1; ++w) before += w < wid ? wred[w] : 0.f;
  // the thread before lane 0 is lane 63 of the wave before: its inclusive sum is (sum of waves < wid-1) + wred[wid-1],
  // which is how `before` was built
  *excl = lane == 0 ? before : before + prev;
  return before + v;
}

// ---- sampling: a row is cut into chunks, a block per chunk for every pass over the row, one block per row
// for what needs the whole row
//
//   chunk_max        the maximum of every chunk
//   chunk_count      how many elements of the chunk lie within fixed distances of the row's maximum (and, for
//                    top-p alone, the chunk's probability mass)
//   chunk_collect    the elements within the chosen distance (at most capg a row) go to the row's list
//   row_threshold    the thresholds of top-k and top-p by bisection on the key space over that list, held in
//                    shared memory (up to CAP candidates: one wave does it) or read from memory by the whole
//                    block; probabilities enter as 64-bit fixed point, so the sums do not depend on the
//                    order in which the list was filled.  A row whose kept set does not fit (a flat
//                    distribution, a huge k) takes the same bisection over the whole row instead.
//   tile_sum         the kept mass of every tile of TILE elements (a wave per tile, lanes in a fixed order)
//   draw             the tile in which the cumulative sum, in index order, passes the target, and a scan of it
//
// Without top-k and top-p only the first and the last two run.  Every pass reads four consecutive elements per
// thread per load where the vocabulary is a multiple of four.
constexpr int TILE = 4096;       // 4 consecutive elements per thread of the draw's scan
constexpr int CAP = 4096;        // candidates held in shared memory
constexpr int CAPG = 32768;      // candidates of a row's list in memory, at most (fewer for very many rows: list_room())
constexpr int NCUT = 12;
constexpr int SB = 256;          // threads of the per-chunk kernels
constexpr int NMC = 4;           // distances at which the mass inside is summed too (top-p alone)
__device__ constexpr int kMassCut[NMC] = {5, 7, 8, 9};   // indices into kCut: 4, 8, 10, 12
__device__ constexpr float kCut[NCUT] = {0.5f, 1.f, 1.5f, 2.f, 3.f, 4.f, 6.f, 8.f, 10.f, 12.f, 16.f, 24.f};

__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// exp(x - m) <= 1 as 24.40 fixed point
__device__ __forceinline__ unsigned long long fixed_mass(float x, float m) {
  return (unsigned long long)(expf(x - m) * 0x1p40f);
}

__device__ __forceinline__ unsigned long long wave_sum_u64(unsigned long long v) {
  return wave_reduce(v, [](unsigned long long a, unsigned long long b) { return a + b; });
}

// Where a row's intermediate results live (all arrays are per row; `chunks` and `tiles` per row).
struct SampleWork {
  float* pmax;                   // [B][chunks]
  int* pcnt;                     // [B][chunks][NCUT]
  unsigned long long* pmass;     // [B][chunks][1 + NMC]: the chunk's mass, and its mass within kCut[kMassCut[i]] of the maximum
  uint32_t* cand;                // [B][capg]
  unsigned long long* cmass;     // [B][capg]: the candidates' masses, for lists too long for shared memory
  uint32_t* thr;                 // [B]
  float* tsum;                   // [B][tiles]
  int* tlast;                    // [B][tiles]
  int chunks, tiles, tiles_per_chunk, capg;
};

// f(index, logit / T, valid) for the elements [lo, hi) of a row (lo a multiple of four); every lane of the block
// runs every call (those past the end with valid = false), in an order that depends on nothing but the thread,
// the block's size NT and the range.
template <int VEC, int NT, class F>
__device__ __forceinline__ void for_range(const float* __restrict__ row, int lo, int hi, float inv_t, F&& f) {
  const int tid = threadIdx.x;
  if constexpr (VEC == 4) {
    constexpr int U = 4;
    const int G0 = lo >> 2, G = hi >> 2;
    const float4* r4 = reinterpret_cast<const float4*>(row);
    for (int g0 = G0; g0 < G; g0 += NT * U) {
      float4 x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = r4[min(g0 + u * NT + tid, G - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int g = g0 + u * NT + tid;
        const bool ok = g < G;
        f(4 * g + 0, x[u].x * inv_t, ok);
        f(4 * g + 1, x[u].y * inv_t, ok);
        f(4 * g + 2, x[u].z * inv_t, ok);
        f(4 * g + 3, x[u].w * inv_t, ok);
      }
    }
  } else {
    constexpr int U = 8;
    for (int i0 = lo; i0 < hi; i0 += NT * U) {
      float x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = row[min(i0 + u * NT + tid, hi - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) f(i0 + u * NT + tid, x[u] * inv_t, i0 + u * NT + tid < hi);
    }
  }
}

// The row's maximum from its chunks' (every wave computes it for itself).
__device__ __forceinline__ float row_max(const SampleWork& w, int b) {
  float m = -INFINITY;
  for (int c = threadIdx.x & 63; c < w.chunks; c += 64) m = fmaxf(m, w.pmax[(size_t)b * w.chunks + c]);
  return wave_max(m);
}

template <int VEC>
__global__ __launch_bounds__(SB) void chunk_max_kernel(const float* __restrict__ logits, SampleWork w, int V, float inv_t) {
  __shared__ float red[16];
  const int b = blockIdx.y, c = blockIdx.x;
  const float* row = logits + (size_t)b * V;
  const int lo = c * w.tiles_per_chunk * TILE, hi = min(V, lo + w.tiles_per_chunk * TILE);
  float lmax = -INFINITY;
  for_range<VEC, SB>(row, lo, hi, inv_t, [&](int, float x, bool ok) { lmax = fmaxf(lmax, ok ? x : -INFINITY); });
  const float m = block_max(lmax, red);
  if (threadIdx.x == 0) {
    w.pmax[(size_t)b * w.chunks + c] = m;
  }
}

template <int VEC>
__global__ __launch_bounds__(SB) void chunk_count_kernel(const float* __restrict__ logits, SampleWork w, int V, float inv_t,
                                                         int whole_mass) {
  __shared__ int wave_cnt[SB / 64][NCUT];
  __shared__ unsigned long long wave_mass[SB / 64][1 + NMC];
  const int b = blockIdx.y, c = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const float* row = logits + (size_t)b * V;
  const int lo = c * w.tiles_per_chunk * TILE, hi = min(V, lo + w.tiles_per_chunk * TILE);
  const float m = row_max(w, b);
  int cnt[NCUT];
#pragma unroll
  for (int j = 0; j < NCUT; ++j) cnt[j] = 0;
  unsigned long long mass[1 + NMC];
#pragma unroll
  for (int i = 0; i <= NMC; ++i) mass[i] = 0;
  for_range<VEC, SB>(row, lo, hi, inv_t, [&](int, float x, bool ok) {
    const float d = ok ? m - x : INFINITY;
#pragma unroll
    for (int j = 0; j < NCUT; ++j) cnt[j] += d <= kCut[j];
    if (whole_mass && ok) {
      const unsigned long long e = fixed_mass(x, m);
      mass[0] += e;
#pragma unroll
      for (int i = 0; i < NMC; ++i) mass[1 + i] += d <= kCut[kMassCut[i]] ? e : 0ull;
    }
  });
  if (whole_mass) {
#pragma unroll
    for (int i = 0; i <= NMC; ++i) mass[i] = wave_sum_u64(mass[i]);
  }
#pragma unroll
  for (int j = 0; j < NCUT; ++j) cnt[j] = wave_reduce(cnt[j], [](int a, int b) { return a + b; });
  if (lane == 0) {
#pragma unroll
    for (int j = 0; j < NCUT; ++j) wave_cnt[wave][j] = cnt[j];
#pragma unroll
    for (int i = 0; i <= NMC; ++i) wave_mass[wave][i] = mass[i];
  }
  __syncthreads();
  if (threadIdx.x < NCUT) {
    int t = 0;
    for (int v = 0; v < SB / 64; ++v) t += wave_cnt[v][threadIdx.x];
    w.pcnt[((size_t)b * w.chunks + c) * NCUT + threadIdx.x] = t;
  }
  if (threadIdx.x < 1 + NMC) {
    unsigned long long t = 0;
    for (int v = 0; v < SB / 64; ++v) t += wave_mass[v][threadIdx.x];
    w.pmass[((size_t)b * w.chunks + c) * (1 + NMC) + threadIdx.x] = t;
  }
}

// The row's counts per distance (and, for top-p alone, its mass and the masses within some distances) from the
// chunks', into tot[NCUT] and z[1 + NMC] in shared memory; then the distance whose elements become the list:
// for top-k the nearest that holds k; for top-p alone the nearest whose mass clearly exceeds p times the row's,
// else the widest that fits; -1 if none does.  All threads of the block call it (blockDim.x >= 256) and get the
// same answer.
__device__ __forceinline__ int choose_cut(const SampleWork& w, int b, bool need_k, int top_k, float top_p, int* tot,
                                          unsigned long long* z) {
  const int t = threadIdx.x;
  if (t < NCUT * 16) {
    const int j = t / 16, part = t % 16;
    int sum = 0;
    for (int c = part; c < w.chunks; c += 16) sum += w.pcnt[((size_t)b * w.chunks + c) * NCUT + j];
#pragma unroll
    for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
    if (part == 0) tot[j] = sum;
  }
  if (t >= NCUT * 16 && t < NCUT * 16 + 1 + NMC && !need_k) {
    unsigned long long sum = 0;
    for (int c = 0; c < w.chunks; ++c) sum += w.pmass[((size_t)b * w.chunks + c) * (1 + NMC) + (t - NCUT * 16)];
    z[t - NCUT * 16] = sum;
  }
  __syncthreads();
  int cut = -1;
  if (!need_k) {
    const unsigned long long target = (unsigned long long)((double)top_p * (double)z[0]);
#pragma unroll
    for (int i = 0; i < NMC; ++i) {
      const int c = tot[kMassCut[i]];
      if (cut == -1 && c >= 1 && c <= w.capg && z[1 + i] > target + (target >> 16)) cut = kMassCut[i];
    }
    if (cut >= 0) return cut;
  }
#pragma unroll
  for (int j = 0; j < NCUT; ++j) {
    const int c = tot[j];
    if (need_k) { if (cut == -1 && c >= top_k && c <= w.capg) cut = j; if (cut == -1 && c > w.capg) cut = -2; }
    else if (c >= 1 && c <= w.capg) cut = j;
  }
  return cut;
}

template <int VEC>
__global__ __launch_bounds__(SB) void chunk_collect_kernel(const float* __restrict__ logits, SampleWork w, int V, float inv_t,
                                                           int top_k, float top_p) {
  __shared__ int tot[NCUT];
  __shared__ unsigned long long z[1 + NMC];
  const int b = blockIdx.y, c = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const bool need_k = top_k > 0 && top_k < V;
  const int cut = choose_cut(w, b, need_k, top_k, top_p, tot, z);
  if (cut < 0) return;
  const float* row = logits + (size_t)b * V;
  const int lo = c * w.tiles_per_chunk * TILE, hi = min(V, lo + w.tiles_per_chunk * TILE);
  const float m = row_max(w, b);
  float dcut = kCut[0];
#pragma unroll
  for (int j = 0; j < NCUT; ++j) if (j == cut) dcut = kCut[j];
  // Where this chunk's candidates go in the row's list: after those of the chunks before it, whose numbers the
  // counting kernel left (no atomic on memory: thousands of them on one address took most of a millisecond).
  // Within the chunk a counter in shared memory hands out the places.
  __shared__ int before, fill;
  if (threadIdx.x == 0) { before = 0; fill = 0; }
  __syncthreads();
  {
    int mine = 0;
    for (int cc = threadIdx.x; cc < c; cc += SB) mine += w.pcnt[((size_t)b * w.chunks + cc) * NCUT + cut];
    mine = wave_reduce(mine, [](int a, int b) { return a + b; });
    if (lane == 0 && mine) atomicAdd(&before, mine);
  }
  __syncthreads();
  uint32_t* list = w.cand + (size_t)b * w.capg + before;
  const int room = w.capg - before;
  for_range<VEC, SB>(row, lo, hi, inv_t, [&](int, float x, bool ok) {
    const bool in = ok && (m - x <= dcut);
    const unsigned long long mask = __ballot(in);
    if (mask) {
      const int leader = __ffsll((long long)mask) - 1;
      int base = 0;
      if (lane == leader) base = atomicAdd(&fill, __popcll(mask));
      base = __shfl(base, leader, 64);
      const int pos = base + __popcll(mask & ((1ull << lane) - 1ull));
      if (in && pos < room) list[pos] = order_key(x);
    }
  });
}

// The thresholds by bisection over the whole row, for what a list could not settle; all threads of a block of ST call it.
template <int VEC>
__device__ __forceinline__ uint32_t whole_row_threshold(const float* __restrict__ row, int V, float inv_t, float m, uint32_t key_m,
                                                        uint32_t thr, bool k_done, bool p_done, int top_k, float top_p, float* red,
                                                        int* ired) {
  if (!k_done) {
    uint32_t lo = 0, hi = key_m;
    while (lo < hi) {
      const uint32_t mid = lo + (uint32_t)(((uint64_t)hi - lo + 1) >> 1);
      int c = 0;
      for_range<VEC, ST>(row, 0, V, inv_t, [&](int, float x, bool ok) { c += ok && order_key(x) >= mid; });
      if (block_count(c, ired) >= top_k) lo = mid; else hi = mid - 1;
    }
    thr = lo;
  }
  if (!p_done) {
    float z = 0.f;
    for_range<VEC, ST>(row, 0, V, inv_t, [&](int, float x, bool ok) { if (ok && order_key(x) >= thr) z += expf(x - m); });
    const float target = top_p * block_sum(z, red);
    uint32_t lo = thr, hi = key_m;
    while (lo < hi) {
      const uint32_t mid = lo + (uint32_t)(((uint64_t)hi - lo + 1) >> 1);
      float s = 0.f;
      for_range<VEC, ST>(row, 0, V, inv_t, [&](int, float x, bool ok) { if (ok && order_key(x) >= mid) s += expf(x - m); });
      if (block_sum(s, red) > target) lo = mid; else hi = mid - 1;
    }
    thr = lo;
  }
  return thr;
}

// The thresholds by bisection over the row's list of the n elements within the chosen distance of the maximum m (cut < 0: there is
// none); list, list_mass: CAP elements of shared memory; z_row: (top-p alone) the whole row's mass.  All threads of a block of ST call it.
template <int VEC>
__device__ __forceinline__ uint32_t list_threshold(const float* __restrict__ row, const SampleWork& w, int b, int V, float inv_t, float m,
                                                   int cut, int n, unsigned long long z_row, int top_k, float top_p, uint32_t* list,
                                                   unsigned long long* list_mass, float* red, int* ired) {
  __shared__ uint32_t found[3];                           // threshold, top-k done, top-p done
  __shared__ unsigned long long wsum[ST / 64];
  __shared__ uint32_t wmin[ST / 64];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t key_m = order_key(m);
  const bool need_k = top_k > 0 && top_k < V, need_p = top_p < 1.f;
  uint32_t thr = 0;
  bool k_done = !need_k, p_done = !need_p;
  if (tid == 0) { found[0] = 0; found[1] = 0; found[2] = 0; }
  if (cut >= 0 && n > CAP) {
    // a long list: the same bisections by the whole block over the list in memory
    const uint32_t* gl = w.cand + (size_t)b * w.capg;
    unsigned long long* gm = w.cmass + (size_t)b * w.capg;
    auto block_sum_u64 = [&](unsigned long long v) {
      v = wave_sum_u64(v);
      __syncthreads();
      if (lane == 0) wsum[wave] = v;
      __syncthreads();
      unsigned long long t = 0;
      for (int x = 0; x < ST / 64; ++x) t += wsum[x];
      return t;
    };
    uint32_t kmin = 0xffffffffu;
    for (int j = tid; j < n; j += ST) {
      const uint32_t key = gl[j];
      kmin = min(kmin, key);
      if (need_p) gm[j] = fixed_mass(key_value(key), m);
    }
    kmin = wave_reduce(kmin, [](uint32_t a, uint32_t b) { return min(a, b); });
    if (lane == 0) wmin[wave] = kmin;
    __syncthreads();                                      // also: the masses are written
    for (int x = 0; x < ST / 64; ++x) kmin = min(kmin, wmin[x]);
    uint32_t t = kmin;
    if (need_k) {
      uint32_t lo = kmin, hi = key_m;
      while (lo < hi) {
        const uint32_t mid = lo + (uint32_t)(((uint64_t)hi - lo + 1) >> 1);
        int c = 0;
        for (int j = tid; j < n; j += ST) c += gl[j] >= mid;
        if (block_count(c, ired) >= top_k) lo = mid; else hi = mid - 1;
      }
      t = lo;
    }
    k_done = true;
    thr = need_k ? t : 0u;
    if (need_p) {
      unsigned long long kept = 0;
      for (int j = tid; j < n; j += ST) if (gl[j] >= t) kept += gm[j];
      kept = block_sum_u64(kept);
      const unsigned long long z = need_k ? kept : z_row;
      const unsigned long long target = (unsigned long long)((double)top_p * (double)z);
      if (kept > target) {
        uint32_t lo = t, hi = key_m;
        while (lo < hi) {
          const uint32_t mid = lo + (uint32_t)(((uint64_t)hi - lo + 1) >> 1);
          unsigned long long sum = 0;
          for (int j = tid; j < n; j += ST) if (gl[j] >= mid) sum += gm[j];
          if (block_sum_u64(sum) > target) lo = mid; else hi = mid - 1;
        }
        thr = lo;
        p_done = true;
      }
    }
  } else if (cut >= 0) {
    for (int j = tid; j < n; j += ST) list[j] = w.cand[(size_t)b * w.capg + j];
    __syncthreads();
    if (wave == 0) {
      uint32_t kmin = 0xffffffffu;
      for (int j = lane; j < n; j += 64) kmin = min(kmin, list[j]);
      kmin = wave_reduce(kmin, [](uint32_t a, uint32_t b) { return min(a, b); });
      uint32_t t = kmin;
      if (need_k) {
        uint32_t lo = kmin, hi = key_m;                   // count(list >= lo) = n >= k
        while (lo < hi) {
          const uint32_t mid = lo + (uint32_t)(((uint64_t)hi - lo + 1) >> 1);
          int c = 0;
          for (int j0 = 0; j0 < n; j0 += 64) c += __popcll(__ballot(j0 + lane < n && list[min(j0 + lane, n - 1)] >= mid));
          if (c >= top_k) lo = mid; else hi = mid - 1;
        }
        t = lo;
      }
      bool p_ok = !need_p;
      if (need_p) {
        unsigned long long kept = 0;
        for (int j = lane; j < n; j += 64) {
          const unsigned long long mass = fixed_mass(key_value(list[j]), m);
          list_mass[j] = mass;
          if (list[j] >= t) kept += mass;
        }
        kept = wave_sum_u64(kept);                        // the mass of the list at and above the threshold so far
        const unsigned long long z = need_k ? kept : z_row;
        const unsigned long long target = (unsigned long long)((double)top_p * (double)z);
        if (kept > target) {                              // else the nucleus reaches below the list
          uint32_t lo = t, hi = key_m;
          while (lo < hi) {
            const uint32_t mid = lo + (uint32_t)(((uint64_t)hi - lo + 1) >> 1);
            unsigned long long sum = 0;
            for (int j = lane; j < n; j += 64) if (list[j] >= mid) sum += list_mass[j];
            sum = wave_sum_u64(sum);
            if (sum > target) lo = mid; else hi = mid - 1;
          }
          t = lo;
          p_ok = true;
        }
      }
      if (lane == 0) { found[0] = t; found[1] = 1; found[2] = p_ok; }
    }
    __syncthreads();
    if (found[1]) { k_done = true; if (found[2]) { p_done = true; thr = found[0]; } else if (need_k) thr = found[0]; }
  }
  return whole_row_threshold<VEC>(row, V, inv_t, m, key_m, thr, k_done, p_done, top_k, top_p, red, ired);
}

template <int VEC>
__global__ __launch_bounds__(ST) void row_threshold_kernel(const float* __restrict__ logits, SampleWork w, int V, float inv_t,
                                                           int top_k, float top_p) {
  __shared__ float red[16];
  __shared__ int ired[ST / 64];
  __shared__ uint32_t list[CAP];
  __shared__ unsigned long long list_mass[CAP];
  __shared__ int tot[NCUT];
  __shared__ unsigned long long z_sh[1 + NMC];
  const int b = blockIdx.x;
  const float m = row_max(w, b);
  const int cut = choose_cut(w, b, top_k > 0 && top_k < V, top_k, top_p, tot, z_sh);
  const uint32_t thr = list_threshold<VEC>(logits + (size_t)b * V, w, b, V, inv_t, m, cut, cut >= 0 ? min(tot[cut], w.capg) : 0, z_sh[0],
                                           top_k, top_p, list, list_mass, red, ired);
  if (threadIdx.x == 0) w.thr[b] = thr;
}

// The same for one row by one block, which counts and collects for itself: for the few rows with a small k whose lists
// of the one pass settle nothing.  Two passes over the row more than bisecting a list, thirty to sixty less than bisecting the row.
template <int VEC>
__device__ __forceinline__ uint32_t row_threshold_alone(const float* __restrict__ row, const SampleWork& w, int b, int V, float inv_t, float m,
                                                        int top_k, float top_p, uint32_t* list, unsigned long long* list_mass, float* red,
                                                        int* ired) {
  __shared__ int filled;
  const int tid = threadIdx.x, lane = tid & 63;
  int cnt[NCUT];
#pragma unroll
  for (int j = 0; j < NCUT; ++j) cnt[j] = 0;
  for_range<VEC, ST>(row, 0, V, inv_t, [&](int, float x, bool ok) {
    const float d = ok ? m - x : INFINITY;
#pragma unroll
    for (int j = 0; j < NCUT; ++j) cnt[j] += d <= kCut[j];
  });
  if (tid == 0) filled = 0;
  int cut = -1, n = 0;
  float dcut = 0.f;
#pragma unroll
  for (int j = 0; j < NCUT; ++j) {
    const int c = block_count(cnt[j], ired);
    if (cut == -1 && c >= top_k) {
      cut = c <= w.capg ? j : -2;
      n = c;
      dcut = kCut[j];
    }
  }
  if (cut >= 0) {
    uint32_t* out = w.cand + (size_t)b * w.capg;
    for_range<VEC, ST>(row, 0, V, inv_t, [&](int, float x, bool ok) {
      const bool in = ok && (m - x <= dcut);
      const unsigned long long mask = __ballot(in);
      if (mask) {
        const int leader = __ffsll((long long)mask) - 1;
        int base = 0;
        if (lane == leader) base = atomicAdd(&filled, __popcll(mask));
        base = __shfl(base, leader, 64);
        if (in) out[base + __popcll(mask & ((1ull << lane) - 1ull))] = order_key(x);
      }
    });
    __syncthreads();
  }
  return list_threshold<VEC>(row, w, b, V, inv_t, m, cut, n, 0ull, top_k, top_p, list, list_mass, red, ired);
}

// The kept mass of the row's tiles t, t + step, ... below t_end (a wave), and the last index with a positive probability
// in each (-1: none).
template <int VEC>
__device__ __forceinline__ void tile_sums(const float* __restrict__ row, const SampleWork& w, int b, int V, float inv_t, float m,
                                          uint32_t thr, int t, int t_end, int step) {
  const int lane = threadIdx.x & 63;
  for (; t < t_end; t += step) {
    float s = 0.f;
    int last_kept = -1;
    const int base = t * TILE;
    auto take = [&](int i, float x) {
      if (order_key(x) >= thr) {
        const float e = expf(x - m);
        s += e;
        if (e > 0.f) last_kept = max(last_kept, i);
      }
    };
    if constexpr (VEC == 4) {
      const float4* r4 = reinterpret_cast<const float4*>(row);
      const int G = V >> 2;
#pragma unroll 4
      for (int q = 0; q < TILE / 256; ++q) {
        const int g = base / 4 + q * 64 + lane;
        const float4 x = r4[min(g, G - 1)];
        if (g < G) { take(4 * g, x.x * inv_t); take(4 * g + 1, x.y * inv_t); take(4 * g + 2, x.z * inv_t); take(4 * g + 3, x.w * inv_t); }
      }
    } else {
      for (int i = base + lane; i < min(V, base + TILE); i += 64) take(i, row[i] * inv_t);
    }
    s = wave_sum(s);
    last_kept = wave_reduce(last_kept, [](int a, int b) { return max(a, b); });
    if (lane == 0) {
      w.tsum[(size_t)b * w.tiles + t] = s;
      w.tlast[(size_t)b * w.tiles + t] = last_kept;
    }
  }
}

// (wave v takes the chunk's tiles v, v + 4, ...)
template <int VEC>
__global__ __launch_bounds__(SB) void tile_sum_kernel(const float* __restrict__ logits, SampleWork w, int V, float inv_t,
                                                      int filtered) {
  const int b = blockIdx.y, c = blockIdx.x;
  tile_sums<VEC>(logits + (size_t)b * V, w, b, V, inv_t, row_max(w, b), filtered ? w.thr[b] : 0u,
                 c * w.tiles_per_chunk + (threadIdx.x >> 6), min(w.tiles, (c + 1) * w.tiles_per_chunk), SB / 64);
}

// The draw within the tile t_sel (-1: the row's last kept token) that the running sums chose, whose predecessors hold tile_before;
// e: the probabilities of the thread's four elements, 0 for what is not kept.
// All threads of a block of ST call it, pick: two ints in shared memory.
__device__ __forceinline__ void draw_in_tile(const float (&e)[4], int* __restrict__ out, int b, int t_sel, int last_of_row, float target,
                                             float tile_before, float* wred, int* pick) {
  const int tid = threadIdx.x;
  __syncthreads();
  if (t_sel < 0) {                                       // u * total rounded up to the total: the last kept token
    if (tid == 0) out[b] = max(last_of_row, 0);
    return;
  }
  if (tid == 0) { pick[0] = -1; pick[1] = -1; }
  const int base = t_sel * TILE + tid * 4;
  float mine = 0.f;
  int my_last = -1;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (e[j] > 0.f) my_last = base + j;
    mine += e[j];
  }
  float excl;
  const float incl = tile_before + block_inclusive_scan(mine, wred, &excl);
  const float before = tile_before + excl;
  if (my_last >= 0) atomicMax(&pick[1], my_last);
  if (target >= before && target < incl) {               // at most one thread: `before` is the thread before's `incl`
    float acc = before;
    int c = my_last;                                     // if rounding lets the run end early: its last positive one
    bool hit = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (!hit && e[j] > 0.f) {
        acc += e[j];
        if (target < acc) { c = base + j; hit = true; }
      }
    }
    pick[0] = c;
  }
  __syncthreads();
  // the tile's sum by waves and by the scan can differ in the last bit: past the scan's end means the tile's last
  if (tid == 0) out[b] = pick[0] >= 0 ? pick[0] : max(pick[1], 0);
}

// Inverse CDF in index order: the running sums of the tiles (one thread, in order), the tile in which the sum
// passes u times the total, and a scan of that tile, four consecutive elements per thread.
// All threads of a block of ST call it.
__device__ __forceinline__ void draw_from_tiles(const float* __restrict__ row, int* __restrict__ out, float u, const SampleWork& w, int b,
                                                int V, float inv_t, float m, uint32_t thr, float* wred) {
  __shared__ float prefix[1024];                          // inclusive running sums of up to 1024 tiles at a time
  __shared__ int pick[2];
  __shared__ float carry[2];
  const int tid = threadIdx.x;
  const float* tsum = w.tsum + (size_t)b * w.tiles;
  int last_kept = -1;
  for (int t = tid; t < w.tiles; t += ST) last_kept = max(last_kept, w.tlast[(size_t)b * w.tiles + t]);
  if (tid == 0) { pick[0] = -1; pick[1] = -1; carry[0] = 0.f; carry[1] = 0.f; }
  __syncthreads();
  atomicMax(&pick[1], last_kept);
  // the total first (groups of 1024 tiles), then the tile of the target
  for (int sweep = 0; sweep < 2; ++sweep) {
    const float target = u * carry[0];
    float before_group = 0.f;
    for (int t0 = 0; t0 < w.tiles; t0 += 1024) {
      const int n = min(w.tiles - t0, 1024);
      __syncthreads();
      for (int t = tid; t < n; t += ST) prefix[t] = tsum[t0 + t];
      __syncthreads();
      if (tid == 0) {
        float acc = before_group;
        for (int t = 0; t < n; ++t) { acc += prefix[t]; prefix[t] = acc; }
        if (sweep == 0) carry[0] = acc;
      }
      __syncthreads();
      if (sweep == 1 || w.tiles <= 1024) {
        const float tgt = sweep == 1 ? target : u * carry[0];
        for (int t = tid; t < n; t += ST) {
          const float lo = t == 0 ? before_group : prefix[t - 1];
          if (tgt >= lo && tgt < prefix[t]) { pick[0] = t0 + t; carry[1] = lo; }   // at most one tile
        }
      }
      before_group = prefix[n - 1];
    }
    if (w.tiles <= 1024) break;
  }
  __syncthreads();
  const int tile = pick[0];
  float e[4] = {0.f, 0.f, 0.f, 0.f};
  if (tile >= 0) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int i = tile * TILE + tid * 4 + j;
      if (i < V) {
        const float x = row[i] * inv_t;
        if (order_key(x) >= thr) e[j] = expf(x - m);
      }
    }
  }
  draw_in_tile(e, out, b, tile, pick[1], u * carry[0], carry[1], wred, pick);
}

// The rows' uniform numbers as the launch's own argument: no copy to the device, no buffer that has to outlive the call.
struct HeldUniforms {
  float v[ALICE_SAMPLE_HELD_ROWS];
  __device__ __forceinline__ float operator[](int b) const { return v[b]; }
};

// Uniforms: const float* in device memory, or HeldUniforms.
template <class Uniforms>
__global__ __launch_bounds__(ST) void draw_kernel(const float* __restrict__ logits, int* __restrict__ out,
                                                  const Uniforms uniform, SampleWork w, int V, float inv_t, int filtered) {
  __shared__ float wred[ST / 64];
  const int b = blockIdx.x;
  draw_from_tiles(logits + (size_t)b * V, out, uniform[b], w, b, V, inv_t, row_max(w, b), filtered ? w.thr[b] : 0u, wred);
}

// ---- top-k of up to TOPK_MOST in one pass over the row
//
//   chunk_topk   the chunk's elements in registers; the largest of every 256th part goes to shared memory, and one of these
//                that at least k reach (and at most (256 - k) / 16 more, ties apart) is a bound that at least k of the chunk's
//                elements reach: what reaches it (about -256 ln(1 - k/256) elements where the large ones are spread, and less than
//                topk_shape() expects) goes to the chunk's list with its index.  A chunk in which more do
//                (ties at the bound: masked elements, most often) lists what lies above it and names the key it left out.
//                Whatever the row's k largest are, ties among them included, they are in the lists if the k-th of what is
//                listed lies above every key that a chunk left out; and what was left out does not matter if its mass is zero.
//   row_topk     a block a row: the same bound once more over the lists' elements, then every survivor counts the larger ones
//                (the threshold of top-k) and adds up the mass at and above itself (top-p, the same fixed point); the sums of
//                the tiles from the kept elements alone, each lane's share in index order as tile_sum adds them (what it adds
//                for the others is zero), and the draw, in which the drawn tile is put together from the kept elements too.
//
// So a row is read once.  64 rows of 256,000, top-k 50, top-p 0.95: 15 + 12 us (22 + 23 before the bound was found by counting,
// and before all threads took part in what the survivors do; five passes over the row 103).  Back to back 8 rows take 19 us
// (32), one 17 (25), 64 of 32,768 16 (26).  The one pass takes 1.6 times its reads' time, row_topk the latency of some twenty
// phases, 0.5 us each, most of it for instructions that no launch before left in the CU's cache.  Rows that the lists do not settle (one that holds no number or no finite maximum, too many ties at the
// threshold itself) are counted and collected by their one block as the kernels for any k do it.  One row of 256,000 with 1,000 elements
// that are not masked: 22 us (32 before); with 5,120 ties at the top 168 (175; 41 by the five passes).
constexpr int TOPK_MOST = 200;       // beyond, the bound of 256 maxima lets too much through
constexpr int TOPK_LIST = 7168;      // elements of a row's lists in shared memory
constexpr int TOPK_LEFT = 1024;      // survivors
constexpr int TOPK_TILES = 128;      // tiles a row

struct TopkShape {
  int tiles, chunks, room;           // tiles a chunk, chunks a row, elements a chunk's list
};
// Fewer elements a chunk while 1,024 blocks are not reached and the lists' expected length fits; chunks of 0: not this way.
__host__ inline TopkShape topk_shape(int B, int tiles, int top_k, int capg) {
  if (top_k > TOPK_MOST || tiles > TOPK_TILES) return {0, 0, 0};
  const float expected = -256.f * logf(1.f - top_k / 256.f) * 1.1f + 16.f;
  int per = 1;
  while (per < 4 && ((long)B * ceil_div(tiles, per) > 1024 || ceil_div(tiles, per) * expected > 0.9f * TOPK_LIST)) per *= 2;
  const int chunks = ceil_div(tiles, per);
  if (chunks * expected > 0.9f * TOPK_LIST || expected * 1.1f > capg / chunks) return {0, 0, 0};
  return {per, chunks, capg / chunks};
}

// A bound that at least k (1 <= k <= 256) of 256 keys in shared memory reach, and few more where the keys are spread: bit by bit
// below what all keys have in common, by counting the lanes at and above, until k to k + (256 - k) / 16 are left, or (ties)
// the k-th largest itself.  It is one of the keys.  One wave's work: sixteen that did the same were in each other's way and took
// 4 us, every key against every other by four waves 2.9.
__device__ __forceinline__ uint32_t bound_of_256(const uint32_t* keys, int k, uint32_t* largest) {
  const uint4 v = reinterpret_cast<const uint4*>(keys)[threadIdx.x & 63];
  auto smaller = [](uint32_t a, uint32_t b) { return min(a, b); };
  const uint32_t hi = __builtin_amdgcn_readfirstlane(wave_reduce(max(max(v.x, v.y), max(v.z, v.w)), [](uint32_t a, uint32_t b) { return max(a, b); }));
  const uint32_t lo = __builtin_amdgcn_readfirstlane(wave_reduce(min(min(v.x, v.y), min(v.z, v.w)), smaller));
  *largest = hi;
  if (hi == lo) return hi;
  const int top = 31 - __builtin_clz(hi ^ lo), enough = k + (256 - k) / 16;
  uint32_t t = hi & ~((2u << top) - 1u);                   // all keys reach it
  for (int bit = top; bit >= 0; --bit) {
    const uint32_t c = t | (1u << bit);
    const int n = __popcll(__ballot(v.x >= c)) + __popcll(__ballot(v.y >= c)) + __popcll(__ballot(v.z >= c)) + __popcll(__ballot(v.w >= c));
    if (n < k) continue;
    t = c;
    if (n <= enough) break;
  }
  return wave_reduce(min(min(v.x >= t ? v.x : ~0u, v.y >= t ? v.y : ~0u), min(v.z >= t ? v.z : ~0u, v.w >= t ? v.w : ~0u)), smaller);
}

// 32 elements a thread, so that a CU holds all its blocks of a large step at once (with 64 and 256 threads a fourth
// block had to wait for a first: 64 rows of 256,000 took 22 us, and take 15).
template <int TILES>
constexpr int topk_threads() { return TILES == 4 ? 512 : 256; }

template <int VEC, int TILES>
__global__ __launch_bounds__(topk_threads<TILES>(), 6) void chunk_topk_kernel(const float* __restrict__ logits, SampleWork w, int V, float inv_t, int top_k,
                                                        TopkShape sh) {
  constexpr int NT = topk_threads<TILES>(), NE = TILES * TILE / NT;      // threads, elements a thread
  __shared__ __align__(16) uint32_t keys[256];
  __shared__ uint32_t wmin[NT / 64];
  __shared__ int fill, odd;
  const int b = blockIdx.y, c = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
  const float* row = logits + (size_t)b * V;
  const int lo = c * TILES * TILE, hi = min(V, lo + TILES * TILE);
  if (tid == 0) fill = odd = 0;
  auto index = [&](int e, int t) { return VEC == 4 ? lo + ((e >> 2) * NT + t) * 4 + (e & 3) : lo + e * NT + t; };
  float x[NE];
#pragma unroll
  for (int e = 0; e < NE; e += 4) {
    if constexpr (VEC == 4) {
      const float4 v = *reinterpret_cast<const float4*>(row + min(index(e, tid), V - 4));
      x[e] = v.x; x[e + 1] = v.y; x[e + 2] = v.z; x[e + 3] = v.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) x[e + i] = row[min(index(e + i, tid), V - 1)];
    }
  }
  uint32_t key[NE], most = 0;                              // 0: no element
  bool nan = false;
#pragma unroll
  for (int e = 0; e < NE; ++e) {
    const float v = x[e] * inv_t;
    nan = nan || v != v;                                   // (an element read twice at the row's end is looked at twice)
    key[e] = order_key(v);
  }
  if (hi - lo < TILES * TILE) {
    int t = tid;
    asm volatile("" : "+v"(t));
#pragma unroll
    for (int e = 0; e < NE; ++e) key[e] = index(e, t) < hi ? key[e] : 0u;
  }
#pragma unroll
  for (int e = 0; e < NE; ++e) most = max(most, key[e]);
  constexpr int PER = NT / 256;                            // threads a maximum
  if constexpr (PER >= 2) most = max(most, dpp_move<DPP_XOR1>(most));
  if constexpr (PER >= 4) most = max(most, dpp_move<DPP_XOR2>(most));
  if (tid % PER == 0) keys[tid / PER] = most;
  __syncthreads();
  if (nan) odd = 1;
  if (tid < 64) {
    uint32_t largest;
    const uint32_t from = bound_of_256(keys, top_k, &largest);
    if (tid == 0) wmin[0] = max(from, 1u);
  }
  lds_barrier();
  const uint32_t bound = wmin[0];
  unsigned long long* list = w.cmass + (size_t)b * w.capg + (size_t)c * sh.room;
  // What reaches a key goes to the list: a wave counts its elements, takes their places at once and fills them in turn.
  auto put = [&](uint32_t from) {
    int n = 0;
#pragma unroll
    for (int e = 0; e < NE; ++e) n += __popcll(__ballot(key[e] >= from));
    int at = 0;
    if (lane == 0 && n > 0) at = atomicAdd(&fill, n);
    at = __builtin_amdgcn_readfirstlane(at);
    asm volatile("" : "+v"(from));                         // (the masks of all elements are not kept: no registers for them)
#pragma unroll
    for (int e = 0; e < NE; ++e) {
      const unsigned long long mask = __ballot(key[e] >= from);
      if (mask == 0) continue;
      const int pos = at + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
      int at_index = tid;
      asm volatile("" : "+v"(at_index));                   // (nor their indices)
      if (key[e] >= from && pos < sh.room) list[pos] = ((unsigned long long)key[e] << 32) | (uint32_t)index(e, at_index);
      at += __popcll(mask);
    }
  };
  put(bound);
  lds_barrier();
  // More than there is room for (ties, most often those of masked elements, or large elements in few threads' places): what
  // lies above the bound alone, if that fits, else above the chunk's k-th largest; the ones tied with it are left out,
  // and the row is settled if its threshold lies above them.
  uint32_t tie = 0;
  int n = fill;
  if (n > sh.room) {
    __syncthreads();
    auto count = [&](uint32_t from) {                      // the chunk's elements at and above a key
      int k = 0;
#pragma unroll
      for (int e = 0; e < NE; ++e) k += key[e] >= from;
      k = wave_reduce(k, [](int a, int b) { return a + b; });
      if (lane == 0) wmin[tid >> 6] = (uint32_t)k;
      __syncthreads();
      k = 0;
      for (int x = 0; x < NT / 64; ++x) k += (int)wmin[x];
      __syncthreads();
      return k;
    };
    tie = bound;
    if (count(bound + 1) > sh.room) {
      uint32_t from = bound, to = 0xfffffffeu;             // at least top_k at and above `from`, fewer above `to`
      while (from < to) {
        const uint32_t mid = from + ((to - from) >> 1) + 1;
        if (count(mid) >= top_k) from = mid; else to = mid - 1;
      }
      tie = count(from) > sh.room ? from : from - 1;       // (all of them fit: nothing is left out but what is below)
    }
    if (tid == 0) fill = 0;
    __syncthreads();
    put(tie + 1);
    __syncthreads();
    n = fill;
  }
  if (tid == 0) {
    w.tlast[(size_t)b * w.tiles + c] = (odd || n > sh.room) ? -1 : n;
    w.tsum[(size_t)b * w.tiles + c] = __uint_as_float(tie);
  }
}

template <int VEC, class Uniforms>
__global__ __launch_bounds__(ST) void row_topk_kernel(const float* __restrict__ logits, int* __restrict__ out,
                                                      const Uniforms uniform, SampleWork w, int V, float inv_t, int top_k,
                                                      float top_p, TopkShape sh) {
  __shared__ __align__(16) unsigned long long list[TOPK_LIST];       // then the tiles' sums by lane and the drawn tile
  __shared__ __align__(16) uint32_t lkey[TOPK_LEFT + 4];             // the survivors; 0 up to a multiple of four
  __shared__ __align__(16) unsigned long long lmass[TOPK_LEFT + 4];
  __shared__ __align__(16) int lat[TOPK_LEFT + 4], lslot[TOPK_LEFT + 4];
  __shared__ __align__(16) uint32_t keys[256], wmin[ST / 64];
  __shared__ __align__(16) unsigned long long wsum[ST / 64];
  __shared__ int n_left, last_kept, rounds, pick[2];
  __shared__ __align__(16) float red[16], wred[ST / 64], tsum[TOPK_TILES];
  __shared__ float carry[2];
  __shared__ int ired[ST / 64];
  __shared__ uint32_t best;
  const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const float* row = logits + (size_t)b * V;
  const float u = uniform[b];
  // where the chunks' lists go, by every wave for itself: lane c has chunk c and 64 + c
  const int* counts = w.tlast + (size_t)b * w.tiles;
  const uint32_t* left_out = reinterpret_cast<const uint32_t*>(w.tsum + (size_t)b * w.tiles);
  const int c0 = lane < sh.chunks ? counts[lane] : 0, c1 = 64 + lane < sh.chunks ? counts[64 + lane] : 0;
  const uint32_t t0 = lane < sh.chunks ? left_out[lane] : 0u, t1 = 64 + lane < sh.chunks ? left_out[64 + lane] : 0u;
  if (tid < TOPK_TILES) tsum[tid] = 0.f;
  if (tid < 256) keys[tid] = 0;
  if (tid == 0) { n_left = 0; last_kept = -1; rounds = 0; best = 0; pick[0] = -1; pick[1] = -1; carry[1] = 0.f; }
  lds_barrier();                                           // (the counts are on their way)
  const uint32_t tie = wave_reduce(max(t0, t1), [](uint32_t a, uint32_t b) { return max(a, b); });
  bool settled = !__any(c0 < 0 || c1 < 0);
  auto scan = [&](int v) {
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int before = __shfl_up(v, o, 64);
      v += lane >= o ? before : 0;
    }
    return v;
  };
  const int s0 = scan(max(c0, 0)), s1 = sh.chunks > 64 ? scan(max(c1, 0)) : 0;
  const int n0 = __builtin_amdgcn_readlane(s0, 63), n = n0 + __builtin_amdgcn_readlane(s1, 63);
  settled = settled && n >= 1 && n <= TOPK_LIST;
  uint32_t key_m = 0;
  if (settled) {
    // the lists' elements, several waves a chunk where there are few; the bound again, from the largest of 256 groups.  A group
    // is by the place in all lists one after the other, not by the thread that moves an element: where not every wave has a chunk's
    // share (6, 9 .. 15 chunks) fewer threads than 4 k may move all, and a bound that every element reaches settles nothing.
    constexpr int NW = ST / 64;
    const int share = max(NW / sh.chunks, 1), sub = wave % share;
    for (int c = wave / share; c < sh.chunks; c += NW / share) {
      const int end = c < 64 ? __builtin_amdgcn_readlane(s0, c) : n0 + __builtin_amdgcn_readlane(s1, c - 64);
      const int len = c < 64 ? __builtin_amdgcn_readlane(c0, c) : __builtin_amdgcn_readlane(c1, c - 64);
      const unsigned long long* src = w.cmass + (size_t)b * w.capg + (size_t)c * sh.room;
      for (int i = sub * 64 + lane; i < len; i += share * 64) {
        const unsigned long long el = src[i];
        list[end - len + i] = el;
        atomicMax(&keys[(end - len + i) / 4 % 256], (uint32_t)(el >> 32));
      }
    }
    __syncthreads();
    if (wave == 0) {
      uint32_t largest;
      const uint32_t from = bound_of_256(keys, top_k, &largest);
      if (lane == 0) { wmin[0] = from; wmin[1] = largest; }
    }
    __syncthreads();
    const uint32_t bound = wmin[0];
    key_m = wmin[1];
    for (int i = tid; i < n; i += ST)
      if ((uint32_t)(list[i] >> 32) >= bound) {
        const int pos = atomicAdd(&n_left, 1);
        if (pos < TOPK_LEFT) {
          lkey[pos] = (uint32_t)(list[i] >> 32);
          lat[pos] = (int)(uint32_t)list[i];
        }
      }
    __syncthreads();
    settled = n_left <= TOPK_LEFT && fabsf(key_value(key_m)) < INFINITY;
  }
  // 2^split threads a survivor look at the others, so that all 1,024 have work (a thread a survivor: of the 23 us that this
  // kernel took 12 went into a few waves' loops over the others)
  float m = 0.f;
  int nl = 0, quads = 0, at = 0, split = 0, who = 0, part = 0;
  uint32_t key = 0, thr = 0xffffffffu;
  unsigned long long z = 0;
  bool kept_k = false, first = false;                      // first: of the threads of a survivor
  auto all_parts = [&](uint32_t v) {                       // their sum, in all of them
    if (split >= 1) v += dpp_move<DPP_XOR1>(v);
    if (split >= 2) v += dpp_move<DPP_XOR2>(v);
    if (split >= 3) v += dpp_move<DPP_HALF_MIRROR>(v);     // (the quads of 8 lanes are uniform by now)
    return v;
  };
  if (settled) {
    m = key_value(key_m);
    nl = n_left;
    quads = (nl + 3) >> 2;
    split = nl <= ST / 8 ? 3 : nl <= ST / 4 ? 2 : nl <= ST / 2 ? 1 : 0;
    who = tid >> split;
    part = tid & ((1 << split) - 1);
    first = part == 0 && who < nl;
    key = who < nl ? lkey[who] : 0u;
    at = who < nl ? lat[who] : 0;
    if (tid >= nl && tid < quads * 4) { lkey[tid] = 0; lmass[tid] = 0; lslot[tid] = -1; lat[tid] = 0; }
    __syncthreads();
    uint32_t larger = 0;
    if (who < nl) {
#pragma unroll 4
      for (int j = part; j < quads; j += 1 << split) {
        const uint4 o = reinterpret_cast<const uint4*>(lkey)[j];
        larger += (o.x > key) + (o.y > key) + (o.z > key) + (o.w > key);
      }
    }
    larger = all_parts(larger);
    kept_k = who < nl && (int)larger < top_k;
    if (kept_k) thr = key;
    thr = wave_reduce(thr, [](uint32_t a, uint32_t b) { return min(a, b); });
    const unsigned long long mass = kept_k && first ? fixed_mass(key_value(key), m) : 0ull;
    const unsigned long long z_wave = wave_sum_u64(mass);
    if (first) lmass[who] = mass;
    if (lane == 0) { wmin[wave] = thr; wsum[wave] = z_wave; }
    __syncthreads();
#pragma unroll
    for (int x = 0; x < ST / 64; ++x) { thr = min(thr, wmin[x]); z += wsum[x]; }
    // what was left out is not among the k largest, or its mass is zero
    settled = tie == 0 || (nl >= top_k && thr > tie) || expf(key_value(tie) - m) == 0.f;
  }
  if (!settled) {
    float lmax = -INFINITY;
    for_range<VEC, ST>(row, 0, V, inv_t, [&](int, float x, bool ok) { lmax = fmaxf(lmax, ok ? x : -INFINITY); });
    const float m = block_max(lmax, red);
    static_assert(TOPK_LIST >= CAP + CAP / 2, "the lists of the bisection take the place of the chunks' lists");
    const uint32_t thr = row_threshold_alone<VEC>(row, w, b, V, inv_t, m, top_k, top_p, reinterpret_cast<uint32_t*>(list + CAP), list, red, ired);
    __syncthreads();
    tile_sums<VEC>(row, w, b, V, inv_t, m, thr, wave, w.tiles, ST / 64);
    __syncthreads();
    draw_from_tiles(row, out, u, w, b, V, inv_t, m, thr, wred);
    return;
  }
  float* lanes = reinterpret_cast<float*>(list);           // [tiles][64]: the tiles' sums by lane, then the drawn tile's elements
  static_assert(sizeof(list) >= (TOPK_TILES * 64 + TILE) * sizeof(float) && TILE == 4 * ST, "both lie where the lists were");
  float4* drawn = reinterpret_cast<float4*>(lanes + TOPK_TILES * 64);
  for (int i = tid; i < w.tiles * 16; i += ST) reinterpret_cast<float4*>(lanes)[i] = float4{0.f, 0.f, 0.f, 0.f};
  drawn[tid] = float4{0.f, 0.f, 0.f, 0.f};
  if (top_p < 1.f) {
    // the largest key at and above which lies more than the target
    const unsigned long long target = (unsigned long long)((double)top_p * (double)z);
    unsigned long long above = 0;
    if (kept_k) {
#pragma unroll 2
      for (int j = part; j < quads; j += 1 << split) {
        const uint4 o = reinterpret_cast<const uint4*>(lkey)[j];
        const ulonglong2 m0 = reinterpret_cast<const ulonglong2*>(lmass)[2 * j], m1 = reinterpret_cast<const ulonglong2*>(lmass)[2 * j + 1];
        above += (o.x >= key ? m0.x : 0ull) + (o.y >= key ? m0.y : 0ull) + (o.z >= key ? m1.x : 0ull) + (o.w >= key ? m1.y : 0ull);
      }
    }
    // (three pieces of 21 bits and one more: their sums over eight parts stay below 32 bits)
    unsigned long long sum = 0;
#pragma unroll
    for (int p = 0; p < 64; p += 21) sum += (unsigned long long)all_parts((uint32_t)(above >> p) & 0x1fffffu) << p;
    if (kept_k && first && sum > target) atomicMax(&best, key);
    __syncthreads();
    thr = best;
  }
  // the tiles' sums: a lane of tile_sum adds its elements in index order
  const bool kept = who < nl && key >= thr;
  const float e = kept ? expf(key_value(key) - m) : 0.f;
  const int slot = (at / TILE) * 64 + (VEC == 4 ? (at >> 2) & 63 : at & 63);
  if (first) lslot[who] = kept ? slot : -1;
  __syncthreads();
  uint32_t turn = 0;                                       // kept elements of the same lane before this one
  if (kept) {
#pragma unroll 2
    for (int j = part; j < quads; j += 1 << split) {
      const int4 o = reinterpret_cast<const int4*>(lslot)[j], i = reinterpret_cast<const int4*>(lat)[j];
      turn += ((o.x == slot) & (i.x < at)) + ((o.y == slot) & (i.y < at)) + ((o.z == slot) & (i.z < at)) + ((o.w == slot) & (i.w < at));
    }
  }
  turn = all_parts(turn);
  if (kept && first) {
    if (e > 0.f) atomicMax(&last_kept, at);
    atomicMax(&rounds, (int)turn + 1);
  }
  __syncthreads();
  const int n_rounds = rounds;
  for (int r = 0; r < n_rounds; ++r) {
    if (kept && first && (int)turn == r) lanes[slot] += e;
    __syncthreads();
  }
  for (int t = wave; t < w.tiles; t += ST / 64) {
    const float s = wave_sum(lanes[t * 64 + lane]);
    if (lane == 0) tsum[t] = s;
  }
  __syncthreads();
  // their running sums in order: every thread adds up what lies before its tile and zeros, all in registers at once
  float total = 0.f, before = 0.f;
  const int mine = tid & (TOPK_TILES - 1);
#pragma unroll
  for (int t0 = 0; t0 < TOPK_TILES; t0 += 64) {
    if (t0 >= w.tiles) break;
    float4 s[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) s[t] = reinterpret_cast<const float4*>(tsum + t0)[t];
#pragma unroll
    for (int t = 0; t < 64; ++t) {
      const float x = reinterpret_cast<const float*>(s)[t];
      total += x;
      before += t0 + t < mine ? x : 0.f;
    }
  }
  const float target = u * total;
  if (tid < w.tiles && target >= before && target < before + tsum[tid]) { pick[0] = tid; carry[1] = before; }      // at most one tile
  __syncthreads();
  const int tile = pick[0];
  if (kept && first && at / TILE == tile) reinterpret_cast<float*>(drawn)[at & (TILE - 1)] = e;
  __syncthreads();
  const float4 own = drawn[tid];
  const float ex[4] = {own.x, own.y, own.z, own.w};
  draw_in_tile(ex, out, b, tile, last_kept, target, carry[1], wred, pick);
}

// How long a row's list may be: 32,768 candidates, fewer (down to what fits shared memory) when the lists of
// all rows would take more than 200 MB.
__host__ inline int list_room(int B) {
  long room = (16L << 20) / (B > 0 ? B : 1);
  return (int)(room > CAPG ? CAPG : (room < CAP ? CAP : room));
}

// chunks, tiles and tiles per chunk of a call
__host__ inline void sample_shape(int B, int V, int* chunks, int* tiles, int* per) {
  *tiles = (V + TILE - 1) / TILE;
  *per = ((long)B * *tiles + 1023) / 1024;
  if (*per < 1) *per = 1;
  *chunks = (*tiles + *per - 1) / *per;
}

}  // namespace

// How many chunks a row is cut into; the workspace holds B * chunks floats and as many ints, which is never more
// than ALICE_ARGMAX_MAX_PARTIALS of each: the bound that sizes the static workspace of alice_argmax_static.
extern "C" int alice_argmax_chunks(int B, int V) {
  if (V < 16384) return 1;
  int c = ALICE_ARGMAX_MAX_PARTIALS / (B > 0 ? B : 1);
  if (c > V / 8192) c = V / 8192;
  return c < 2 ? 1 : (c > 64 ? 64 : c);
}

extern "C" int alice_argmax(const float* logits, int* out, float* work_v, int* work_i, int B, int V, hipStream_t stream) {
  ALICE_CHECK(B >= 0 && V >= 1, "argmax: bad sizes B=%d V=%d", B, V);
  if (B == 0) return 0;
  const int chunks = alice_argmax_chunks(B, V);
  ALICE_CHECK(chunks == 1 || (work_v && work_i), "argmax: the workspace is missing");
  ALICE_CHECK(B <= 65535 * 32, "argmax: too many rows");
  if (chunks == 1) {
    argmax_kernel<<<dim3(B, 1), ST, 0, stream>>>(logits, nullptr, out, nullptr, nullptr, V, 1);
  } else {
    argmax_kernel<<<dim3(B, chunks), ST, 0, stream>>>(logits, nullptr, out, work_v, work_i, V, chunks);
    ALICE_LAUNCH_CHECK();
    argmax_kernel<<<dim3(B, 1), ST, 0, stream>>>(work_v, work_i, out, nullptr, nullptr, chunks, 1);
  }
  ALICE_LAUNCH_CHECK();
  return 0;
}

// ---- argmax without a workspace argument
//
// The chunk maxima of the two-stage argmax live in a file-scope device array instead of a buffer that the caller
// allocates.  Every GPU holds its own copy of the array at its own address, which the host learns once per
// device from hipGetSymbolAddress (in host code the array's name is only a stand-in, not a device address).
// Nothing in the array has to start at zero: stage one writes every pair that stage two reads.
static_assert(ALICE_ARGMAX_STATIC_MAX_PAIRS >= ALICE_ARGMAX_MAX_PARTIALS,
              "the static workspace must hold what the chunk rule can ask for");
static __device__ __align__(256) unsigned char argmax_scratch[ALICE_ARGMAX_STATIC_MAX_PAIRS * 8];

namespace {
constexpr int MAX_DEVICES = 64;
void* g_argmax_scratch_ptr[MAX_DEVICES] = {};       // per device, set once; a pointer store is atomic on the host

// The address of the current device's copy of the array; nullptr (and the error set) on failure.
void* argmax_scratch_of_current_device() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    alice_set_error("argmax (static): no current device, or a device number beyond %d", MAX_DEVICES - 1);
    return nullptr;
  }
  void* p = __atomic_load_n(&g_argmax_scratch_ptr[dev], __ATOMIC_ACQUIRE);
  if (p) return p;
  hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(argmax_scratch));
  if (e != hipSuccess || !p) {
    alice_set_error("argmax (static): hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(e));
    return nullptr;
  }
  __atomic_store_n(&g_argmax_scratch_ptr[dev], p, __ATOMIC_RELEASE);   // two threads racing here store the same address
  return p;
}
}  // namespace

extern "C" int alice_argmax_static_init() { return argmax_scratch_of_current_device() ? 0 : 1; }

extern "C" int alice_argmax_static(const float* logits, int* out, int B, int V, hipStream_t stream) {
  ALICE_CHECK(B >= 0 && V >= 1, "argmax: bad sizes B=%d V=%d", B, V);
  if (B == 0) return 0;
  ALICE_CHECK(logits && out, "argmax (static): logits and out must be given");
  ALICE_CHECK(B <= 65535 * 32, "argmax: too many rows");
  const int chunks = alice_argmax_chunks(B, V);
  if (chunks == 1) {
    argmax_kernel<<<dim3(B, 1), ST, 0, stream>>>(logits, nullptr, out, nullptr, nullptr, V, 1);
    ALICE_LAUNCH_CHECK();
    return 0;
  }
  ALICE_CHECK((long)B * chunks <= ALICE_ARGMAX_STATIC_MAX_PAIRS,
              "argmax (static): %d rows in %d chunks need %ld partial results, the static workspace holds %d",
              B, chunks, (long)B * chunks, ALICE_ARGMAX_STATIC_MAX_PAIRS);
  void* scratch = argmax_scratch_of_current_device();
  if (!scratch) return 1;
  float* work_v = reinterpret_cast<float*>(scratch);
  int* work_i = reinterpret_cast<int*>(reinterpret_cast<unsigned char*>(scratch) + (size_t)ALICE_ARGMAX_STATIC_MAX_PAIRS * 4);
  argmax_kernel<<<dim3(B, chunks), ST, 0, stream>>>(logits, nullptr, out, work_v, work_i, V, chunks);
  ALICE_LAUNCH_CHECK();
  argmax_kernel<<<dim3(B, 1), ST, 0, stream>>>(work_v, work_i, out, nullptr, nullptr, chunks, 1);
  ALICE_LAUNCH_CHECK();
  return 0;
}

// Number of 32-bit words of workspace a call needs.
extern "C" long alice_sample_workspace(int B, int V) {
  int chunks, tiles, per;
  sample_shape(B > 0 ? B : 1, V, &chunks, &tiles, &per);
  const long rows = B > 0 ? B : 1;
  // pmass and cmass first (8-byte elements), then the 4-byte arrays
  const long capg = list_room(B);
  return rows * chunks * 2 * (1 + NMC) + rows * capg * 2 + rows * chunks + rows * chunks * NCUT + rows * capg + rows + rows * tiles * 2 + 16;
}

namespace {
template <class Uniforms>
int sample_launch(const float* logits, int* out, const Uniforms& uniform, void* work, int B, int V, float temperature, int top_k,
                  float top_p, hipStream_t stream) {
  ALICE_CHECK(B >= 0 && V >= 1, "sample: bad sizes B=%d V=%d", B, V);
  ALICE_CHECK(temperature > 0.f, "sample: temperature must be positive (use argmax for greedy)");
  ALICE_CHECK(top_k >= 0 && top_p > 0.f, "sample: top_k must not be negative and top_p must be positive");
  ALICE_CHECK(B <= 65535, "sample: %d rows are more than one launch takes", B);
  ALICE_CHECK(work != nullptr && ((uintptr_t)work & 7) == 0, "sample: the workspace is missing or not 8-byte aligned");
  if (B == 0) return 0;
  SampleWork w;
  sample_shape(B, V, &w.chunks, &w.tiles, &w.tiles_per_chunk);
  w.capg = list_room(B);
  const size_t rows = (size_t)B;
  w.pmass = (unsigned long long*)work;
  w.cmass = w.pmass + rows * w.chunks * (1 + NMC);
  w.pmax = (float*)(w.cmass + rows * w.capg);
  w.pcnt = (int*)(w.pmax + rows * w.chunks);
  w.cand = (uint32_t*)(w.pcnt + rows * w.chunks * NCUT);
  w.thr = w.cand + rows * w.capg;
  w.tsum = (float*)(w.thr + rows);
  w.tlast = (int*)(w.tsum + rows * w.tiles);
  const float inv_t = 1.f / temperature;
  const bool need_k = top_k > 0 && top_k < V, need_p = top_p < 1.f;
  const int filtered = need_k || need_p;
  const bool vec = V % 4 == 0 && ((uintptr_t)logits & 15) == 0;
  if (need_k) {                                            // a small k: the row is read once
    const TopkShape sh = topk_shape(B, w.tiles, top_k, w.capg);
    if (sh.chunks > 0) {
#define GO(VEC)                                                                                             \
  do {                                                                                                      \
    const dim3 grid(sh.chunks, B);                                                                          \
    if (sh.tiles == 4) chunk_topk_kernel<VEC, 4><<<grid, topk_threads<4>(), 0, stream>>>(logits, w, V, inv_t, top_k, sh);  \
    else if (sh.tiles == 2) chunk_topk_kernel<VEC, 2><<<grid, topk_threads<2>(), 0, stream>>>(logits, w, V, inv_t, top_k, sh); \
    else chunk_topk_kernel<VEC, 1><<<grid, topk_threads<1>(), 0, stream>>>(logits, w, V, inv_t, top_k, sh);                \
    ALICE_LAUNCH_CHECK();                                                                                   \
    row_topk_kernel<VEC><<<B, ST, 0, stream>>>(logits, out, uniform, w, V, inv_t, top_k, top_p, sh);        \
  } while (0)
      if (vec) GO(4); else GO(1);
#undef GO
      ALICE_LAUNCH_CHECK();
      return 0;
    }
  }
  const dim3 cgrid(w.chunks, B);
#define GO(VEC)                                                                                                             \
  do {                                                                                                                      \
    chunk_max_kernel<VEC><<<cgrid, SB, 0, stream>>>(logits, w, V, inv_t);                                                   \
    if (filtered) {                                                                                                         \
      chunk_count_kernel<VEC><<<cgrid, SB, 0, stream>>>(logits, w, V, inv_t, need_k ? 0 : 1);                               \
      chunk_collect_kernel<VEC><<<cgrid, SB, 0, stream>>>(logits, w, V, inv_t, top_k, top_p);                                   \
      row_threshold_kernel<VEC><<<B, ST, 0, stream>>>(logits, w, V, inv_t, top_k, top_p);                                   \
    }                                                                                                                       \
    tile_sum_kernel<VEC><<<cgrid, SB, 0, stream>>>(logits, w, V, inv_t, filtered);                                          \
  } while (0)
  if (vec) GO(4); else GO(1);
#undef GO
  ALICE_LAUNCH_CHECK();
  draw_kernel<<<B, ST, 0, stream>>>(logits, out, uniform, w, V, inv_t, filtered);
  ALICE_LAUNCH_CHECK();
  return 0;
}

uint64_t splitmix64(uint64_t x) {
  x += 0x9E3779B97F4A7C15ull;
  uint64_t z = x;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}
}  // namespace

extern "C" int alice_sample(const float* logits, int* out, const float* uniform, void* work, int B, int V,
                            float temperature, int top_k, float top_p, hipStream_t stream) {
  return sample_launch(logits, out, uniform, work, B, V, temperature, top_k, top_p, stream);
}

// The same for at most ALICE_SAMPLE_HELD_ROWS rows, row i with the draws[i]-th uniform number of request requests[i] under
// `seed` (host arrays; read before the call returns).  Against numbers made as an array, copied through a pinned buffer and
// read from device memory, 64 rows of 256,000: the host's part of a call 36 -> 12 us, and a copy fewer on the stream.
extern "C" int alice_sample_drawn(const float* logits, int* out, unsigned long long seed, const unsigned long long* requests,
                                  const unsigned long long* draws, void* work, int B, int V, float temperature, int top_k, float top_p,
                                  hipStream_t stream) {
  ALICE_CHECK(B >= 0 && B <= ALICE_SAMPLE_HELD_ROWS, "sample: %d rows are more than a launch holds the uniform numbers of", B);
  ALICE_CHECK(B == 0 || (requests && draws), "sample: the rows' requests or draws are missing");
  HeldUniforms u = {};
  for (int i = 0; i < B; ++i) {
    const uint64_t row = splitmix64(seed ^ (requests[i] * 0xD1B54A32D192ED03ull));
    u.v[i] = (float)(splitmix64(row + draws[i]) >> 40) / (float)(1 << 24);             // 24 bits: exact
  }
  return sample_launch(logits, out, u, work, B, V, temperature, top_k, top_p, stream);
}
