// Attention of single tokens over a row-major paged cache with the masks and softmax terms of
// alice_attention_masked, the keys split over blocks: 32-bit arithmetic on operands of either dtype (the decode kernel
// of the mixers that the matrix-core decode kernel does not take, and of the true 32-bit path).
//
// A block takes one token, one kv head and one run of 256 visible keys, a wave 32 of them.  A key row is read by as many lanes as
// it has pieces of 16 bytes, so that a wave's load covers whole rows (a lane a row, each load touching 64 lines of which it used
// 16 bytes, moved them several times); a lane holds its piece of the group's queries in registers, its partial products meet
// by lane moves, and the key row serves the whole group.  The block's maximum and sum a head come from two barriers; then the
// threads turn to the values: a thread owns 16 bytes of the value row's width for a share of the keys, with one accumulator set
// a head, eight loads on their way at a time and the first eight asked for before the scores; the shares meet by lane
// moves and through LDS, four heads at a time.  With per-value-head outputs the second phase runs once for every kv head's values.
// Each block leaves (maximum, sum, unnormalised output) per head; attn_split_combine_kernel merges the runs in their order, adds the
// sink to the denominator, turns the output back where the values were cached turned, applies gate and factor, and writes the
// result (or the per-value-head outputs in float32 for the mix of the heads that follows).
// Eight sequences of 500 to 1,500 keys, 16 heads on 4 kv heads of 128 in bfloat16: 25 us before, 12 now, of which reading is 3:
// what bounds it is the chain of waits (place, key, score, maximum, sum, value), one block on a CU.
#include "common.h"
#include "alice_hip.h"

namespace {

constexpr int KEYS = 256;
constexpr int WAVES = 8, NT = 64 * WAVES, WKEYS = KEYS / WAVES;      // of a block; keys a wave scores

struct SplitArgs {
  const int* positions;
  const int* seq_of_token;
  const int* block_table;
  int bt_stride, nH, nKV, d, dv, page_size;
  float scale;
  int window, chunk, keep_first, n_splits, value_heads;
  const float* slopes;
  float* part_ml;      // [T, nH, splits, 2]
  float* part_o;       // [T, nH, value heads (or 1), splits, dv]
};

template <typename T> __device__ __forceinline__ void unpack16(const uint4& w, float* f);
template <> __device__ __forceinline__ void unpack16<float>(const uint4& w, float* f) {
  f[0] = __uint_as_float(w.x); f[1] = __uint_as_float(w.y); f[2] = __uint_as_float(w.z); f[3] = __uint_as_float(w.w);
}
template <> __device__ __forceinline__ void unpack16<bf16_t>(const uint4& w, float* f) {
  const uint32_t v[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf16_bits_to_f32(v[i] & 0xffffu);
    f[2 * i + 1] = bf16_bits_to_f32(v[i] >> 16);
  }
}

template <int CTRL>
__device__ __forceinline__ float lane_move(float v) { return __uint_as_float(dpp_move<CTRL>(__float_as_uint(v))); }
// v and the value of the lane 16 (32) away, added
__device__ __forceinline__ float sum_over_16(float v) {
  auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(x[0]) + __uint_as_float(x[1]);
}
__device__ __forceinline__ float sum_over_32(float v) {
  auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(x[0]) + __uint_as_float(x[1]);
}

// (128 registers let a second block work while one waits; the widest groups need more)
// U: loads of keys, of values on their way at a time, no more than a wave has of its rows.
template <typename T, int PER, int U>
__global__ __launch_bounds__(NT, PER <= 8 ? 4 : 2) void attn_split_kernel(const T* __restrict__ q, const T* __restrict__ k_pool,
                                                            const T* __restrict__ v_pool, SplitArgs a) {
  constexpr bool FULL = sizeof(T) == 4;
  constexpr int VEC = 16 / sizeof(T);
  constexpr int HG = PER < 4 ? PER : 4;               // heads that meet in LDS at a time
  constexpr int UK = U, UV = U;
  constexpr int OWN = PER >= 4 ? PER / 4 : 1;         // heads of a key whose sums a lane ends up with
  __shared__ float ps[PER][KEYS];
  __shared__ int rows_of[KEYS];                       // the row of each of the block's keys in kv head 0's part of its page
  __shared__ float wred[WAVES][PER];
  __shared__ __align__(16) float ored[WAVES][HG][256];

  const int t = blockIdx.x, kvh = blockIdx.y, split = blockIdx.z, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = a.d, dv = a.dv, per = a.nH / a.nKV, h0 = kvh * per;
  const int n_vh = a.value_heads > 0 ? a.value_heads : 1;
  const int pos = a.positions[t];
  const int* bt = a.block_table + (size_t)a.seq_of_token[t] * a.bt_stride;
  const int start = a.chunk > 0 ? (pos / a.chunk) * a.chunk : (a.window > 0 ? max(0, pos + 1 - a.window) : 0);
  const int n_first = (a.keep_first > 0 && a.window > 0 && a.chunk == 0) ? min(a.keep_first, start) : 0;
  const int n_keys = n_first + pos + 1 - start;
  const int v0 = split * KEYS, nk = max(0, min(KEYS, n_keys - v0));
  if (nk == 0) {                                      // a run behind this token's keys
    for (int i = tid; i < per; i += NT) {
      float* ml = a.part_ml + (((size_t)t * a.nH + h0 + i) * a.n_splits + split) * 2;
      ml[0] = -INFINITY;
      ml[1] = 0.f;
    }
    for (int i = tid; i < per * n_vh * dv; i += NT)
      a.part_o[(((size_t)t * a.nH + h0) * n_vh + i / dv) * a.n_splits * dv + (size_t)split * dv + i % dv] = 0.f;
    return;
  }
  // this thread's key
  const bool has = tid < nk;
  const int vi = v0 + tid;
  const int kp = has ? (vi < n_first ? vi : start + (vi - n_first)) : 0;
  if (has) rows_of[tid] = bt[kp / a.page_size] * a.nKV * a.page_size + kp % a.page_size;
  // this lane's piece of the group's queries (zero beyond the group and beside the row)
  const int EK = d / VEC;
  int row_log = 2;                                    // lanes a row: a power of two, at least 4
  while ((1 << row_log) < EK) ++row_log;
  const int piece = lane & ((1 << row_log) - 1), key_of = lane >> row_log, KL = 64 >> row_log;
  const bool in_row = piece < EK;
  const int k_at = min(piece, EK - 1) * VEC;
  float qf[PER][VEC];
#pragma unroll
  for (int hh = 0; hh < PER; ++hh) {
    const uint4 w = *reinterpret_cast<const uint4*>(q + ((size_t)t * a.nH + h0 + min(hh, per - 1)) * d + k_at);
    unpack16<T>(w, qf[hh]);
#pragma unroll
    for (int e = 0; e < VEC; ++e) qf[hh][e] = in_row && hh < per ? qf[hh][e] : 0.f;
  }
  __syncthreads();
  // Loads are clamped to the block's keys, not left out: what a branch surrounds the compiler waits for at its end.
  const int key0 = wave * WKEYS, all_loads = WKEYS >> (6 - row_log);
  const int loads = nk > key0 ? min((nk - key0 + KL - 1) >> (6 - row_log), all_loads) : 0;
  auto load_keys = [&](uint4 (&w)[UK], int j) {
#pragma unroll
    for (int u = 0; u < UK; ++u) {
      const int i = min(key0 + min(j + u, all_loads - 1) * KL + key_of, nk - 1);
      w[u] = *reinterpret_cast<const uint4*>(k_pool + ((size_t)rows_of[i] + (size_t)kvh * a.page_size) * d + k_at);
    }
  };
  const int EC = dv / VEC;
  int EC2 = 1;
  while (EC2 < EC) EC2 <<= 1;
  const int KG = NT / EC2, ec = tid & (EC2 - 1), kg = tid / EC2;
  auto load_values = [&](uint4 (&w)[UV], int z, int i0) {    // of the keys i0 + kg, i0 + kg + KG, ..
    const int vh = a.value_heads > 0 ? z : kvh, at = min(ec, EC - 1) * VEC;
#pragma unroll
    for (int u = 0; u < UV; ++u)
      w[u] = *reinterpret_cast<const uint4*>(v_pool + ((size_t)rows_of[min(i0 + u * KG + kg, nk - 1)] + (size_t)vh * a.page_size) * dv + at);
  };
  uint4 kw[UK], vw[UV];
  load_keys(kw, 0);
  load_values(vw, 0, 0);
  // A lane's partial products meet over the row's lanes: over the first two distances each lane keeps half of the heads and hands
  // the other half over, then every lane's own heads are summed over the rest.
  const bool odd1 = lane & 1, odd2 = lane & 2;
  const int own0 = PER >= 4 ? (odd1 ? PER / 2 : 0) + (odd2 ? PER / 4 : 0) : PER == 2 && odd1 ? 1 : 0;
  auto score_keys = [&](const uint4 (&w)[UK], int j) {
    float sum[UK][OWN];
#pragma unroll
    for (int u = 0; u < UK; ++u) {
      const uint4 x = in_row ? w[u] : uint4{0u, 0u, 0u, 0u};
      float kf[VEC], dot[PER];
      unpack16<T>(x, kf);
#pragma unroll
      for (int hh = 0; hh < PER; ++hh) {
        dot[hh] = qf[hh][0] * kf[0];
#pragma unroll
        for (int e = 1; e < VEC; ++e) dot[hh] = fmaf(qf[hh][e], kf[e], dot[hh]);
      }
      if constexpr (PER >= 2) {
#pragma unroll
        for (int i = 0; i < PER / 2; ++i) {
          const float mine = odd1 ? dot[i + PER / 2] : dot[i], other = odd1 ? dot[i] : dot[i + PER / 2];
          dot[i] = mine + lane_move<DPP_XOR1>(other);
        }
      } else {
        dot[0] += lane_move<DPP_XOR1>(dot[0]);
      }
      if constexpr (PER >= 4) {
#pragma unroll
        for (int i = 0; i < PER / 4; ++i) {
          const float mine = odd2 ? dot[i + PER / 4] : dot[i], other = odd2 ? dot[i] : dot[i + PER / 4];
          dot[i] = mine + lane_move<DPP_XOR2>(other);
        }
      } else {
        dot[0] += lane_move<DPP_XOR2>(dot[0]);
      }
#pragma unroll
      for (int i = 0; i < OWN; ++i) sum[u][i] = dot[i];
    }
    auto meet = [&](auto partner_sum) {
#pragma unroll
      for (int u = 0; u < UK; ++u)
#pragma unroll
        for (int i = 0; i < OWN; ++i) sum[u][i] = partner_sum(sum[u][i]);
    };
    if (row_log == 3) {
      meet([](float v) { return v + lane_move<DPP_ROR12>(v); });                          // (from the lane 4 on: right in the row's first four)
    } else if (row_log >= 4) {
      meet([](float v) { v += lane_move<DPP_ROR8>(v); return v + lane_move<DPP_ROR4>(v); });
    }
    if (row_log >= 5) meet([](float v) { return sum_over_16(v); });
    if (row_log >= 6) meet([](float v) { return sum_over_32(v); });
    if (piece < 4) {
#pragma unroll
      for (int u = 0; u < UK; ++u) {
        if (j + u >= loads) break;
#pragma unroll
        for (int i = 0; i < OWN; ++i) ps[own0 + i][key0 + (j + u) * KL + key_of] = sum[u][i];
      }
    }
  };
  for (int j = 0; j < loads; j += UK) {
    score_keys(kw, j);
    if (j + UK < loads) load_keys(kw, j + UK);
  }
  lds_barrier();
  // scores, the block's maximum a head, the weights and their sum
  float sc[PER];
#pragma unroll
  for (int hh = 0; hh < PER; ++hh) {
    float s = has ? ps[hh][tid & (KEYS - 1)] * a.scale : 0.f;
    if (a.slopes && hh < per) s = fmaf(a.slopes[h0 + hh], (float)(kp - pos), s);
    sc[hh] = has ? s : -INFINITY;
    const float m = wave_max(sc[hh]);
    if (lane == 0) wred[wave][hh] = m;
  }
  lds_barrier();
  float mx[PER];
#pragma unroll
  for (int hh = 0; hh < PER; ++hh) mx[hh] = fmaxf(fmaxf(wred[0][hh], wred[1][hh]), fmaxf(wred[2][hh], wred[3][hh]));   // (the waves of KEYS threads)
  lds_barrier();
#pragma unroll
  for (int hh = 0; hh < PER; ++hh) {
    const float p = has ? (FULL ? expf(sc[hh] - mx[hh]) : __expf(sc[hh] - mx[hh])) : 0.f;
    if (tid < KEYS) ps[hh][tid] = p;
    const float s = wave_sum(p);
    if (lane == 0) wred[wave][hh] = s;
  }
  lds_barrier();
#pragma unroll
  for (int hh = 0; hh < PER; ++hh) {
    if (tid == hh && hh < per) {
      float* ml = a.part_ml + (((size_t)t * a.nH + h0 + hh) * a.n_splits + split) * 2;
      ml[0] = mx[hh];
      ml[1] = (wred[0][hh] + wred[1][hh]) + (wred[2][hh] + wred[3][hh]);
    }
  }
  // values: thread (kg, ec) takes the keys kg, kg + KG, .. and 16 bytes of the row's width
  for (int z = 0; z < n_vh; ++z) {
    float acc[PER][VEC];
#pragma unroll
    for (int hh = 0; hh < PER; ++hh)
#pragma unroll
      for (int i = 0; i < VEC; ++i) acc[hh][i] = 0.f;
    auto add_values = [&](const uint4 (&w)[UV], int i0) {
#pragma unroll
      for (int u = 0; u < UV; ++u) {
        const int i = i0 + u * KG + kg;
        if (i < nk) {
          float vf[VEC];
          unpack16<T>(w[u], vf);
#pragma unroll
          for (int hh = 0; hh < PER; ++hh) {
            const float p = ps[hh][i];
#pragma unroll
            for (int e = 0; e < VEC; ++e) acc[hh][e] = fmaf(p, vf[e], acc[hh][e]);
          }
        }
      }
    };
    for (int i0 = 0; i0 < nk; i0 += UV * KG) {
      if (z > 0 || i0 > 0) load_values(vw, z, i0);
      add_values(vw, i0);
    }
    // the shares of the keys meet: lane moves within a wave, then the waves through LDS
    auto meet = [&](auto partner_sum) {
#pragma unroll
      for (int hh = 0; hh < PER; ++hh)
#pragma unroll
        for (int e = 0; e < VEC; ++e) acc[hh][e] = partner_sum(acc[hh][e]);
    };
    if (EC2 <= 1) meet([](float v) { return v + lane_move<DPP_XOR1>(v); });
    if (EC2 <= 2) meet([](float v) { return v + lane_move<DPP_XOR2>(v); });
    if (EC2 <= 4) meet([](float v) { return v + __shfl_xor(v, 4, 64); });
    if (EC2 <= 8) meet([](float v) { return v + lane_move<DPP_ROR8>(v); });
    if (EC2 <= 16) meet([](float v) { return sum_over_16(v); });
    if (EC2 <= 32) meet([](float v) { return sum_over_32(v); });
#pragma unroll
    for (int g0 = 0; g0 < PER; g0 += HG) {
      if (g0 >= per) break;
      lds_barrier();                                    // ored is free again
      if (lane < EC2 && ec < EC) {
#pragma unroll
        for (int hh = 0; hh < HG; ++hh)
#pragma unroll
          for (int e = 0; e < VEC; e += 4)
            *reinterpret_cast<float4*>(&ored[wave][hh][ec * VEC + e]) = float4{acc[g0 + hh][e], acc[g0 + hh][e + 1], acc[g0 + hh][e + 2], acc[g0 + hh][e + 3]};
      }
      lds_barrier();
      for (int i = tid; i < min(HG, per - g0) * dv; i += NT) {
        const int hh = i / dv, e = i - hh * dv;
        float o = ored[0][hh][e];
#pragma unroll
        for (int x = 1; x < WAVES; ++x) o += ored[x][hh][e];
        a.part_o[((((size_t)t * a.nH + h0 + g0 + hh) * n_vh + z) * a.n_splits + split) * dv + e] = o;
      }
    }
  }
}

struct CombineArgs {
  const int* positions;
  int nH, nKV, dv, n_splits, value_heads;
  const float* part_ml;
  const float* part_o;
  const float* sink;
  const float* vcos;
  const float* vsin;
  const float* gate;
  int gate_stride, gate_mode;
  float out_scale;
  float* out32;
};

template <typename T>
__global__ void attn_split_combine_kernel(T* __restrict__ out, CombineArgs a) {
  constexpr bool FULL = sizeof(T) == 4;
  const int t = blockIdx.x, h = blockIdx.y, z = blockIdx.z, dv = a.dv, S = a.n_splits;
  const int n_vh = a.value_heads > 0 ? a.value_heads : 1;
  const float* ml = a.part_ml + ((size_t)t * a.nH + h) * S * 2;
  float M = -INFINITY;
  for (int s = 0; s < S; ++s) M = fmaxf(M, ml[2 * s]);
  const float sk = a.sink ? a.sink[h] : -INFINITY;
  const float Mf = fmaxf(M, sk);
  float L = a.sink ? (FULL ? expf(sk - Mf) : __expf(sk - Mf)) : 0.f;
  for (int s = 0; s < S; ++s) {
    const float w = ml[2 * s] > -INFINITY ? (FULL ? expf(ml[2 * s] - Mf) : __expf(ml[2 * s] - Mf)) : 0.f;
    L = fmaf(ml[2 * s + 1], w, L);
  }
  const float inv = L > 0.f ? 1.f / L : 0.f;
  const float* po = a.part_o + (((size_t)t * a.nH + h) * n_vh + z) * S * dv;
  const int pos = a.positions[t];
  for (int m = threadIdx.x; 2 * m < dv; m += blockDim.x) {            // the pair (2m, 2m + 1); a last odd element alone
    const bool two = 2 * m + 1 < dv;
    float o0 = 0.f, o1 = 0.f;
    for (int s = 0; s < S; ++s) {
      const float w = ml[2 * s] > -INFINITY ? (FULL ? expf(ml[2 * s] - Mf) : __expf(ml[2 * s] - Mf)) : 0.f;
      o0 = fmaf(po[(size_t)s * dv + 2 * m], w, o0);
      if (two) o1 = fmaf(po[(size_t)s * dv + 2 * m + 1], w, o1);
    }
    o0 *= inv;
    o1 *= inv;
    if (a.vcos) {
      const float c = a.vcos[(size_t)pos * (dv >> 1) + m], sn = a.vsin[(size_t)pos * (dv >> 1) + m];
      const float u = o0, v = o1;
      o0 = fmaf(u, c, __fmul_rn(v, sn));
      o1 = fmaf(v, c, -__fmul_rn(u, sn));
    }
    if (a.out32) {
      float* dst = a.out32 + (((size_t)t * a.nH + h) * a.nKV + z) * dv;
      dst[2 * m] = o0;
      if (two) dst[2 * m + 1] = o1;
      continue;
    }
    if (a.gate) {
      const float* g = a.gate + (size_t)t * a.gate_stride;
      o0 *= sigmoid_f(a.gate_mode == 2 ? g[h * dv + 2 * m] : g[h], FULL);
      if (two) o1 *= sigmoid_f(a.gate_mode == 2 ? g[h * dv + 2 * m + 1] : g[h], FULL);
    }
    T* dst = out + ((size_t)t * a.nH + h) * dv;
    store_f32(dst, 2 * m, o0 * a.out_scale);
    if (two) store_f32(dst, 2 * m + 1, o1 * a.out_scale);
  }
}

}  // namespace

extern "C" int alice_attention_split_supported(int dtype, int nH, int nKV, int d, int dv) {
  const int vec = dtype == DT_F32 ? 4 : 8;
  return nKV >= 1 && nH % nKV == 0 && nH / nKV <= 16 && d >= vec && dv >= vec && d % vec == 0 && dv % vec == 0 && d <= 256 && dv <= 256;
}

// The number of key runs for at most max_keys visible keys a token, and the float32 workspace for T tokens.
extern "C" int alice_attention_split_runs(int max_keys) { return max(1, ceil_div(max_keys, KEYS)); }
extern "C" long alice_attention_split_workspace(int T, int nH, int nKV, int dv, int runs, int per_value_head) {
  return (long)T * nH * runs * 2 + (long)T * nH * (per_value_head ? nKV : 1) * runs * dv;
}

// alice_attention_masked's result by the key-split kernels; max_keys: the most keys any token of the step sees (the
// caller knows it from the step's longest context and the mask); work: alice_attention_split_workspace floats.
extern "C" int alice_attention_split(const void* q, int dtype, const void* k_pool, const void* v_pool, void* out, float* out32,
                                     const int* positions, const int* seq_of_token, const int* block_table, int bt_stride,
                                     int T, int nH, int nKV, int d, int dv, int page_size, float scale, int window, int chunk,
                                     int keep_first, int max_keys, const float* bias_slopes, const float* sink,
                                     const float* vrot_cos, const float* vrot_sin, const float* gate, int gate_stride,
                                     int gate_mode, float out_scale, float* work, hipStream_t stream) {
  ALICE_CHECK(dtype_ok(dtype), "attention: unknown dtype %d", dtype);
  ALICE_CHECK(alice_attention_split_supported(dtype, nH, nKV, d, dv), "attention: heads %d / %d of sizes %d and %d are outside this kernel's range", nH, nKV, d, dv);
  ALICE_CHECK(q && k_pool && v_pool && (out || out32) && positions && seq_of_token && block_table && work, "attention: a pointer is missing");
  ALICE_CHECK(T >= 0 && page_size > 0 && bt_stride > 0 && max_keys >= 1, "attention: bad sizes");
  ALICE_CHECK(window >= 0 && chunk >= 0 && keep_first >= 0, "attention: window, chunk and keep_first must not be negative (0 turns them off)");
  ALICE_CHECK((vrot_cos == nullptr) == (vrot_sin == nullptr) && (vrot_cos == nullptr || dv % 2 == 0), "attention: turning the output back needs both tables and an even value head size");
  ALICE_CHECK(gate == nullptr || (gate_mode == 1 && gate_stride >= nH) || (gate_mode == 2 && gate_stride >= nH * dv),
              "attention: gate rows of %d elements are too short", gate_stride);
  ALICE_CHECK(((uintptr_t)q & 15) == 0 && ((uintptr_t)k_pool & 15) == 0 && ((uintptr_t)v_pool & 15) == 0, "attention: operands are not aligned");
  if (T == 0) return 0;
  const int runs = alice_attention_split_runs(max_keys);
  ALICE_CHECK(runs <= 65535 && nKV <= 65535 && nH <= 65535, "attention: too many heads or keys for one launch");
  const int n_vh = out32 ? nKV : 0;
  float* part_ml = work;
  float* part_o = work + (size_t)T * nH * runs * 2;
  SplitArgs a{positions, seq_of_token, block_table, bt_stride, nH, nKV, d, dv, page_size, scale, window, chunk, keep_first, runs, n_vh,
              bias_slopes, part_ml, part_o};
  const int per = nH / nKV;
  dim3 grid(T, nKV, runs);
  // A wave's 32 keys are that many loads of whole rows, half as many as lanes read a row, and so are a thread's values: what is asked for
  // beyond is a row that was read (32 sequences of 2,000 keys in bfloat16, 8 own kv heads of 32: 32.1 us with eight loads of which six
  // are such, 23.8 with two; 16 of 64: 67.6 with eight, 59.9 with four).
  const int piece = 16 / (dtype == DT_F32 ? 4 : 2), widest = max(ceil_div(d, piece), ceil_div(dv, piece));
#define GO2(TT, PER, U) attn_split_kernel<TT, PER, U><<<grid, NT, 0, stream>>>((const TT*)q, (const TT*)k_pool, (const TT*)v_pool, a)
#define GO(TT, PER, MOST)                            \
  do {                                               \
    if (widest <= 4) GO2(TT, PER, 2);                \
    else if (widest <= 8) GO2(TT, PER, 4);           \
    else GO2(TT, PER, MOST);                         \
  } while (0)
#define BY_PER(TT)                    \
  do {                                \
    if (per <= 1) GO(TT, 1, 8);       \
    else if (per <= 2) GO(TT, 2, 8);  \
    else if (per <= 4) GO(TT, 4, 8);  \
    else if (per <= 8) GO(TT, 8, 4);  \
    else GO(TT, 16, 4);               \
  } while (0)
  if (dtype == DT_F32) BY_PER(float);
  else BY_PER(bf16_t);
#undef BY_PER
#undef GO
#undef GO2
  ALICE_LAUNCH_CHECK();
  CombineArgs c{positions, nH, nKV, dv, runs, n_vh, part_ml, part_o, sink, vrot_cos, vrot_sin, gate, gate_stride, gate_mode, out_scale, out32};
  dim3 g2(T, nH, out32 ? nKV : 1);
  const int threads = dv > 128 ? 128 : 64;
  if (dtype == DT_F32) attn_split_combine_kernel<float><<<g2, threads, 0, stream>>>((float*)out, c);
  else attn_split_combine_kernel<bf16_t><<<g2, threads, 0, stream>>>((bf16_t*)out, c);
  ALICE_LAUNCH_CHECK();
  return 0;
}
