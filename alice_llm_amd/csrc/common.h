// Shared device helpers and the host-side error channel of the HIP library.
// Everything here targets gfx950 (CDNA4): 64-lane wavefronts, 160 KB LDS per CU.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdio.h>
#include <atomic>

#define ALICE_WAVE 64

// Storage types.  DT_F32 / DT_BF16 are the dtype codes of the C interface.
enum { DT_F32 = 0, DT_BF16 = 1 };

struct bf16_t {
  uint16_t bits;
};

__device__ __forceinline__ float bf16_to_f32(bf16_t v) {
  return __uint_as_float(((uint32_t)v.bits) << 16);
}
__device__ __forceinline__ float bf16_bits_to_f32(uint32_t bits16) {
  return __uint_as_float(bits16 << 16);
}
// Round to nearest even; NaN stays NaN (the hardware conversion of gfx950).
__device__ __forceinline__ bf16_t f32_to_bf16(float f) {
  bf16_t r;
  r.bits = __builtin_bit_cast(uint16_t, (__bf16)f);
  return r;
}
// Two values rounded and packed, the first in the low half.
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  f32x2_t v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

template <typename T> __device__ __forceinline__ float load_f32(const T* p, size_t i);
template <> __device__ __forceinline__ float load_f32<float>(const float* p, size_t i) { return p[i]; }
template <> __device__ __forceinline__ float load_f32<bf16_t>(const bf16_t* p, size_t i) { return bf16_to_f32(p[i]); }

template <typename T> __device__ __forceinline__ void store_f32(T* p, size_t i, float v);
template <> __device__ __forceinline__ void store_f32<float>(float* p, size_t i, float v) { p[i] = v; }
template <> __device__ __forceinline__ void store_f32<bf16_t>(bf16_t* p, size_t i, float v) { p[i] = f32_to_bf16(v); }

// Rounds through the storage type: what a value becomes when it is stored and read back.
template <typename T> __device__ __forceinline__ float round_to(float v);
template <> __device__ __forceinline__ float round_to<float>(float v) { return v; }
template <> __device__ __forceinline__ float round_to<bf16_t>(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// A reduction over the 64 lanes, every lane gets the result: the butterfly over lane distances 32, 16, 8, 4, 2, 1 by lane-swap
// and DPP moves, a few cycles each, where a shuffle goes through the LDS unit (about 60 cycles a step, one waiting for the
// other).  The same partners in the same order as shuffles by 32 .. 1, so sums have the same bits: after the step over 8 a
// row of 16 lanes repeats itself every 8, which makes a rotation by 4 the exchange over 4.  All 64 lanes must be active: a swap
// with a lane that is not leaves a lane its own value twice, and the sum is wrong in every lane.
// (Before and after, everything else equal: the draw behind 64 rows of 256,000 logits 49.2 and 47.2 us, a 2B decode step of
// eight sequences with its 53 norms 1,973 and 1,952 us.)
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_move(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true); }
constexpr int DPP_ROR12 = 0x12C, DPP_ROR8 = 0x128, DPP_ROR4 = 0x124, DPP_XOR2 = 0x4E, DPP_XOR1 = 0xB1, DPP_HALF_MIRROR = 0x141;

template <typename T, typename F>
__device__ __forceinline__ T wave_reduce(T v, F op) {
  static_assert(sizeof(T) == 4 || sizeof(T) == 8, "one or two registers a value");
  if constexpr (sizeof(T) == 4) {
    uint32_t u = __builtin_bit_cast(uint32_t, v);
    auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    u = __builtin_bit_cast(uint32_t, (T)op(__builtin_bit_cast(T, (uint32_t)a[0]), __builtin_bit_cast(T, (uint32_t)a[1])));
    auto b = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    v = op(__builtin_bit_cast(T, (uint32_t)b[0]), __builtin_bit_cast(T, (uint32_t)b[1]));
    v = op(v, __builtin_bit_cast(T, dpp_move<DPP_ROR8>(__builtin_bit_cast(uint32_t, v))));
    v = op(v, __builtin_bit_cast(T, dpp_move<DPP_ROR4>(__builtin_bit_cast(uint32_t, v))));
    v = op(v, __builtin_bit_cast(T, dpp_move<DPP_XOR2>(__builtin_bit_cast(uint32_t, v))));
    return op(v, __builtin_bit_cast(T, dpp_move<DPP_XOR1>(__builtin_bit_cast(uint32_t, v))));
  } else {
    auto two = [](uint32_t lo, uint32_t hi) { return __builtin_bit_cast(T, (unsigned long long)lo | (unsigned long long)hi << 32); };
    auto lo_of = [](T x) { return (uint32_t)__builtin_bit_cast(unsigned long long, x); };
    auto hi_of = [](T x) { return (uint32_t)(__builtin_bit_cast(unsigned long long, x) >> 32); };
    auto a = __builtin_amdgcn_permlane32_swap(lo_of(v), lo_of(v), false, false);
    auto b = __builtin_amdgcn_permlane32_swap(hi_of(v), hi_of(v), false, false);
    v = op(two(a[0], b[0]), two(a[1], b[1]));
    auto c = __builtin_amdgcn_permlane16_swap(lo_of(v), lo_of(v), false, false);
    auto d = __builtin_amdgcn_permlane16_swap(hi_of(v), hi_of(v), false, false);
    v = op(two(c[0], d[0]), two(c[1], d[1]));
    v = op(v, two(dpp_move<DPP_ROR8>(lo_of(v)), dpp_move<DPP_ROR8>(hi_of(v))));
    v = op(v, two(dpp_move<DPP_ROR4>(lo_of(v)), dpp_move<DPP_ROR4>(hi_of(v))));
    v = op(v, two(dpp_move<DPP_XOR2>(lo_of(v)), dpp_move<DPP_XOR2>(hi_of(v))));
    return op(v, two(dpp_move<DPP_XOR1>(lo_of(v)), dpp_move<DPP_XOR1>(hi_of(v))));
  }
}
__device__ __forceinline__ float wave_sum(float v) { return wave_reduce(v, [](float a, float b) { return a + b; }); }
__device__ __forceinline__ float wave_max(float v) { return wave_reduce(v, [](float a, float b) { return fmaxf(a, b); }); }

// Sum over a block of up to 1024 threads (whole waves); every thread gets the result.  `red` holds 16 floats, one a wave.  Every wave adds
// up the waves' sums by itself: one barrier fewer than through the first wave.
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_sum(v);
  __syncthreads();                       // `red` may still be read from an earlier call
  if (lane == 0) red[wid] = v;
  __syncthreads();
  return wave_sum(lane < nw ? red[lane] : 0.f);
}
__device__ __forceinline__ float block_max(float v, float* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) red[wid] = v;
  __syncthreads();
  return wave_max(lane < nw ? red[lane] : -INFINITY);
}

// A barrier between phases that exchange data through LDS only: it waits for the wave's LDS accesses, not for its
// loads and stores of global memory (rows fetched ahead, results on their way out), which __syncthreads() would also
// wait for at every phase.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// tanh at full precision for the 32-bit path, a fast form for the bfloat16 path.
__device__ __forceinline__ float tanh_full(float x) { return tanhf(x); }
__device__ __forceinline__ float tanh_fast(float x) {
  // tanh(x) = 1 - 2 / (2^(2 log2e x) + 1) with the hardware's exp2 and reciprocal (about 1 ulp each):
  // absolute error about 2e-7; 2^x overflows to +inf and underflows to 0, which give exactly +-1.
  float e = __builtin_amdgcn_exp2f(x * 2.8853900817779268f);
  return fmaf(-2.f, __builtin_amdgcn_rcpf(e + 1.f), 1.f);
}
__device__ __forceinline__ float gelu_tanh_f(float z, bool full) {
  if (full) {
    const float u = 0.7978845608028654f * (z + 0.044715f * z * z * z);
    return 0.5f * z * (1.f + tanh_full(u));
  }
  // 0.5 (1 + tanh u) = 1 / (1 + 2^(-2 log2e u)), u = sqrt(2 / pi) (z + 0.044715 z^3): no difference of nearly equal numbers for
  // negative z, and half the instructions of the tanh above it.
  const float q = z * fmaf(z * z, -0.10294323957f, -2.3022081981f);
  return z * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(q));
}

// z / (1 + e^-z) by one division, rounded once, here and in unary_act() below.  (By the hardware's reciprocal and a product the l2
// error over [-9, 9] goes from 4.3e-8 to 4.6e-8, for 0.7 % of a prompt whose feed-forwards are SiLU gates.)
__device__ __forceinline__ float silu_f(float z, bool full) { return z / (1.f + (full ? expf(-z) : __expf(-z))); }

// The gated product of two stacked matrices' outputs (gate g, up u), the epilogue ALICE_EPI_GEGLU.  Its
// parameter picks the form: 0 gives gelu_tanh(g) * u; a positive `limit` gives the limited form
// g' = min(g, limit), u' = clamp(u, -limit, limit), g' * sigmoid(1.702 g') * (u' + 1); a negative one
// (ALICE_GATED_SILU) gives g * sigmoid(g) * u.
__device__ __forceinline__ float gated_act(float g, float u, float limit, bool full) {
  if (limit < 0.f) return silu_f(g, full) * u;
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    const float e = full ? expf(-1.702f * g) : __expf(-1.702f * g);
    return g * (u + 1.f) / (1.f + e);
  }
  return gelu_tanh_f(g, full) * u;
}
// The function of one output element, the epilogue ALICE_EPI_SOFTCAP.  Its parameter picks the form: a positive cap
// gives cap * tanh(v / cap); ALICE_UNARY_RELU2 (-1) the square of max(v, 0); ALICE_UNARY_SILU (-2) v * sigmoid(v).
__device__ __forceinline__ float unary_act(float v, float p, bool full) {
  if (p < -1.5f) return silu_f(v, full);
  if (p < 0.f) {
    const float r = fmaxf(v, 0.f);
    return r * r;
  }
  return p * (full ? tanh_full(v / p) : tanh_fast(v / p));
}
__device__ __forceinline__ float sigmoid_f(float z, bool full) { return 1.f / (1.f + (full ? expf(-z) : __expf(-z))); }

// Where element (row r, column i) of a [T, H] bfloat16 output goes: row-major, or fragment order for the
// matrix-core kernels ([T/16][H/32][64][8], see linear_mfma.hip).
__device__ __forceinline__ size_t out_index(int layout, int r, int i, int H) {
  if (layout == 0) return (size_t)r * H + i;
  return ((size_t)((size_t)(r >> 4) * (H >> 5) + (i >> 5)) * 64 + ((i & 31) >> 3) * 16 + (r & 15)) * 8 + (i & 7);
}

// Whole quotients by a divisor that the host knows: a kernel that waits for nothing else yet spends 25 dependent instructions
// on a division by a run-time number.  Exact while a * divisor < 2^31 (the host's number is 2^31 / divisor, rounded up).
__device__ __forceinline__ uint32_t quotient(uint32_t a, uint32_t reciprocal) { return (uint32_t)(((uint64_t)a * reciprocal) >> 31); }
static inline uint32_t reciprocal_of(uint32_t divisor) { return (uint32_t)(((1ull << 31) + divisor - 1) / divisor); }

// ---- host side -------------------------------------------------------------------------
void alice_set_error(const char* fmt, ...);

#define ALICE_CHECK(cond, ...)            \
  do {                                    \
    if (!(cond)) {                        \
      alice_set_error(__VA_ARGS__);       \
      return 1;                           \
    }                                     \
  } while (0)

// Blocks of a kernel take more LDS than they may without asking: the device is asked once for each kernel, whichever thread comes first.
// told: the kernel's own, a bit a device.
inline bool lds_granted(const void* kernel, int bytes, std::atomic<uint64_t>& told) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess) return false;
  const uint64_t bit = device < 64 ? 1ull << device : 0;
  if (told.load(std::memory_order_acquire) & bit) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  told.fetch_or(bit, std::memory_order_release);
  return true;
}

#define ALICE_LAUNCH_CHECK()                                                   \
  do {                                                                         \
    hipError_t e_ = hipGetLastError();                                         \
    if (e_ != hipSuccess) {                                                    \
      alice_set_error("%s:%d: launch failed: %s", __FILE__, __LINE__,          \
                      hipGetErrorString(e_));                                  \
      return 2;                                                                \
    }                                                                          \
  } while (0)

static inline int ceil_div(long a, long b) { return (int)((a + b - 1) / b); }

// Calls `F<T>(...)`-style lambdas with the storage type that a dtype code names.
#define DISPATCH_DTYPE(code, T, ...)                         \
  do {                                                       \
    if ((code) == DT_F32) { using T = float; __VA_ARGS__; }  \
    else { using T = bf16_t; __VA_ARGS__; }                  \
  } while (0)

static inline bool dtype_ok(int code) { return code == DT_F32 || code == DT_BF16; }
