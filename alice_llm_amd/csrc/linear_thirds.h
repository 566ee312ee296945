// The 32-bit products on the bfloat16 matrix instruction (linear_thirds.hip): their plan and launch.
#pragma once
#include <hip/hip_runtime.h>

constexpr int THIRDS_BK = 32;       // slices of the inner dimension are multiples of this

struct ThirdsPlan {
  int tile, split;
  float us;                         // estimated
};
ThirdsPlan alice_linear_thirds_plan(int M, int N, int K, bool geglu, int min_split, int max_split);
// x, w and y float32, x and w on 16 bytes, K a multiple of 4.
int alice_linear_thirds(const float* x, const float* w, float* y, int M, int N, int K, int epi, float param, int full, const ThirdsPlan& p,
                        hipStream_t stream);
