// Sums over one head with four channels per lane (a DPP row of 16 lanes holds the head).
#pragma once
#include "common.h"

namespace rwkv {

// The sums are those of a wavefront with one channel per lane (wave_sum: channel i adds what i ^ 32, 16, 8, 4, 2, 1 holds), so
// that the kernels that do this inside a larger one agree bitwise: the first four levels are lane exchanges, the last two lie
// within a lane.
__device__ __forceinline__ float head_sum_tail(float (&t)[4]) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    t[e] += __builtin_bit_cast(float, lane_xor_dpp<4>(__builtin_bit_cast(int, t[e])));
    t[e] = dpp_add<0x4E>(t[e]);  // lane ^ 2
    t[e] = dpp_add<0xB1>(t[e]);  // lane ^ 1
  }
  return (t[0] + t[2]) + (t[1] + t[3]);
}
__device__ __forceinline__ float head_sum(const float (&v)[4]) {
  float t[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) t[e] = dpp_add<0x128>(v[e]);  // lane ^ 8
  return head_sum_tail(t);
}
// sum of a * b with a fused first level (wave_sum_dpp_of_product)
__device__ __forceinline__ float head_sum_of_product(const float (&a)[4], const float (&b)[4]) {
  float t[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float p;
    {
#pragma clang fp contract(off)
      p = a[e] * b[e];
    }
    t[e] = fmaf(a[e], b[e], __builtin_bit_cast(float, lane_xor_dpp<8>(__builtin_bit_cast(int, p))));
  }
  return head_sum_tail(t);
}

}  // namespace rwkv
