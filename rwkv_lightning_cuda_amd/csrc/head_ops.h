// Values of one head with four channels per lane (a DPP row of 16 lanes holds the head): sums, fp16 products, loads.
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
// f16(a * b) of four values with one rounding each, what the compiler makes of a product that is only converted
// (v_fma_mixlo_f16) where a lane has one channel; with four it would convert pairs, which rounds twice.
__device__ __forceinline__ half4_t mul_f16(const float (&a)[4], const float (&b)[4]) {
  uint2_t r;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    uint32_t d;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0\n\tv_fma_mixhi_f16 %0, %3, %4, 0"
        : "=&v"(d)
        : "v"(a[2 * i]), "v"(b[2 * i]), "v"(a[2 * i + 1]), "v"(b[2 * i + 1]));
    r[i] = d;
  }
  return __builtin_bit_cast(half4_t, r);
}
// four values at p; VEC: p is aligned to them
template <bool VEC>
__device__ __forceinline__ half4_t load4(const half_t* p) {
  if constexpr (VEC) return *reinterpret_cast<const half4_t*>(p);
  return half4_t{p[0], p[1], p[2], p[3]};
}
template <bool VEC>
__device__ __forceinline__ void store4(half_t* p, half4_t v) {
  if constexpr (VEC) {
    *reinterpret_cast<half4_t*>(p) = v;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) p[e] = v[e];
  }
}

// kk normalise, a-gate, new k and the decay logit of four channels (rounding points of cuda/rwkv7_fast_ops_fp16.cu)
struct HeadGate {
  half4_t new_k, neg_kk, kka, w_sum;
};
__device__ __forceinline__ HeadGate head_gate(half4_t k4, half4_t a4, half4_t w4, half4_t kk4, half4_t a04, half4_t ka4, half4_t w04) {
  HeadGate o;
  float u[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) u[e] = h2f(k4[e]) * h2f(kk4[e]);
  const float total = head_sum_of_product(u, u);
  const float inv = 1.0f / fmaxf(sqrtf(total), kKkEps);
  half4_t pkk;
  float kv[4], kf[4], kk[4], av[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    kk[e] = u[e] * inv;
    av[e] = sigmoid_f(h2f(a04[e]) + h2f(a4[e]));
    const float ka = h2f(ka4[e]);
    kv[e] = h2f(k4[e]);
    kf[e] = fmaf(av[e], ka, 1.0f - ka);
    pkk[e] = f2h(kk[e]);
    o.w_sum[e] = f2h(h2f(w4[e]) + h2f(w04[e]));  // rwkv7_add_vec_launch rounding point
  }
  o.new_k = mul_f16(kv, kf);
  // (negated as halves: the compiler does not get a vector of negated floats through without packed fp32)
  o.neg_kk = __builtin_bit_cast(half4_t, __builtin_bit_cast(uint2_t, pkk) ^ uint2_t{0x80008000u, 0x80008000u});
  o.kka = mul_f16(kk, av);
  return o;
}
__device__ __forceinline__ float head_decay(half_t w_sum) {
  return exp2f(-0.8750387749145276f / (1.0f + exp2f(-1.4426950408889634f * h2f(w_sum))));
}
// GroupNorm of the fp16-rounded y, the (r.k.r_k) v bonus and the gate
__device__ __forceinline__ half4_t head_output(const float (&yv)[4], half4_t r4, half4_t k4, half4_t v4, half4_t g4, half4_t rk4, half4_t lw4,
                                               half4_t lb4) {
  float d[4], rk[4], w[4];
  const float mean = head_sum(yv) * (1.0f / 64.0f);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    d[e] = yv[e] - mean;
    rk[e] = mul_f32(h2f(r4[e]), h2f(k4[e]));
    w[e] = h2f(rk4[e]);
  }
  const float var = head_sum_of_product(d, d) * (1.0f / 64.0f);
  const float rstd = rsqrtf(var + kLnxEps);
  const float rkv = head_sum_of_product(rk, w);
  float o[4], gate[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    o[e] = d[e] * rstd * h2f(lw4[e]) + h2f(lb4[e]) + rkv * h2f(v4[e]);
    gate[e] = h2f(g4[e]);
  }
  return mul_f16(o, gate);
}

}  // namespace rwkv
