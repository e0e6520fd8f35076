// WKV7 time-mix recurrence of a model's prefill calls in chunks of 16 tokens on the matrix cores, fp32 state.
//
// Reference semantics: cuda/rwkv7_wkv_fp32_v2.cu:100-126, with the operands of cuda/rwkv7_fast_ops_fp16.cu (kk normalise, a-gate,
// decay) and the per-head GroupNorm, bonus and gate behind it.  Per token (state S [value row i][key column j]):
//   u = S a;  S = S diag(d) + u b^T + v k^T;  y = S r
// Over a chunk with the running products P_t = d_1 .. d_t (per column) and
//   A_t = a_t P_{t-1},  R_t = r_t P_t,  B_s = b_s / P_s,  K_s = k_s / P_s
// the same sums are matrix products:
//   U = S A^T + U [A B^T]_{s<t} + V [A K^T]_{s<t}        (u of every token; the middle term is a triangular solve)
//   Y = S R^T + U [R B^T]_{s<=t} + V [R K^T]_{s<=t}
//   S = (S + U^T B + V^T K) diag(P_16)
// The solve is taken to the left side once per chunk, without the state: A' = (I - [A B^T])^-1 A and K' the same of [A K^T], so
// that U = S A'^T + V K'.  The decay map keeps every d above 0.545, so 1 / P_16 stays below 2e4.
//
// Precision: nothing is held in less than fp32.  The products of decays and [A B^T], [A K^T] are summed in fp64 (v_mfma_f64_16x16x4),
// U and Y in fp32 (v_mfma_f32_16x16x4, twice the rate of the vector unit), the update of the state as products of bf16 pieces that
// add up to the fp32 operands exactly, summed in fp32.  The operands have the bits that kk_a_gate_kernel gives them.  Error of the state
// against 64-bit sums, 2-norm, chunks / token by token (operands of independent channels and tokens, logits uniform over [-6, 2], state
// N(0, 1)): 128 tokens x 1024 heads 5.7e-8 / 5.7e-8, 512 x 64 5.7e-8 / 5.7e-8, 2048 x 64 5.8e-8 / 5.7e-8, 333 x 96 5.9e-8 / 6.0e-8, 64 x 128
// 5.8e-8 / 5.8e-8; keys that follow one another closely under slow decay, 512 x 24: 2.3e-7 / 3.6e-7; the operands of a layer, 7.2B shape
// 7.7e-8 / 1.1e-7, 1.5B 7.6e-8 / 1.2e-7 (median over heads).
//
// A chunk is one unit: results depend on where a call begins (as those of a prefill call's products do, through their tiles).  The
// operator rwkv_hip_wkv7 promises the same bits for every split of a sequence and steps token by token (wkv7.hip).
//
// Operands that are not finite: a product takes zero times such a value to the tokens ahead of it, so they are taken out before the products
// (without_spoilt_tokens).  A token whose k, v, decay or gate is not finite makes its head's outputs from there on and the state NaN - token
// by token it is the outputs, by GroupNorm, and the rows or columns of the state that it reaches first - one whose r is not finite its own
// output.  (us per launch without / with the look at every operand: whole heads, 1024 x 128 tokens 100.0 / 102.0; 96 heads x 333 tokens,
// preparation 19.0 / 19.5, chain 23.9 / 24.0.)
//
// us per layer from the rank-outs to the output projection's input, token by token -> in chunks: 16 x 128 tokens x 64 heads 166 ->
// 95, 3 x 333 x 32 72 -> 48, 1 x 128 x 64 26.4 -> 22.4, 1 x 512 x 64 75 -> 47.  What bounds them: many heads, the issue of VALU
// instructions (some 800 per wavefront and chunk) and the matrix core (2700 clocks), which add up although four wavefronts share a
// SIMD; few heads, launches (three), the latency of one chunk's preparation (6 us) and 0.65 us per link of the chain, most of it LDS
// and the requests for 25 KB per chunk and block, two of which share a CU.
#include <algorithm>

#include "head_ops.h"
#include "ops.h"

namespace rwkv {

namespace {

constexpr int kTok = 16;     // tokens of a chunk
constexpr int kRow = 68;     // floats from row to row of a [16][64] tile in LDS: 16-byte reads down a column touch every bank once
constexpr int kSquare = 20;  // the same for [16][16]

typedef double double4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float2_t __attribute__((ext_vector_type(2)));

// (LDS alone is exchanged over these barriers: requests to memory stay in flight)
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Lane (g, n) = (lane / 16, lane % 16) gives column g of A's row n and row g of B's column n (eight of each to the bf16 product); the
// result's register i is row 4 g + i (fp64: 4 i + g) of column n.
__device__ __forceinline__ float4_t mfma4(float a, float b, float4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ double4_t mfma4(double a, double b, double4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float4_t mfma32(uint4_t a, uint4_t b, float4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// x as the sum of three bf16 numbers (its 24 bits exactly), four values to two dwords per piece
struct Pieces {
  uint2_t p[3];
};
__device__ __forceinline__ Pieces split(const float4_t& x) {
  Pieces o;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float lo = x[2 * h], hi = x[2 * h + 1];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const uint32_t w = __builtin_bit_cast(uint32_t, __builtin_convertvector(float2_t{lo, hi}, bf16x2_t));
      o.p[i][h] = w;
      if (i < 2) {
        lo -= __builtin_bit_cast(float, w << 16);
        hi -= __builtin_bit_cast(float, w & 0xffff0000u);
      }
    }
  }
  return o;
}

// Register e of the 16-lane row g <-> register g of row e, four sets at once.  (Two idle slots between a register's write and the swap
// that reads it.)
__device__ __forceinline__ void transpose4x4(uint4_t (&x)[4]) {
#define RWKV_SWAPS(OP, I, J) OP " %" #I ", %" #J "\n\t"
  asm volatile("s_nop 1\n\t"
               RWKV_SWAPS("v_permlane32_swap_b32", 0, 2) RWKV_SWAPS("v_permlane32_swap_b32", 1, 3)
               RWKV_SWAPS("v_permlane32_swap_b32", 4, 6) RWKV_SWAPS("v_permlane32_swap_b32", 5, 7)
               RWKV_SWAPS("v_permlane32_swap_b32", 8, 10) RWKV_SWAPS("v_permlane32_swap_b32", 9, 11)
               RWKV_SWAPS("v_permlane32_swap_b32", 12, 14) RWKV_SWAPS("v_permlane32_swap_b32", 13, 15)
               "s_nop 1\n\t"
               RWKV_SWAPS("v_permlane16_swap_b32", 0, 1) RWKV_SWAPS("v_permlane16_swap_b32", 2, 3)
               RWKV_SWAPS("v_permlane16_swap_b32", 4, 5) RWKV_SWAPS("v_permlane16_swap_b32", 6, 7)
               RWKV_SWAPS("v_permlane16_swap_b32", 8, 9) RWKV_SWAPS("v_permlane16_swap_b32", 10, 11)
               RWKV_SWAPS("v_permlane16_swap_b32", 12, 13) RWKV_SWAPS("v_permlane16_swap_b32", 14, 15)
               "s_nop 1"
               : "+v"(x[0][0]), "+v"(x[0][1]), "+v"(x[0][2]), "+v"(x[0][3]), "+v"(x[1][0]), "+v"(x[1][1]), "+v"(x[1][2]), "+v"(x[1][3]),
                 "+v"(x[2][0]), "+v"(x[2][1]), "+v"(x[2][2]), "+v"(x[2][3]), "+v"(x[3][0]), "+v"(x[3][1]), "+v"(x[3][2]), "+v"(x[3][3]));
#undef RWKV_SWAPS
}

// num / den of normal numbers, rounded as the division is (but for its last step's scaling)
__device__ __forceinline__ float quotient(float num, float den) {
  float r = rcp_f(den);
  r = fmaf(fmaf(-den, r, 1.0f), r, r);
  const float q = num * r;
  return fmaf(fmaf(-den, q, num), r, q);
}
__device__ __forceinline__ float decay_of(float w) {
  const float e = __builtin_amdgcn_exp2f(-1.4426950408889634f * w);
  return __builtin_amdgcn_exp2f(quotient(-0.8750387749145276f, 1.0f + (e > 1e30f ? 1e30f : e)));
}

struct ChannelConstants {
  half4_t k_k, a0, k_a, w0;
  __device__ __forceinline__ void load(const TmixSeqArgs& fa, int ch) {
    k_k = *reinterpret_cast<const half4_t*>(fa.k_k + ch);
    a0 = *reinterpret_cast<const half4_t*>(fa.a0 + ch);
    k_a = *reinterpret_cast<const half4_t*>(fa.k_a + ch);
    w0 = *reinterpret_cast<const half4_t*>(fa.w0 + ch);
  }
};
struct ChunkRows {  // this lane's four channels of one token
  half4_t r, k, a12, w12, v;
  __device__ __forceinline__ void load(const TmixSeqArgs& fa, const half_t* v_in, int64_t at) {
    r = *reinterpret_cast<const half4_t*>(fa.r + at);
    k = *reinterpret_cast<const half4_t*>(fa.k + at);
    a12 = *reinterpret_cast<const half4_t*>(fa.a12 + at);
    w12 = *reinterpret_cast<const half4_t*>(fa.w12 + at);
    v = *reinterpret_cast<const half4_t*>(v_in + at);
  }
};

struct ChunkTiles {
  float a[kTok][kRow];  // A, then A'
  float r[kTok][kRow];
  union {
    float b[kTok][kRow];
    float y[kTok][kRow];  // (the kernel for whole heads, when b has been used)
  };
  float k[kTok][kRow];
  union {
    struct {
      float ab[kTok][kSquare];  // [s][t]
      float ak[kTok][kSquare];  // [t][s], then K'
    };
    double part[4][kHead];      // products of the four decays of a wavefront: before ab is made
  };
  float rb[kTok][kSquare], rk[kTok][kSquare];  // [t][s]
  float decay[kHead];                          // P_16
  uint4_t spoilt;                              // of each wavefront's tokens (without_spoilt_tokens)
};

// Operands of the state update and V, as the matrix core reads them: lane (g, n) of tile q holds column 16 q + n of the tokens
// 4 g .. 4 g + 3.
struct UpdateOperands {
  uint4_t kb[3][4][kWave];  // pieces of K P_16 (two dwords) and of B P_16
  uint4_t v[4][kWave];      // V in two pieces (fp16 needs no more)
};

__device__ __forceinline__ bool not_finite(half_t x) { return (__builtin_bit_cast(uint16_t, x) & 0x7c00) == 0x7c00; }

// Takes tokens with operands that are not finite out of this lane's column of four tokens (stage_operands): bit i of the result, those that
// leave nothing of the state, bit 4 + i, those that have lost r alone.
__device__ __forceinline__ uint32_t without_spoilt_tokens(uint4_t (&x)[4]) {
  uint32_t spoilt = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t k_a = as_half2(x[0][i]), b_r = as_half2(x[1][i]);
    const float d = __builtin_bit_cast(float, static_cast<uint32_t>(x[3][i]));
    if (__ballot(not_finite(k_a[0]) || not_finite(k_a[1]) || not_finite(b_r[0]) || not_finite(as_half2(x[2][i])[0]) || d != d)) {
      x[0][i] = x[1][i] = x[2][i] = 0u;
      x[3][i] = __builtin_bit_cast(uint32_t, 1.0f);
      spoilt |= 1u << i;
    } else if (__ballot(not_finite(b_r[1]))) {
      x[1][i] &= 0xffffu;
      spoilt |= 16u << i;
    }
  }
  return spoilt;
}

struct Staged {
  half4_t new_k;
  uint32_t lost;  // tokens whose y is NaN, a bit each (the same in all wavefronts)
};

// kk normalise, a-gate, new k and decay of token 4 wave + g, channels 4 n .. 4 n + 3 (the formulas and rounding points of
// kk_a_gate_kernel), then the rows of A, R, B, K and the operands of the update.  `live`: the token exists; one past the end of
// the call leaves the state as it is.
// The products of decays are in fp64, where every A, R, B, K is rounded once.  One barrier inside.
__device__ __forceinline__ Staged stage_operands(ChunkTiles& t, UpdateOperands& uo, const ChunkRows& q, const ChannelConstants& c, bool live,
                                                  int wave, int lane) {
  const int g = lane >> 4, n = lane & 15;
  float u[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) u[e] = h2f(q.k[e]) * h2f(c.k_k[e]);
  const float total = head_sum_of_product(u, u);  // (in any other order -kk of one token in some hundred differs by an fp16 ulp)
  const float inv = quotient(1.0f, fmaxf(sqrtf(total), kKkEps));
  half4_t nk;
  uint4_t x[4];  // this token's (new k, -kk), (kk a, r), (v, v), decay of four channels; then this channel's of four tokens
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float kk = u[e] * inv;
    const float av = sigmoid_f(h2f(c.a0[e]) + h2f(q.a12[e]));
    const float ka = h2f(c.k_a[e]);
    nk[e] = f2h(h2f(q.k[e]) * fmaf(av, ka, 1.0f - ka));
    x[0][e] = live ? __builtin_bit_cast(uint32_t, half2_t{nk[e], f2h(-kk)}) : 0u;
    x[1][e] = live ? __builtin_bit_cast(uint32_t, half2_t{f2h(kk * av), q.r[e]}) : 0u;
    x[2][e] = live ? __builtin_bit_cast(uint32_t, half2_t{q.v[e], q.v[e]}) : 0u;
    x[3][e] = __builtin_bit_cast(uint32_t, live ? decay_of(round_h(h2f(q.w12[e]) + h2f(c.w0[e]))) : 1.0f);
  }
  // NaN where something is not finite (kk a and the decay, which is never infinite: below)
  float spoil = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) spoil = __builtin_amdgcn_fdot2(as_half2(x[0][e]), half2_t{}, spoil, false);
#pragma unroll
  for (int e = 0; e < 4; e += 2) {
    spoil = __builtin_amdgcn_fdot2(half2_t{q.r[e], q.r[e + 1]}, half2_t{}, spoil, false);
    spoil = __builtin_amdgcn_fdot2(half2_t{q.v[e], q.v[e + 1]}, half2_t{}, spoil, false);
  }
  transpose4x4(x);
  const int col = 4 * n + g;  // tokens 4 wave .. 4 wave + 3 of it
  double d[4], p[4];
  auto multiply_decays = [&]() {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      d[i] = static_cast<double>(__builtin_bit_cast(float, static_cast<uint32_t>(x[3][i])));
      p[i] = i == 0 ? d[0] : p[i - 1] * d[i];
    }
  };
  multiply_decays();
  uint32_t spoilt_here = 0;
  if (__builtin_expect(__ballot(spoil != spoil || p[3] != p[3]) != 0, 0)) {  // (a gate that is not a number has made new k one)
    spoilt_here = without_spoilt_tokens(x);
    multiply_decays();
  }
  if (lane == 0) reinterpret_cast<uint32_t*>(&t.spoilt)[wave] = spoilt_here;
  t.part[wave][col] = p[3];
  lds_barrier();
  double first = 1.0, after = 1.0;  // products over the wavefronts before and behind this one
#pragma unroll
  for (int w = 0; w < 4; ++w) {  // (wave-uniform)
    if (w < wave) first *= t.part[w][col];
    if (w > wave) after *= t.part[w][col];
  }
  const double last = first * p[3];
  const uint4_t spoilt = t.spoilt;
  uint32_t lost = 0;
  if (__builtin_expect(__builtin_amdgcn_readfirstlane(spoilt[0] | spoilt[1] | spoilt[2] | spoilt[3]) != 0, 0)) {
    uint32_t all = 0, r = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t m = __builtin_amdgcn_readfirstlane(spoilt[w]);
      all |= (m & 15u) << (4 * w);
      r |= (m >> 4) << (4 * w);
    }
    lost = (0u - (all & (0u - all))) | r;  // from the first one on
  }
  const bool state_lost = lost >> 31;  // (that of r alone has no bits past the tokens)
  if (wave == 3) t.decay[col] = state_lost ? __builtin_nanf("") : static_cast<float>(last);
  double over = __builtin_amdgcn_rcp(last);  // 1 / P_s, from the last token on down
  over = fma(over, fma(-last, over, 1.0), over);
  float4_t ub, uk, tv;
#pragma unroll
  for (int i = 3; i >= 0; --i) {
    const half2_t k_a = as_half2(x[0][i]), b_r = as_half2(x[1][i]);
    const double k = static_cast<double>(h2f(k_a[0])), a = static_cast<double>(h2f(k_a[1]));
    const double b = static_cast<double>(h2f(b_r[0])), r = static_cast<double>(h2f(b_r[1]));
    const int tok = 4 * wave + i;
    t.r[tok][col] = static_cast<float>(r * (first * p[i]));
    t.a[tok][col] = static_cast<float>(a * (i == 0 ? first : first * p[i - 1]));
    t.b[tok][col] = static_cast<float>(b * over);
    t.k[tok][col] = static_cast<float>(k * over);
    ub[i] = static_cast<float>(b * after);  // P_16 / P_s
    uk[i] = static_cast<float>(k * after);
    tv[i] = h2f(as_half2(x[2][i])[0]);
    over *= d[i];
    after *= d[i];
  }
  const Pieces sk = split(uk), sb = split(ub), sv = split(tv);
  const int tile = n >> 2, at = 16 * wave + 4 * (n & 3) + g;
#pragma unroll
  for (int i = 0; i < 3; ++i) uo.kb[i][tile][at] = uint4_t{sk.p[i][0], sk.p[i][1], sb.p[i][0], sb.p[i][1]};
  uo.v[tile][at] = uint4_t{sv.p[0][0], sv.p[0][1], sv.p[1][0], sv.p[1][1]};
  return Staged{nk, lost};
}

// The four products of tokens with tokens, one per wavefront: A B^T, A K^T (s < t), R B^T, R K^T (s <= t).  The first two go through
// the solve into the state and are summed in fp64.
__device__ __forceinline__ void token_products(ChunkTiles& t, uint32_t lost, int wave, int lane) {
  const int g = lane >> 4, n = lane & 15;
  if (wave < 2) {
    const float(&y)[kTok][kRow] = wave ? t.k : t.b;
    double4_t acc = {};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4_t xs = *reinterpret_cast<const float4_t*>(&t.a[n][16 * q + 4 * g]);
      const float4_t ys = *reinterpret_cast<const float4_t*>(&y[n][16 * q + 4 * g]);
#pragma unroll
      for (int i = 0; i < 4; ++i) acc = mfma4(static_cast<double>(xs[i]), static_cast<double>(ys[i]), acc);
    }
    // lane (g, n), register i: token t = 4 i + g, token s = n
    float* dst = wave == 0 ? &t.ab[n][g] : &t.ak[g][n];
    const int step = wave == 0 ? 4 : 4 * kSquare;
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[i * step] = 4 * i + g > n ? static_cast<float>(acc[i]) : 0.0f;
  } else {
    const float(&y)[kTok][kRow] = wave == 2 ? t.b : t.k;
    float4_t acc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float4_t xs = *reinterpret_cast<const float4_t*>(&t.r[n][16 * q + 4 * g]);
      const float4_t ys = *reinterpret_cast<const float4_t*>(&y[n][16 * q + 4 * g]);
      acc[q] = float4_t{};
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[q] = mfma4(xs[i], ys[i], acc[q]);
    }
    float(&dst)[kTok][kSquare] = wave == 2 ? t.rb : t.rk;
#pragma unroll
    for (int i = 0; i < 4; ++i)  // register i: token t = 4 g + i
      dst[4 * g + i][n] = 4 * g + i >= n ? (acc[0][i] + acc[1][i]) + (acc[2][i] + acc[3][i]) : 0.0f;
    if (__builtin_expect(lost != 0, 0)) {  // the rows that make y NaN
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (lost >> (4 * g + i) & 1u) dst[4 * g + i][n] = __builtin_nanf("");
    }
  }
}

// x[t] += m[s] of lane t of the row * x[s], for every t > s, s = S0 .. : the factor is read across the row by the multiply-add itself.
// (The compiler makes a move and an add of this.  Two idle slots between a register's write and a read across lanes.)
#define RWKV_STEP(T, S) "v_fmac_f32_dpp %[x" #T "], %[m" #S "], %[x" #S "] row_newbcast:" #T " row_mask:0xf bank_mask:0xf\n\t"
#define RWKV_X(I) [x##I] "+v"(x[I])
#define RWKV_M(I) [m##I] "v"(m[I])
__device__ __forceinline__ void substitute(const float (&m)[kTok - 1], float (&x)[kTok]) {
  asm volatile("s_nop 1\n\t"
               RWKV_STEP(1, 0) RWKV_STEP(2, 0) RWKV_STEP(3, 0) RWKV_STEP(4, 0) RWKV_STEP(5, 0) RWKV_STEP(6, 0) RWKV_STEP(7, 0) RWKV_STEP(8, 0) RWKV_STEP(9, 0) RWKV_STEP(10, 0) RWKV_STEP(11, 0) RWKV_STEP(12, 0) RWKV_STEP(13, 0) RWKV_STEP(14, 0) RWKV_STEP(15, 0)
               RWKV_STEP(2, 1) RWKV_STEP(3, 1) RWKV_STEP(4, 1) RWKV_STEP(5, 1) RWKV_STEP(6, 1) RWKV_STEP(7, 1) RWKV_STEP(8, 1) RWKV_STEP(9, 1) RWKV_STEP(10, 1) RWKV_STEP(11, 1) RWKV_STEP(12, 1) RWKV_STEP(13, 1) RWKV_STEP(14, 1) RWKV_STEP(15, 1)
               RWKV_STEP(3, 2) RWKV_STEP(4, 2) RWKV_STEP(5, 2) RWKV_STEP(6, 2) RWKV_STEP(7, 2) RWKV_STEP(8, 2) RWKV_STEP(9, 2) RWKV_STEP(10, 2) RWKV_STEP(11, 2) RWKV_STEP(12, 2) RWKV_STEP(13, 2) RWKV_STEP(14, 2) RWKV_STEP(15, 2)
               RWKV_STEP(4, 3) RWKV_STEP(5, 3) RWKV_STEP(6, 3) RWKV_STEP(7, 3) RWKV_STEP(8, 3) RWKV_STEP(9, 3) RWKV_STEP(10, 3) RWKV_STEP(11, 3) RWKV_STEP(12, 3) RWKV_STEP(13, 3) RWKV_STEP(14, 3) RWKV_STEP(15, 3)
               RWKV_STEP(5, 4) RWKV_STEP(6, 4) RWKV_STEP(7, 4) RWKV_STEP(8, 4) RWKV_STEP(9, 4) RWKV_STEP(10, 4) RWKV_STEP(11, 4) RWKV_STEP(12, 4) RWKV_STEP(13, 4) RWKV_STEP(14, 4) RWKV_STEP(15, 4)
               : RWKV_X(0), RWKV_X(1), RWKV_X(2), RWKV_X(3), RWKV_X(4), RWKV_X(5), RWKV_X(6), RWKV_X(7), RWKV_X(8), RWKV_X(9), RWKV_X(10), RWKV_X(11),
                 RWKV_X(12), RWKV_X(13), RWKV_X(14), RWKV_X(15)
               : RWKV_M(0), RWKV_M(1), RWKV_M(2), RWKV_M(3), RWKV_M(4));
  asm volatile("s_nop 1\n\t"
               RWKV_STEP(6, 5) RWKV_STEP(7, 5) RWKV_STEP(8, 5) RWKV_STEP(9, 5) RWKV_STEP(10, 5) RWKV_STEP(11, 5) RWKV_STEP(12, 5) RWKV_STEP(13, 5) RWKV_STEP(14, 5) RWKV_STEP(15, 5)
               RWKV_STEP(7, 6) RWKV_STEP(8, 6) RWKV_STEP(9, 6) RWKV_STEP(10, 6) RWKV_STEP(11, 6) RWKV_STEP(12, 6) RWKV_STEP(13, 6) RWKV_STEP(14, 6) RWKV_STEP(15, 6)
               RWKV_STEP(8, 7) RWKV_STEP(9, 7) RWKV_STEP(10, 7) RWKV_STEP(11, 7) RWKV_STEP(12, 7) RWKV_STEP(13, 7) RWKV_STEP(14, 7) RWKV_STEP(15, 7)
               RWKV_STEP(9, 8) RWKV_STEP(10, 8) RWKV_STEP(11, 8) RWKV_STEP(12, 8) RWKV_STEP(13, 8) RWKV_STEP(14, 8) RWKV_STEP(15, 8)
               RWKV_STEP(10, 9) RWKV_STEP(11, 9) RWKV_STEP(12, 9) RWKV_STEP(13, 9) RWKV_STEP(14, 9) RWKV_STEP(15, 9)
               RWKV_STEP(11, 10) RWKV_STEP(12, 10) RWKV_STEP(13, 10) RWKV_STEP(14, 10) RWKV_STEP(15, 10)
               RWKV_STEP(12, 11) RWKV_STEP(13, 11) RWKV_STEP(14, 11) RWKV_STEP(15, 11)
               RWKV_STEP(13, 12) RWKV_STEP(14, 12) RWKV_STEP(15, 12)
               RWKV_STEP(14, 13) RWKV_STEP(15, 13)
               RWKV_STEP(15, 14)
               : RWKV_X(5), RWKV_X(6), RWKV_X(7), RWKV_X(8), RWKV_X(9), RWKV_X(10), RWKV_X(11),
                 RWKV_X(12), RWKV_X(13), RWKV_X(14), RWKV_X(15)
               : RWKV_M(5), RWKV_M(6), RWKV_M(7), RWKV_M(8), RWKV_M(9), RWKV_M(10), RWKV_M(11), RWKV_M(12), RWKV_M(13), RWKV_M(14));
}
#undef RWKV_STEP
#undef RWKV_X
#undef RWKV_M
// (I - [A B^T])^-1 from the left on A (wavefront 0, a column per lane) and on [A K^T] (wavefront 1, 16 of them): forward
// substitution, the factors out of a row's lanes.
__device__ __forceinline__ void solve(ChunkTiles& t, int wave, int lane) {
  if (wave > 1) return;
  float* col = wave == 0 ? &t.a[0][lane] : &t.ak[0][lane & 15];
  const int stride = wave == 0 ? kRow : kSquare;
  float m[kTok - 1], x[kTok];
#pragma unroll
  for (int s = 0; s < kTok - 1; ++s) m[s] = t.ab[s][lane & 15];
#pragma unroll
  for (int i = 0; i < kTok; ++i) x[i] = col[i * stride];
  substitute(m, x);
  if (wave == 0 || lane < 16) {
#pragma unroll
    for (int i = 1; i < kTok; ++i) col[i * stride] = x[i];
  }
}

// S diag(P_16) + (K^T V + B^T U) P_16 of a tile of 16 columns: six products of the operands' bf16 pieces, all that are not below
// the last bit of a fp32 product; the five small ones are summed apart.  (In fp64 the error is 4.6e-8 instead of 5.7e-8 and the
// products take 540 clocks instead of 100.)
__device__ __forceinline__ float4_t updated(const float4_t& S, const float4_t& p, const uint4_t (&kb)[3], const uint4_t& v, const Pieces& u) {
  const uint4_t b0 = {v[0], v[1], u.p[0][0], u.p[0][1]};
  const uint4_t b1 = {v[2], v[3], u.p[1][0], u.p[1][1]};
  const uint4_t b2 = {0, 0, u.p[2][0], u.p[2][1]};
  const float4_t big = mfma32(kb[0], b0, float4_t{});
  float4_t small = mfma32(kb[2], b0, float4_t{});
  small = mfma32(kb[0], b2, small);
  small = mfma32(kb[1], b1, small);
  small = mfma32(kb[1], b0, small);
  small = mfma32(kb[0], b1, small);
  float4_t r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = fmaf(S[i], p[i], big[i] + small[i]);
  return r;
}
// V of four tokens out of its pieces (exact)
__device__ __forceinline__ float4_t whole(const uint4_t& v) {
  float4_t r;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    r[2 * h] = __builtin_bit_cast(float, v[h] << 16) + __builtin_bit_cast(float, v[2 + h] << 16);
    r[2 * h + 1] = __builtin_bit_cast(float, v[h] & 0xffff0000u) + __builtin_bit_cast(float, v[2 + h] & 0xffff0000u);
  }
  return r;
}
__device__ __forceinline__ float4_t sum4(const float4_t& a, const float4_t& b, const float4_t& c, const float4_t& d) {
  float4_t r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = (a[i] + b[i]) + (c[i] + d[i]);
  return r;
}

// GroupNorm, bonus and gate (the formulas and rounding points of lnx_rkvres_xg_kernel, which the chain ends in; its sums are in the order of a
// lane per channel, these in that of four: the two paths' outputs differ by roundings)
__device__ __forceinline__ half4_t normalised_output(const float (&y)[4], half4_t r, half4_t k, half4_t v, half4_t gate, half4_t r_k, half4_t w,
                                                     half4_t b) {
  const float mean = row16_sum((y[0] + y[1]) + (y[2] + y[3])) * (1.0f / 64.0f);
  float d[4], rk[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    d[e] = y[e] - mean;
    rk[e] = h2f(r[e]) * h2f(k[e]);
  }
  const float var = row16_sum((d[0] * d[0] + d[1] * d[1]) + (d[2] * d[2] + d[3] * d[3])) * (1.0f / 64.0f);
  const float rkv = row16_sum((rk[0] * h2f(r_k[0]) + rk[1] * h2f(r_k[1])) + (rk[2] * h2f(r_k[2]) + rk[3] * h2f(r_k[3])));
  const float rstd = rsqrtf(var + kLnxEps);
  half4_t o;
#pragma unroll
  for (int e = 0; e < 4; ++e) o[e] = f2h((d[e] * rstd * h2f(w[e]) + h2f(b[e]) + rkv * h2f(v[e])) * h2f(gate[e]));
  return o;
}

// ---- many heads: whole ones ----------------------------------------------------------------------------------------
// One block per (sequence, head): wavefront w keeps the value rows 16 w .. 16 w + 15 of the state for the whole call, transposed,
// as four 16 x 16 tiles (lane (g, n), tile q, register i: column j = 16 q + 4 g + i, row 16 w + n) - which is also how the matrix
// core wants them as the right operand of S A'^T and S R^T, and how U leaves it and goes back in: the chain from chunk to chunk
// touches no LDS.  Four blocks per CU (40 KB of LDS, 128 registers, a few spilled); the raised priority around the products is worth 4 %.
__global__ __launch_bounds__(256, 4) void wkv7_chunk_kernel(int T, int C, int H, float* __restrict__ state, TmixSeqArgs fa,
                                                            const half_t* __restrict__ v, half_t* __restrict__ y_tap,
                                                            half_t* __restrict__ out) {
  __shared__ __align__(16) ChunkTiles t;
  __shared__ __align__(16) UpdateOperands uo;
  __shared__ __align__(8) half4_t constants[7][16];  // of the head's channels: registers are what this kernel is short of
  const int bh = blockIdx.x;
  const int bi = bh / H, h = bh - bi * H;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int tok = 4 * wave + g;
  const int ch = h * kHead + 4 * n;
  const int64_t base = static_cast<int64_t>(bi) * T * C + ch;

  float* srow = state + (static_cast<int64_t>(bh) * kHead + 16 * wave + n) * kHead + 4 * g;
  float4_t S[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) S[q] = __builtin_nontemporal_load(reinterpret_cast<const float4_t*>(srow + 16 * q));

  if (wave == 0 && g == 0) {
    const half_t* const from[7] = {fa.k_k, fa.a0, fa.k_a, fa.w0, fa.r_k, fa.lnx_w, fa.lnx_b};
#pragma unroll
    for (int i = 0; i < 7; ++i) constants[i][n] = *reinterpret_cast<const half4_t*>(from[i] + ch);
  }
  lds_barrier();

  ChunkRows next;
  half4_t gate_next;
  auto request = [&](int t0) {
    const int64_t at = base + static_cast<int64_t>(min(t0 + tok, T - 1)) * C;
    next.load(fa, v, at);
    gate_next = *reinterpret_cast<const half4_t*>(fa.g + at);
  };
  request(0);
  for (int t0 = 0; t0 < T; t0 += kTok) {
    const half4_t r4 = next.r, v4 = next.v, gate4 = gate_next;
    const bool live = t0 + tok < T;
    const Staged staged = stage_operands(t, uo, next, ChannelConstants{constants[0][n], constants[1][n], constants[2][n], constants[3][n]}, live, wave, lane);
    __builtin_amdgcn_sched_barrier(0);
    request(t0 + kTok);
    lds_barrier();
    __builtin_amdgcn_s_setprio(1);
    token_products(t, staged.lost, wave, lane);
    __builtin_amdgcn_s_setprio(0);
    lds_barrier();
    solve(t, wave, lane);
    lds_barrier();
    __builtin_amdgcn_s_setprio(1);

    // U, Y and the new state of this wavefront's 16 rows
    const uint4_t vp = uo.v[wave][lane];
    const float4_t V = whole(vp);
    float4_t part[4];
    {
      const float4_t kp = *reinterpret_cast<const float4_t*>(&t.ak[n][4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4_t x = *reinterpret_cast<const float4_t*>(&t.a[n][16 * j + 4 * g]);
        part[j] = mfma4(kp[j], V[j], float4_t{});
#pragma unroll
        for (int i = 0; i < 4; ++i) part[j] = mfma4(x[i], S[j][i], part[j]);
      }
    }
    const float4_t U = sum4(part[0], part[1], part[2], part[3]);
    __builtin_amdgcn_sched_barrier(0);
    {
      const float4_t rb = *reinterpret_cast<const float4_t*>(&t.rb[n][4 * g]);
      const float4_t rk = *reinterpret_cast<const float4_t*>(&t.rk[n][4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float4_t x = *reinterpret_cast<const float4_t*>(&t.r[n][16 * j + 4 * g]);
        part[j] = mfma4(rk[j], V[j], float4_t{});
#pragma unroll
        for (int i = 0; i < 4; ++i) part[j] = mfma4(x[i], S[j][i], part[j]);
        part[j] = mfma4(rb[j], U[j], part[j]);
      }
      const float4_t y = sum4(part[0], part[1], part[2], part[3]);
#pragma unroll
      for (int i = 0; i < 4; ++i) t.y[4 * g + i][16 * wave + n] = y[i];
    }
    const Pieces up = split(U);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      const uint4_t kb[3] = {uo.kb[0][j][lane], uo.kb[1][j][lane], uo.kb[2][j][lane]};
      S[j] = updated(S[j], *reinterpret_cast<const float4_t*>(&t.decay[16 * j + 4 * g]), kb, vp, up);
    }
    __builtin_amdgcn_s_setprio(0);
    lds_barrier();
    const float4_t y4 = *reinterpret_cast<const float4_t*>(&t.y[tok][4 * n]);
    const float yv[4] = {round_h(y4[0]), round_h(y4[1]), round_h(y4[2]), round_h(y4[3])};
    const half4_t o4 = normalised_output(yv, r4, staged.new_k, v4, gate4, constants[4][n], constants[5][n], constants[6][n]);
    if (live) {
      const int64_t at = base + static_cast<int64_t>(t0 + tok) * C;
      *reinterpret_cast<half4_t*>(out + at) = o4;
      if (y_tap) *reinterpret_cast<half4_t*>(y_tap + at) = half4_t{f2h(yv[0]), f2h(yv[1]), f2h(yv[2]), f2h(yv[3])};
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) __builtin_nontemporal_store(S[q], reinterpret_cast<float4_t*>(srow + 16 * q));
}

// ---- few heads: the chunks first, all at once, then the chain over them ---------------------------------------------
// What the chain needs of a chunk, in the order in which its lanes read it (lane (g, n), tile q of 16 columns).
struct ChunkOperands {
  UpdateOperands u;
  float4_t a[4][kWave];  // A'[n][16 q + 4 g ..]
  float4_t r[4][kWave];  // R[n][16 q + 4 g ..]
  float kp[4][kWave];    // K'[n][4 g + q]
  float rb[4][kWave];
  float rk[4][kWave];
  float decay[kHead];
};
static_assert(sizeof(ChunkOperands) == 27904, "28 KB in the figures of this file, of rwkv_hip.h and of the documents; a block of the chain reads V's "
                                               "rows of its own, 3 KB less");

// One block per (sequence, head, chunk).  Tokens t_begin .. t_end - 1 of a call of T.
__global__ __launch_bounds__(256) void wkv7_chunk_prepare_kernel(int T, int C, int H, int t_begin, int t_end, int chunks, TmixSeqArgs fa,
                                                                 const half_t* __restrict__ v, half_t* __restrict__ new_k,
                                                                 ChunkOperands* __restrict__ ws) {
  __shared__ __align__(16) ChunkTiles t;
  const int bh = blockIdx.x / chunks, chunk = blockIdx.x - bh * chunks;
  const int bi = bh / H, h = bh - bi * H;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const int ch = h * kHead + 4 * n;
  const int token = t_begin + chunk * kTok + 4 * wave + g;
  const bool live = token < t_end;
  const int64_t at = (static_cast<int64_t>(bi) * T + min(token, t_end - 1)) * C + ch;
  ChunkOperands& o = ws[blockIdx.x];
  ChunkRows q;
  q.load(fa, v, at);
  ChannelConstants c;
  c.load(fa, ch);
  const Staged staged = stage_operands(t, o.u, q, c, live, wave, lane);
  if (live) *reinterpret_cast<half4_t*>(new_k + at) = staged.new_k;
  lds_barrier();
  token_products(t, staged.lost, wave, lane);
  lds_barrier();
  solve(t, wave, lane);
  // what the solve leaves alone
  o.r[wave][lane] = *reinterpret_cast<const float4_t*>(&t.r[n][16 * wave + 4 * g]);
  o.rb[wave][lane] = t.rb[n][4 * g + wave];
  o.rk[wave][lane] = t.rk[n][4 * g + wave];
  if (wave == 3) o.decay[lane] = t.decay[lane];
  lds_barrier();
  o.a[wave][lane] = *reinterpret_cast<const float4_t*>(&t.a[n][16 * wave + 4 * g]);
  o.kp[wave][lane] = t.ak[n][4 * g + wave];
}

// One block per (sequence, head, 16 value rows), two to a CU; the blocks of a head are eight apart, which puts them on one XCD and their
// operands into its L2 once.  Wavefronts 0 .. 3 carry the state, a tile of 16 columns each: their shares of U meet in LDS, one
// barrier per chunk.  Wavefronts 4 .. 7 make Y out of the states that those leave in LDS, a chunk behind.  Operands are requested two
// chunks ahead: three need 172 registers, which leaves a CU one block (us per call, one block of 32 rows and three chunks ahead above 64
// heads / this: 96 heads x 333 tokens 50.4 / 48.4; one of 16 rows and three chunks: 64 x 2048 192 / 187, 24 x 512 38.7 / 37.0).
constexpr int kChainBlocks = kHead / 16;  // per head
__global__ __launch_bounds__(512, 4) void wkv7_chunk_chain_kernel(int heads, int T, int C, int H, int t_begin, int t_end, int chunks,
                                                                  float* __restrict__ state, const ChunkOperands* __restrict__ ws,
                                                                  const half_t* __restrict__ v, half_t* __restrict__ y) {
  __shared__ float4_t u_part[2][4][kWave], y_part[2][4][kWave], s_tile[2][4][kWave];
  const int bh = static_cast<int>(blockIdx.x / (8 * kChainBlocks) * 8 + (blockIdx.x & 7)), rows16 = blockIdx.x / 8 % kChainBlocks;
  if (bh >= heads) return;
  const int bi = bh / H, h = bh - bi * H;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int q = wave & 3;  // tile of columns
  const int lane = threadIdx.x & 63;
  const int g = lane >> 4, n = lane & 15;
  const ChunkOperands* op = ws + static_cast<int64_t>(bh) * chunks;
  auto pick = [&](const float4_t& x) { return q == 0 ? x[0] : (q == 1 ? x[1] : (q == 2 ? x[2] : x[3])); };
  constexpr int kSets = 2;

  if (wave < 4) {
    float* srow = state + (static_cast<int64_t>(bh) * kHead + 16 * rows16 + n) * kHead + 16 * q + 4 * g;
    float4_t S = *reinterpret_cast<const float4_t*>(srow);
    struct Set {
      float4_t a, p;
      float kp;
      uint4_t v, kb[3];
    };
    Set set[kSets];
    auto request = [&](Set& s, int c) {  // (chunks past the end repeat the last one)
      const ChunkOperands& o = op[min(c, chunks - 1)];
#pragma unroll
      for (int i = 0; i < 3; ++i) s.kb[i] = o.u.kb[i][q][lane];
      s.v = o.u.v[rows16][lane];
      s.a = o.a[q][lane];
      s.kp = o.kp[q][lane];
      s.p = *reinterpret_cast<const float4_t*>(&o.decay[16 * q + 4 * g]);
    };
    // this tile's share of a chunk's U, and the state that the chunk begins with
    auto begin = [&](const Set& s, int c) {
      s_tile[c & 1][q][lane] = S;
      float4_t part = mfma4(s.kp, pick(whole(s.v)), float4_t{});
#pragma unroll
      for (int i = 0; i < 4; ++i) part = mfma4(s.a[i], S[i], part);
      u_part[c & 1][q][lane] = part;
      lds_barrier();
    };
    auto turn = [&](Set& s, const Set& next, int c) {
      const float4_t(&up)[4][kWave] = u_part[c & 1];
      S = updated(S, s.p, s.kb, s.v, split(sum4(up[0][lane], up[1][lane], up[2][lane], up[3][lane])));
      request(s, c + kSets);
      begin(next, c + 1);  // (past the end: what the last turn leaves is not read)
    };
#pragma unroll
    for (int i = 0; i < kSets; ++i) request(set[i], i);
    begin(set[0], 0);
    int c = 0;
    for (; c + kSets <= chunks; c += kSets) {
#pragma unroll
      for (int u = 0; u < kSets; ++u) turn(set[u], set[(u + 1) % kSets], c + u);
    }
#pragma unroll
    for (int u = 0; u < kSets - 1; ++u)
      if (c + u < chunks) turn(set[u], set[u + 1], c + u);
    *reinterpret_cast<float4_t*>(srow) = S;
    return;
  }

  const int64_t base = (static_cast<int64_t>(bi) * T + t_begin) * C + h * kHead + 16 * rows16 + n;
  const int tokens = t_end - t_begin;
  struct Set {
    float4_t r;
    float rb, rk;
    half_t v;
  };
  Set set[kSets];
  auto request = [&](Set& s, int c) {
    c = min(c, chunks - 1);
    const ChunkOperands& o = op[c];
    s.r = o.r[q][lane];
    s.rb = o.rb[q][lane];
    s.rk = o.rk[q][lane];
    s.v = v[base + static_cast<int64_t>(min(c * kTok + 4 * g + q, tokens - 1)) * C];
  };
  // wavefront 4 + q writes the tokens 4 g + q
  auto write_out = [&](int c) {
    const int token = c * kTok + 4 * g + q;
    const float4_t(&part)[4][kWave] = y_part[c & 1];
    const float yv = (part[0][lane][q] + part[1][lane][q]) + (part[2][lane][q] + part[3][lane][q]);
    if (token < tokens) y[base + static_cast<int64_t>(token) * C] = f2h(yv);
  };
  auto turn = [&](Set& s, int c) {
    const int buf = c & 1;
    const float4_t(&up)[4][kWave] = u_part[buf];
    const float u = (up[0][lane][q] + up[1][lane][q]) + (up[2][lane][q] + up[3][lane][q]);
    const float4_t S = s_tile[buf][q][lane];
    float4_t part = mfma4(s.rk, not_finite(s.v) ? 0.0f : h2f(s.v), float4_t{});
#pragma unroll
    for (int i = 0; i < 4; ++i) part = mfma4(s.r[i], S[i], part);
    y_part[buf][q][lane] = mfma4(s.rb, u, part);
    request(s, c + kSets);
    if (c > 0) write_out(c - 1);
    lds_barrier();
  };
#pragma unroll
  for (int i = 0; i < kSets; ++i) request(set[i], i);
  lds_barrier();
  int c = 0;
  for (; c + kSets <= chunks; c += kSets) {
#pragma unroll
    for (int u = 0; u < kSets; ++u) turn(set[u], c + u);
  }
#pragma unroll
  for (int u = 0; u < kSets - 1; ++u)
    if (c + u < chunks) turn(set[u], c + u);
  write_out(chunks - 1);
}

constexpr int kSegment = 512;  // tokens that are prepared at a time: bounds the workspace

enum class ChunkPath { kNone, kWhole, kChain };

// Which calls go in chunks, and how.  us per call with everything from the rank-outs to the output projection's input:
//   heads x tokens             64 x 12   64 x 33   64 x 48   64 x 128  64 x 512  12 x 512  96 x 64  96 x 333  128 x 128
//   three kernels (token by token)  9.7      12.6      14.2      26.4      74.7      62.5     21.3      72.6       37.7
//   whole heads                     7.5      16.1      16.1      37.9     141        140      20.6       -         37.5
//   chain                          10.3      13.5      13.6      22.4      47.4      34.3     20.0      47.9       29.4
//   heads x tokens             160 x 64  160 x 128 160 x 256 192 x 128 192 x 256 192 x 512 224 x 128 224 x 256 320 x 128
//   whole heads                    20.9      37.5      72.0      38.0      72.3     140.6      38.3      72.2      55.6
//   chain                          26.6      35.1      57.6      37.9      60.8     126.4      42.2      71.2      52.7
//   heads x tokens             256 x 8   256 x 16  256 x 17  256 x 128  512 x 64  1024 x 128  2048 x 64
//   one fused kernel (t. by t.)     7.1      11.4      13.1      67.5       52.0      166        160
//   whole heads                     8.0       8.1      12.6      39.0       33.0       92.9       95.3
// A chunk costs the same with one token in it as with sixteen.  The chain needs three launches and pays from a few chunks on, as
// long as there are CUs for the blocks of a head; with more heads the kernel for whole ones has work for every CU (the few percent
// around 320 heads, whose blocks are a round and a quarter, are not worth 28 KB per head and chunk).  Three prompts of the 7.2B shape,
// whole heads / chain, ms a pass: 128 tokens 8.30 / 8.29, 256 14.80 / 14.44, 512 26.2 / 26.2.
// Whole heads pay for the tokens that a last chunk has not: us per layer of a model, chunks less token by token, 17 / 18 / 20 / 21 tokens: 192
// heads -0.1 / -0.4 / -1.3 / -, 320 1.6 / 1.1 / 0.7 / -, 384 1.4 / 1.2 / 0.2 / -0.7, 512 1.1 / 1.0 / 0.2 / -, 1024 -0.5 / -1.4 / -3.1 / -, 2048 0.6 / -1.5 /
// -5.2 / - (up to 512 heads the fused kernel has two of them on a CU); 96 heads 26 / 32 / 42 / 48 / 58 / 63 tokens -1.3 / -1.3 / 2.1 / 1.0 / 3.1 / 1.6,
// 128 heads -1.1 / -0.6 / 0.1 / -0.1 / 2.8 / 1.9.  A chain of four chunks, 48 / 49 / 64 / 65 tokens: 12 heads -0.8 / -0.7 / -1.0 / -0.8, 32 -0.5 / 0.6 / -0.3 /
// 0.0, 48 0.6 / 0.0 / -1.1 / -0.9, 64 0.6 / 0.8 / -0.6 / -0.1.
ChunkPath chunk_path(int heads, int T) {
  if (T < 10) return ChunkPath::kNone;
  if (T <= kTok) return ChunkPath::kWhole;
  if (heads > 128 && T <= (heads > 256 && heads <= 512 ? 20 : 17)) return ChunkPath::kNone;
  if (heads > 192 || (heads > 128 && T < 128)) return ChunkPath::kWhole;
  if (heads <= 32) return T >= 48 ? ChunkPath::kChain : ChunkPath::kNone;
  if (T >= 64) return ChunkPath::kChain;
  return heads > 64 && T >= 26 && T <= 32 ? ChunkPath::kWhole : ChunkPath::kNone;
}

}  // namespace

bool tmix_chunk_pays(int B, int T, int H, const TmixSeqArgs& fa) {
  uintptr_t bits = 0;  // rows of four channels are read at once
  for (const half_t* p : {fa.r, fa.k, fa.a12, fa.w12, fa.g, fa.k_k, fa.a0, fa.k_a, fa.w0, fa.r_k, fa.lnx_w, fa.lnx_b})
    bits |= reinterpret_cast<uintptr_t>(p);
  return bits % sizeof(half4_t) == 0 && chunk_path(B * H, T) != ChunkPath::kNone;
}

bool tmix_chunk_chains(int B, int T, int H) { return chunk_path(B * H, T) == ChunkPath::kChain; }

size_t tmix_chunk_workspace_bytes(int B, int T, int H) {
  if (!tmix_chunk_chains(B, T, H)) return 0;
  return sizeof(ChunkOperands) * B * H * ceil_div(std::min(T, kSegment), kTok);
}

int tmix_chunk_launch(hipStream_t st, int B, int T, int C, int H, float* state, const TmixSeqArgs& fa, const half_t* v, void* workspace,
                      half_t* new_k, half_t* y, bool want_y, half_t* y2) {
  const int heads = B * H;
  if (chunk_path(heads, T) == ChunkPath::kWhole) {
    hipLaunchKernelGGL(wkv7_chunk_kernel, dim3(heads), dim3(256), 0, st, T, C, H, state, fa, v, want_y ? y : nullptr, y2);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
  }
  RWKV_REQUIRE(workspace, "tmix_chunk: no workspace");
  ChunkOperands* ws = static_cast<ChunkOperands*>(workspace);
  for (int t0 = 0; t0 < T; t0 += kSegment) {
    const int t1 = std::min(T, t0 + kSegment);
    const int chunks = ceil_div(t1 - t0, kTok);
    hipLaunchKernelGGL(wkv7_chunk_prepare_kernel, dim3(heads * chunks), dim3(256), 0, st, T, C, H, t0, t1, chunks, fa, v, new_k, ws);
    RWKV_LAUNCH_CHECK();
    hipLaunchKernelGGL(wkv7_chunk_chain_kernel, dim3(ceil_div(heads, 8) * 8 * kChainBlocks), dim3(512), 0, st, heads, T, C, H, t0, t1, chunks, state,
                       ws, v, y);
    RWKV_LAUNCH_CHECK();
  }
  return lnx_launch(st, static_cast<int64_t>(B) * T * H, H, y, fa.r, new_k, v, fa.r_k, fa.lnx_w, fa.lnx_b, fa.g, y2);
}

}  // namespace rwkv
