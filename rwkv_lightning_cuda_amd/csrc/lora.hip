// LoRA pairs of the RWKV-7 time-mix block (decay w, in-context rate a, gate g, value residual v).
//
// Reference: rank-in cuda/rwkv7_v3a_ops.cu:813-940 (fp32 dot over C, fp16 hidden), rank-out
// :942-1130 (tanh / sigmoid applied to the fp16 hidden in fp32 and NOT re-rounded, fp32 dot over the
// rank, v-residual gate fused for the v group :1118-1123); unfused variants :209-367,685-811,1132-1270;
// dispatch src/rwkv7_fast_v4.cu:961-1014,1217-1260.
//
// rank-in is a plain small-N linear layer over fp16 weights [R,C] and reuses the GEMV / streaming GEMM kernels.
//
// rank-out is out[M,C] = act(h[M,R]) . W2[C,R]^T: a short reduction (R = 32..512) and many outputs, on
// v_mfma_f32_32x32x16_f16.  The activated hidden stays fp32 in the reference, so it enters the matrix core as
// two fp16 terms, hi = f16(a) and lo = f16(a - hi): hi + lo carries 22 bits of a, both products with the fp16
// weight are exact in fp32, and the result differs from an fp32 dot only by summation order.  Without an
// activation the hidden is fp16 already and the lo term is skipped.  One launch takes up to four problems
// (w, a, g, v of a layer): grid = (C/128, row tiles, problems), block = 2 groups of 4 wavefronts x 32 output
// channels (the groups take alternate 16-wide steps of the rank and add up through LDS), the 32 x R slice of
// act(h) of a row tile staged in LDS; many rows take wider blocks (lora_out_wide_kernel).
#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "ops.h"

namespace rwkv {

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kLoraMaxR = 512;
constexpr int kLoraRows = 32;   // rows per block: one MFMA tile
constexpr int kLoraCols = 128;  // output channels per block: 32 per wavefront
constexpr int kLoraKG = 2;       // wavefront groups that split the rank between them (even / odd 16-wide steps)
constexpr int kLoraThreads = 2 * kLoraCols * kLoraKG;
constexpr int kLoraStage = (kLoraRows * (kLoraMaxR / 8 + 1) + kLoraThreads - 1) / kLoraThreads;  // pieces per thread

// Eight values of the hidden, activated, as two fp16 terms; exact zeros where `live` is not set.
template <int ACT>
__device__ __forceinline__ void activate8(const uint4_t& raw, bool live, uint4_t& hi, uint4_t& lo) {
  const half8_t x = __builtin_bit_cast(half8_t, raw);
  half8_t h, l;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float f = h2f(x[e]);
    if constexpr (ACT == RWKV_ACT_TANH) f = tanh_f(f);
    if constexpr (ACT == RWKV_ACT_SIGMOID) f = sigmoid_f(f);
    h[e] = f2h(f);
    l[e] = f2h(f - h2f(h[e]));
  }
  hi = __builtin_bit_cast(uint4_t, h);
  lo = __builtin_bit_cast(uint4_t, l);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    hi[e] = live ? hi[e] : 0u;
    lo[e] = live ? lo[e] : 0u;
  }
}
// The choice of the activation stands around eight values or more: asked per value it kept the exponentials and reciprocals of a thread
// in line one behind the other (us of the four problems of a layer, weights out of HBM, per value / around: 4096 channels, 250 rows 11.5 /
// 10.9, 2048 rows 56.3 / 54.5; 2048 channels, 333 rows 8.5 / 8.0, 192 rows 6.0 / 5.5).
template <typename Stage>
__device__ __forceinline__ void with_activation(int act, Stage stage) {
  if (act == RWKV_ACT_TANH) stage(std::integral_constant<int, RWKV_ACT_TANH>{});
  else if (act == RWKV_ACT_SIGMOID) stage(std::integral_constant<int, RWKV_ACT_SIGMOID>{});
  else stage(std::integral_constant<int, RWKV_ACT_NONE>{});
}

// Every lane requests its whole weight row (up to 16 pieces of 8), its pieces of the 32 x R hidden slice and its
// piece of the epilogue operands (v, v_first) in one go; the block turns the hidden slice into hi / lo fp16 in LDS (one barrier), each
// wavefront runs its MFMA steps, both groups lay their 32 x 128 sums out in LDS (over the hi / lo tiles, free by
// then) and all threads add the two in group order, apply the epilogue and write 16 bytes of a row each.
//
// Every load is issued without a per-lane branch around it: addresses past the rank or the last row are clamped to
// a valid one and the value is dropped afterwards.  (A load under a per-lane branch, or merged with a default
// value, makes the compiler wait for all loads in flight inside the branch: the trips to memory then run one
// after the other.)  Conditions that are the same for a whole wavefront cost nothing of the kind.
//
// LDS rows are R + 8 halves apart: for ranks that are multiples of 16 the ds_read_b128 of lane (j, h) at
// j * (2R + 16) + 16h bytes is conflict-free (other ranks lose some LDS bandwidth), and the zeroed 8-half pad is
// what the last MFMA step of a rank that is not a multiple of 16 reads (its weights are the clamped, finite ones).
constexpr int kLoraOutLd = kLoraCols + 4;  // fp32 row of the output tile in LDS

__global__ __launch_bounds__(kLoraThreads) void lora_out_kernel(LoraOutMultiArgs a) {
  __shared__ __attribute__((aligned(16))) half_t hi_s[kLoraRows * (kLoraMaxR + 8)];
  __shared__ __attribute__((aligned(16))) half_t lo_s[kLoraRows * (kLoraMaxR + 8)];
  static_assert(kLoraRows * kLoraOutLd * 4 <= kLoraRows * (kLoraMaxR + 8) * 2, "output tile exceeds the hidden tile");
  const LoraOutProblem& p = a.p[blockIdx.z];
  const int R = p.R;
  const int ld = R + 8;
  // wavefront-wide values, said so to the compiler: conditions on them become scalar branches
  const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
  const int kg = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);  // its share of the rank: steps kg, kg + 2, ...
  const int lane = threadIdx.x & 63;
  const int j = lane & 31;
  const int h = lane >> 5;
  const int c = blockIdx.x * kLoraCols + wave * 32 + j;
  const bool split = p.act != RWKV_ACT_NONE;
  const half_t* wrow = p.w2 + static_cast<int64_t>(c < a.C ? c : a.C - 1) * R;
  // packed weights: one 1 KiB piece per wavefront and rank step, consecutive lanes 16 bytes apart.  (Out of the
  // [C,R] matrix the 64 lanes of a request touch 64 different cache lines, and the address unit takes four times
  // as long over it.)
  const int steps = (R + 15) >> 4;
  const half_t* wpk = p.w2p ? p.w2p + (static_cast<int64_t>(blockIdx.x * (kLoraCols / 32) + wave) * steps * 64 + lane) * 8 : nullptr;

  // this lane's W2 values: k = 16*step + 8h .. +8 of output channel c
  constexpr int kSteps = kLoraMaxR / 16 / kLoraKG;
  half8_t w[kSteps];
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    const int k0 = (i * kLoraKG + kg) * 16;  // the same for the whole wavefront
    if (k0 < R) {
      const int k = k0 + h * 8;
      w[i] = *reinterpret_cast<const half8_t*>(wpk ? wpk + static_cast<int64_t>(i * kLoraKG + kg) * 512 : wrow + (k < R ? k : R - 8));
    }
  }

  // the epilogue's view of the tile: thread t owns channels 8*(t%16) .. +8 of row t/16
  const int orow = threadIdx.x >> 4;
  const int ocol = blockIdx.x * kLoraCols + (threadIdx.x & 15) * 8;
  const bool ocol_ok = ocol < a.C;
  // without a bias any readable address does (C values of W2); the values are dropped in the epilogue
  uint4_t bias_raw = *reinterpret_cast<const uint4_t*>((p.bias ? p.bias : p.w2) + (ocol_ok ? ocol : 0));

  const int m0 = blockIdx.y * kLoraRows;
  const int mn = min(kLoraRows, a.M - m0);
  // As many threads per row as the rows (their power of two) leave, so that few rows take one turn of the threads and none is spent on
  // the pad.  Rows that do not exist are not staged: what lies there meets rows of the product that are not stored.  (us of the four
  // problems, all 32 rows staged piece by piece / this: 4096 channels, 8 rows 7.5 / 6.2, 64 rows 7.9 / 7.8, 125 rows 8.8 / 8.4; 2048
  // channels, 13 rows 5.0 / 4.2, 128 rows 5.4 / 5.0; 768 channels, 50 rows 4.3 / 3.8.  Of the 6.5 us of a rank-480 gate alone at 32 rows
  // two are activations, which every 128 channels make again.)
  const int tpr_log = 9 - (mn > 1 ? 32 - __builtin_clz(mn - 1) : 0);
  static_assert(kLoraThreads == 512, "threads per row");
  const int hrow = threadIdx.x >> tpr_log;
  const int ks0 = (threadIdx.x & ((1 << tpr_log) - 1)) * 8;
  const half_t* hsrc = p.h + static_cast<int64_t>(m0 + (hrow < mn ? hrow : mn - 1)) * R;
  uint4_t hv[kLoraStage];
#pragma unroll
  for (int i = 0; i < kLoraStage; ++i) {
    const int ks = ks0 + ((i * 8) << tpr_log);
    if ((i * 8) << tpr_log < R) hv[i] = *reinterpret_cast<const uint4_t*>(hsrc + (ks < R ? ks : R - 8));
  }
  const int64_t o = static_cast<int64_t>(m0 + (orow < mn ? orow : mn - 1)) * a.C + (ocol_ok ? ocol : 0);
  // without the v-residual gate: the output row itself, readable and unused
  half8_t v8 = *reinterpret_cast<const half8_t*>((p.vres ? p.v : p.out) + o);
  half8_t vf8 = *reinterpret_cast<const half8_t*>((p.vres ? p.v_first : p.out) + o);
  __builtin_amdgcn_sched_barrier(0);
  // keeps the conversion of the bias below the loads above: moved up beside its own load, it would wait for the
  // weights before the hidden slice is even requested
  asm volatile("" : "+v"(bias_raw));
  const half8_t bias8 = __builtin_bit_cast(half8_t, bias_raw);

#pragma unroll
  for (int i = 0; i < kLoraStage; ++i) {
    if ((i * 8) << tpr_log < R) {
      const int ks = ks0 + ((i * 8) << tpr_log);
      uint4_t hi, lo;
      with_activation(p.act, [&](auto act_c) { activate8<decltype(act_c)::value>(hv[i], true, hi, lo); });
      if (ks < R) {
        *reinterpret_cast<uint4_t*>(&hi_s[hrow * ld + ks]) = hi;
        if (split) *reinterpret_cast<uint4_t*>(&lo_s[hrow * ld + ks]) = lo;
      }
    }
  }
  if (ks0 == 0) {  // the pad holds exact zeros
    *reinterpret_cast<half8_t*>(&hi_s[hrow * ld + R]) = half8_t{};
    if (split) *reinterpret_cast<half8_t*>(&lo_s[hrow * ld + R]) = half8_t{};
  }
  __syncthreads();

  float16_t acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
#pragma unroll
  for (int i = 0; i < kSteps; ++i) {
    const int k = (i * kLoraKG + kg) * 16;
    if (k < R) {
      const half8_t ah = *reinterpret_cast<const half8_t*>(&hi_s[j * ld + k + h * 8]);
      acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, w[i], acc, 0, 0, 0);
      if (split) {
        const half8_t al = *reinterpret_cast<const half8_t*>(&lo_s[j * ld + k + h * 8]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, w[i], acc, 0, 0, 0);
      }
    }
  }
  __syncthreads();  // the hidden tiles are free: group 0 lays its sums over hi_s, group 1 over lo_s
  // accumulator v of lane (j, h): row 8*(v/4) + 4h + v%4, column wave*32 + j
  float* tile = reinterpret_cast<float*>(kg == 0 ? hi_s : lo_s);
#pragma unroll
  for (int v = 0; v < 16; ++v) tile[(8 * (v / 4) + 4 * h + (v % 4)) * kLoraOutLd + wave * 32 + j] = acc[v];
  __syncthreads();

  const float* t0 = reinterpret_cast<const float*>(hi_s) + orow * kLoraOutLd + (threadIdx.x & 15) * 8;
  const float* t1 = reinterpret_cast<const float*>(lo_s) + orow * kLoraOutLd + (threadIdx.x & 15) * 8;
  float sum[8];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const float4_t s0 = *reinterpret_cast<const float4_t*>(t0 + 4 * q);
    const float4_t s1 = *reinterpret_cast<const float4_t*>(t1 + 4 * q);
#pragma unroll
    for (int e = 0; e < 4; ++e) sum[4 * q + e] = s0[e] + s1[e];
  }
  half8_t res;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float b = p.bias ? h2f(bias8[e]) : 0.0f;
    if (p.vres) {
      const float vv = h2f(v8[e]);
      const float gate = sigmoid_f(b + sum[e]);
      res[e] = f2h(vv + (h2f(vf8[e]) - vv) * gate);
    } else {
      res[e] = f2h(sum[e] + b);
    }
  }
  if (orow < mn && ocol_ok) *reinterpret_cast<half8_t*>(p.out + o) = res;
}

// The same products for many rows.  The kernel above evaluates the activation of a hidden value once per 128 output channels
// and takes the sums through LDS and two barriers; this one takes 32 rows x 32*NW channels per block.  The weights are the
// A operand: accumulator v of lane (j, h) is row j of the tile, and the channels are dealt to A's rows so that a lane's 16
// values are 16 consecutive channels (16*h + v of the wavefront's 32) and leave in 16-byte stores straight from the registers.
// A wavefront walks the whole rank with the weights of eight steps in flight (16 wavefronts: four, which their registers allow; with
// four the 8-wavefront block takes 14.2 us instead of 12.1 for 125 rows in a 7.2B prefill, whose weights come out of HBM); its sums are built as above (even and odd
// steps apart, hi before lo, then added), so the bits are the same.
// Per rank step a CU's wavefronts ask as many cycles of LDS (the hidden) and of the vector memory path (the weights) as of
// the matrix core.  Tiles of 64 rows or 64 channels per wavefront ask for half of one of them and lose as much to occupancy
// (2048 rows x 4096 channels, ranks 128 / 128 / 480 / 96: 66-92 us against 57).
template <int NW>
__global__ __launch_bounds__(NW * 64) void lora_out_wide_kernel(LoraOutMultiArgs a) {
  extern __shared__ __align__(16) unsigned char lds_raw[];
  constexpr int kTpr = NW * 64 / kLoraRows;                      // threads that stage one row
  constexpr int kStage = (kLoraMaxR / 8 + 1 + kTpr - 1) / kTpr;  // pieces of 8 per thread, the zeroed pad among them
  constexpr int kDepth = NW == 8 ? 8 : 4;                        // rank steps whose weights are in flight
  const LoraOutProblem& p = a.p[blockIdx.z];
  const int R = p.R;
  const int ld = R + 8;
  const int steps = (R + 15) >> 4;
  const bool split = p.act != RWKV_ACT_NONE;
  half_t* hi_s = reinterpret_cast<half_t*>(lds_raw);
  half_t* lo_s = hi_s + kLoraRows * ld;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int j = lane & 31;
  const int h = lane >> 5;
  const int m0 = blockIdx.y * kLoraRows;
  const int mn = min(kLoraRows, a.M - m0);
  const int c0 = (blockIdx.x * NW + wave) * 32;  // the wavefront's channels
  const bool busy = c0 < a.C;                    // C % 32 == 0: all of them exist, or none

  // this lane's row of A
  const int cl = 16 * ((j >> 2) & 1) + 4 * (j >> 3) + (j & 3);
  const half_t* wp = p.w2p ? p.w2p + (static_cast<int64_t>(busy ? c0 >> 5 : 0) * steps * 64 + cl + 32 * h) * 8
                           : p.w2 + static_cast<int64_t>(busy ? c0 + cl : cl) * R + 8 * h;
  const int stride = p.w2p ? 512 : 16;
  // the half step past a rank of 8 mod 16 meets zeros of the hidden: any finite weights do (the packed ones exist and are zero)
  const int tail = !p.w2p && h && (R & 15) ? 8 : 0;
  half8_t w[kDepth];
  auto request = [&](int s) { return *reinterpret_cast<const half8_t*>(wp + s * stride - (s == steps - 1 ? tail : 0)); };

  // the hidden slice is requested first, then the weights of the first steps, all without a branch per lane (see above)
  {
    const int row = threadIdx.x / kTpr;
    const int ks0 = (threadIdx.x % kTpr) * 8;
    const half_t* src = p.h + static_cast<int64_t>(m0 + (row < mn ? row : mn - 1)) * R;
    uint4_t hv[kStage];
#pragma unroll
    for (int i = 0; i < kStage; ++i) {
      const int ks = ks0 + i * kTpr * 8;
      if (i * kTpr * 8 <= R) hv[i] = *reinterpret_cast<const uint4_t*>(src + (ks < R ? ks : R - 8));
    }
#pragma unroll
    for (int u = 0; u < kDepth; ++u) w[u] = request(min(u, steps - 1));
    with_activation(p.act, [&](auto act_c) {
      constexpr int kAct = decltype(act_c)::value;
#pragma unroll
      for (int i = 0; i < kStage; ++i) {
        if (i * kTpr * 8 <= R) {
          const int ks = ks0 + i * kTpr * 8;
          uint4_t hi, lo;
          activate8<kAct>(hv[i], row < mn && ks < R, hi, lo);  // rows past M and the pad hold exact zeros
          if (ks <= R) {
            *reinterpret_cast<uint4_t*>(&hi_s[row * ld + ks]) = hi;
            if constexpr (kAct != RWKV_ACT_NONE) *reinterpret_cast<uint4_t*>(&lo_s[row * ld + ks]) = lo;
          }
        }
      }
    });
  }
  __syncthreads();
  if (!busy) return;

  float16_t acc[2];  // even and odd rank steps
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[0][v] = acc[1][v] = 0.0f;
  const half_t* hp = hi_s + j * ld + 8 * h;
  const half_t* lp = lo_s + j * ld + 8 * h;
  for (int s0 = 0; s0 < steps; s0 += kDepth) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) {
      const int s = s0 + u;
      if (s < steps) {  // the same for the whole block
        acc[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[u], *reinterpret_cast<const half8_t*>(hp + 16 * s), acc[u & 1], 0, 0, 0);
        if (split)
          acc[u & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[u], *reinterpret_cast<const half8_t*>(lp + 16 * s), acc[u & 1], 0, 0, 0);
        w[u] = request(min(s + kDepth, steps - 1));
      }
    }
  }

  if (j >= mn) return;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int c = c0 + 16 * h + 8 * q;
    const int64_t o = static_cast<int64_t>(m0 + j) * a.C + c;
    half8_t bias8 = {}, v8 = {}, vf8 = {}, res;
    if (p.bias) bias8 = *reinterpret_cast<const half8_t*>(p.bias + c);
    if (p.vres) {
      v8 = *reinterpret_cast<const half8_t*>(p.v + o);
      vf8 = *reinterpret_cast<const half8_t*>(p.v_first + o);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float sum = acc[0][8 * q + e] + acc[1][8 * q + e];
      const float b = p.bias ? h2f(bias8[e]) : 0.0f;
      if (p.vres) {
        const float vv = h2f(v8[e]);
        res[e] = f2h(vv + (h2f(vf8[e]) - vv) * sigmoid_f(b + sum));
      } else {
        res[e] = f2h(sum + b);
      }
    }
    *reinterpret_cast<half8_t*>(p.out + o) = res;
  }
}

// the longest problem first: its blocks would be the launch's tail otherwise
static LoraOutMultiArgs longest_first(const LoraOutMultiArgs& a) {
  LoraOutMultiArgs o = a;
  const auto cost = [](const LoraOutProblem& p) { return p.R * (p.act != RWKV_ACT_NONE ? 2 : 1); };
  std::stable_sort(o.p, o.p + o.n, [&](const LoraOutProblem& x, const LoraOutProblem& y) { return cost(x) > cost(y); });
  return o;
}

template <int NW>
int lora_out_wide_launch(hipStream_t st, const LoraOutMultiArgs& a) {
  const LoraOutMultiArgs o = longest_first(a);
  size_t lds = 0;
  for (int i = 0; i < o.n; ++i)
    lds = std::max(lds, static_cast<size_t>(kLoraRows) * (o.p[i].R + 8) * (o.p[i].act != RWKV_ACT_NONE ? 4 : 2));
  if (lds > 65536)
    RWKV_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(&lora_out_wide_kernel<NW>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds)));
  hipLaunchKernelGGL((lora_out_wide_kernel<NW>), dim3(ceil_div(o.C, 32 * NW), ceil_div(o.M, kLoraRows), o.n), dim3(NW * 64), lds, st, o);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

__global__ __launch_bounds__(256) void lora_pack_w2_kernel(int C, int R, const half_t* __restrict__ w2, half_t* __restrict__ packed,
                                                           int64_t n_pieces) {
  const int64_t piece = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;  // (band, step, lane)
  if (piece >= n_pieces) return;
  const int steps = (R + 15) >> 4;
  const int lane = static_cast<int>(piece & 63);
  const int step = static_cast<int>((piece >> 6) % steps);
  const int band = static_cast<int>((piece >> 6) / steps);
  const int c = band * 32 + (lane & 31);
  const int k = step * 16 + (lane >> 5) * 8;
  half8_t v;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = static_cast<half_t>(0.0f);
  if (c < C && k < R) v = *reinterpret_cast<const half8_t*>(w2 + static_cast<int64_t>(c) * R + k);  // R % 8 == 0
  *reinterpret_cast<half8_t*>(packed + piece * 8) = v;
}

// Whole column blocks of the rank-out kernel (kLoraCols channels = four 32-channel bands): the wavefronts of the
// last block read their bands without a clamp, so the bands past C exist and hold zeros.
size_t lora_pack_w2_halfs(int C, int R) {
  return static_cast<size_t>(ceil_div(C, kLoraCols)) * (kLoraCols / 32) * ((R + 15) >> 4) * 512;
}

int lora_pack_w2_launch(hipStream_t st, int C, int R, const half_t* w2, half_t* packed) {
  RWKV_REQUIRE(C > 0 && R > 0 && R % 8 == 0 && w2 && packed, "lora_pack_w2: bad arguments (C=%d, R=%d)", C, R);
  const int64_t n_pieces = static_cast<int64_t>(lora_pack_w2_halfs(C, R) / 8);
  hipLaunchKernelGGL(lora_pack_w2_kernel, dim3(static_cast<unsigned>((n_pieces + 255) / 256)), dim3(256), 0, st, C, R, w2, packed,
                     n_pieces);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int lora_out_multi(hipStream_t st, const LoraOutMultiArgs& a) {
  RWKV_REQUIRE(a.n >= 1 && a.n <= 4, "lora_out: %d problems (1..4)", a.n);
  RWKV_REQUIRE(a.M > 0 && a.C > 0 && a.C % 32 == 0, "lora_out: C (%d) must be a positive multiple of 32", a.C);
  for (int i = 0; i < a.n; ++i) {
    const LoraOutProblem& p = a.p[i];
    RWKV_REQUIRE(p.R > 0 && p.R % 8 == 0 && p.R <= kLoraMaxR, "lora_out: rank %d must be a multiple of 8, at most %d",
                 p.R, kLoraMaxR);
    RWKV_REQUIRE(p.h && p.w2 && p.out, "lora_out: NULL tensor");
    RWKV_REQUIRE(!p.vres || (p.v && p.v_first && p.bias), "lora_out: v-residual gate needs v, v_first and v0");
    RWKV_REQUIRE((reinterpret_cast<uintptr_t>(p.h) | reinterpret_cast<uintptr_t>(p.w2) | reinterpret_cast<uintptr_t>(p.out) |
                  reinterpret_cast<uintptr_t>(p.bias) | reinterpret_cast<uintptr_t>(p.v) |
                  reinterpret_cast<uintptr_t>(p.v_first) | reinterpret_cast<uintptr_t>(p.w2p)) % 16 == 0,
                 "lora_out: tensors must be 16-byte aligned");
  }
  // the grid's second dimension ends at 65535
  constexpr int kMostRows = 65535 * kLoraRows;
  if (a.M > kMostRows) {
    LoraOutMultiArgs part = a;
    for (int m0 = 0; m0 < a.M; m0 += part.M) {
      part.M = std::min(kMostRows, a.M - m0);
      for (int i = 0; i < a.n; ++i) {
        part.p[i].h = a.p[i].h + static_cast<int64_t>(m0) * a.p[i].R;
        part.p[i].out = a.p[i].out + static_cast<int64_t>(m0) * a.C;
        if (a.p[i].vres) {
          part.p[i].v = a.p[i].v + static_cast<int64_t>(m0) * a.C;
          part.p[i].v_first = a.p[i].v_first + static_cast<int64_t>(m0) * a.C;
        }
      }
      const int rc = lora_out_multi(st, part);
      if (rc != RWKV_OK) return rc;
    }
    return RWKV_OK;
  }
  // As long as all blocks of the small tile are on the chip at once, two per CU, it is the faster one (its rank is walked by two groups
  // of wavefronts, all weights of which are requested at once); past that, what the blocks repeat counts.  us of the four problems of a
  // layer, weights out of HBM, small tile / 32 x 256: 4096 channels, 64 rows (256 blocks) 7.8 / 11.2, 96 (384) 8.7 / 11.3, 125 (512) 8.4 /
  // 11.3, 192 (768) 12.1 / 11.9; 2560 channels, 190 rows (480) 7.0 / 8.3; 2048 channels, 256 rows (512) 6.3 / 7.4, 333 (704) 9.3 / 8.0; 768
  // channels, 512 rows (384) 4.9 / 5.8, 768 (576) 7.3 / 6.9.
  const int row_tiles = ceil_div(a.M, kLoraRows);
  const int64_t cus = device_cu_count();
  const int64_t small = static_cast<int64_t>(ceil_div(a.C, kLoraCols)) * row_tiles * a.n;
  // A problem on its own, whose blocks all take as long, runs in rounds of a block per CU, and from rank 128 on a round of the 32 x
  // 256 tile is as long as two of the small one: it is taken where it needs no more than half as many.  us, small tile / 32 x 256, rank
  // 128 without activation: 4096 channels, 500 rows (2 rounds / 1) 6.3 / 6.7, 700 (3 / 2) 8.5 / 10.7, 1000 (4 / 2) 10.5 / 11.1, 1200 (5 / 3)
  // 12.2 / 15.1; rank 480 with one 11.6 / 11.7, 15.5 / 16.7, 19.6 / 19.3, 23.2 / 24.9; rank 96 with one, 700 rows 8.5 / 7.5.
  const int64_t wide8 = static_cast<int64_t>(ceil_div(a.C, 256)) * row_tiles;
  const bool uneven = a.n == 1 && a.p[0].R >= 128 && 2 * ((wide8 + cus - 1) / cus) > (small + cus - 1) / cus;
  if (a.n == 1 ? small * 2 > 3 * cus : small > 2 * cus) {
    // twice as many channels per block where that still leaves two blocks per CU and no channel of a block unused: 32 x 256 / 32 x
    // 512 at 4096 channels and 500 rows 21.4 / 19.2, 1000 39.0 / 37.4, 2048 68.4 / 57.9; 2048 channels and 999 rows 17.9 / 13.1, 2048
    // 29.2 / 28.7 (before, with the small tile's blocks walking several row tiles: 33.7, 60.5, 107.6; 26.5, 50.1)
    const bool wide = a.C % 512 == 0 && static_cast<int64_t>(a.C / 512) * row_tiles * a.n >= 2 * cus;
    if (wide) return lora_out_wide_launch<16>(st, a);
    if (!uneven) return lora_out_wide_launch<8>(st, a);
  }
  // (with fewer blocks the last ones would share a CU with the first, the longest)
  const LoraOutMultiArgs o = 2 * small >= 3 * cus ? longest_first(a) : a;
  hipLaunchKernelGGL(lora_out_kernel, dim3(ceil_div(o.C, kLoraCols), row_tiles, o.n), dim3(kLoraThreads), 0, st, o);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

}  // namespace rwkv

using namespace rwkv;

extern "C" {

int rwkv_hip_lora_in(rwkv_stream_t s, int M, int C, int R, const void* x, const void* w1, void* h) {
  RWKV_REQUIRE(x && w1 && h, "lora_in: NULL tensor");
  return linear_any_m(as_stream(s), RWKV_FMT_F16, M, R, C, static_cast<const half_t*>(x), w1, nullptr, nullptr,
                      RWKV_EPI_NONE, 0, h);
}

int rwkv_hip_lora_out(rwkv_stream_t s, int M, int C, int R, int act, const void* h, const void* w2, const void* bias,
                      int vres, const void* v, const void* v_first, void* out) {
  RWKV_REQUIRE(act == RWKV_ACT_NONE || act == RWKV_ACT_TANH || act == RWKV_ACT_SIGMOID, "lora_out: bad act %d", act);
  LoraOutMultiArgs a = {};
  LoraOutProblem& p = a.p[0];
  p.h = static_cast<const half_t*>(h);
  p.w2 = static_cast<const half_t*>(w2);
  p.bias = static_cast<const half_t*>(bias);
  p.v = static_cast<const half_t*>(v);
  p.v_first = static_cast<const half_t*>(v_first);
  p.out = static_cast<half_t*>(out);
  p.R = R; p.act = act; p.vres = vres;
  a.n = 1; a.M = M; a.C = C;
  return lora_out_multi(as_stream(s), a);
}

}  // extern "C"
