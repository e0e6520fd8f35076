// WKV7 time-mix recurrence for gfx950, fp32 state.
//
// Reference semantics: cuda/rwkv7_wkv_fp32_v2.cu:100-126 (per token, thread i owns state row i):
//   sa = sum_j S[i][j]*a[j];  S[i][j] = S[i][j]*d[j] + sa*b[j] + k[j]*v[i];  y[i] = sum_j S[i][j]*r[j]
// with the decay map d = exp(-e^-1/2 * sigmoid(w)) of :13-14,26-28.
//
// Lanes keep a few rows x 4 or 8 columns of the 64 x 64 state in registers for the whole call.  The per-column operands of a
// token are staged in LDS and each lane reads only the columns it owns; the two row sums of a step (sa and y) are reduced over
// the lanes that share a row with DPP adds.  The staging converts what the caller has (raw decay logits or decays, or the
// model's own fp16 rows) on the way into LDS.  Long calls: wkv7_feed_kernel; single tokens, short calls, very many heads and the
// model's fused pass: wkv7_seq_kernel.  Every variant and every split of T over several calls gives bitwise the same result.
// (A model's calls of more than a few tokens go in chunks of 16 instead: wkv7_chunk.hip.)
#include <type_traits>
#include "ops.h"

namespace rwkv {

constexpr float kWScaleLog2e = -0.8750387749145276f;  // -e^-1/2 * log2(e), rwkv7_wkv_fp32_v2.cu:13
constexpr float kNLog2e = -1.4426950408889634f;       // rwkv7_wkv_fp32_v2.cu:14

__device__ __forceinline__ float decay_from_logit(float w) {
  return exp2f(kWScaleLog2e / (1.0f + exp2f(kNLog2e * w)));
}

// Operands of the stand-alone recurrence, all [B,T,C]: w as raw decay logits or decays (w_mode).
template <typename IO, typename WT>
struct SeqOperands {
  const IO *r, *k, *v, *a, *b;
  const WT* w;
  int w_mode;
};

// ---- sequence kernel -------------------------------------------------------------------------
// grid = B*H*PARTS, block = 1024/RPL/PARTS threads: 16/RPL wavefronts per head, RPL state rows per lane.  Lane (g, c) = (lane / 16,
// lane % 16) of wavefront q owns rows 4*RPL*q + RPL*g .. +RPL-1 and columns 4c .. 4c+3, so the 16 lanes of one DPP row hold
// complete state rows and the wavefronts never exchange data.  The block stages the operands kSeqChunk tokens at a time,
// double-buffered; a step costs each lane six LDS reads (its four columns of the five operands and its v values) against
// 28*RPL VALU operations.  y goes back through LDS so that the global stores are coalesced.
constexpr int kSeqChunk = 8;

// FUSED (the model's row-tiled time-mix path, fp16 io): the operands are not read as fp32 tensors but derived
// while staging from the fp16 rows r, k, a12, w12 - the arithmetic of kk_a_gate_kernel, one wavefront per token,
// lane = channel - and y is not stored but taken through the per-head GroupNorm, the (r.k.r_k) v bonus and the
// gate - the arithmetic of lnx_rkvres_xg_kernel on the fp16-rounded y - so that three launches and the fp32
// operand tensors between them become one launch.  Bitwise the same results as the three kernels.
//
// PARTS > 1: the rows of a head's state are independent of each other (row i needs only its own sum over the columns, v_i and
// the per-column operands), so with few heads a head is cut into PARTS row ranges that run on separate CUs.  Not with FUSED: the
// GroupNorm needs whole heads.
//
// STRAIGHT = false leaves out the unrolled eight-step body: single-token calls move a head's state once and are
// bound by that traffic, so they want the registers for more blocks per CU instead (148 -> under 100 VGPRs).
template <typename IO, typename WT, int RPL, int PARTS, bool FUSED, bool STRAIGHT = true>
__global__ __launch_bounds__(1024 / RPL / PARTS) void wkv7_seq_kernel(int T, int C, int H, float* __restrict__ state,
                                                              const IO* __restrict__ v, IO* __restrict__ y,
                                                              TmixSeqArgs fa, SeqOperands<IO, WT> ro) {
  constexpr bool RAW = !FUSED;
  static_assert(PARTS == 1 || !FUSED, "the fused pass needs whole heads");
  constexpr int NT = 1024 / RPL / PARTS;
  constexpr int kVSlots = (kSeqChunk * kHead + NT - 1) / NT;
  typedef float rows_t __attribute__((ext_vector_type(RPL)));
  __shared__ __align__(16) float ops[2][kSeqChunk][5][kHead];  // [buffer][token][a,b,d,k,r][column]
  __shared__ __align__(16) float vs[2][kSeqChunk][kHead];      // [buffer][token][row]
  __shared__ __align__(16) float ys[2][kSeqChunk][kHead];
  // Where to the 15 idle lanes of a row store in step_out.  The single-token variant keeps to 32 KB of LDS instead
  // (five blocks per CU) and stores under a branch.
  constexpr bool kSpare = STRAIGHT;
  __shared__ __align__(16) float spare[kSpare ? NT * RPL : 4];
  __shared__ __align__(16) float gs[FUSED ? 2 : 1][FUSED ? kSeqChunk : 1][kHead];  // FUSED: the gate rows

  const int bh = blockIdx.x / PARTS;
  const int bi = bh / H;
  const int h = bh - bi * H;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int row_lo = (blockIdx.x % PARTS) * (kHead / PARTS);         // this block's rows
  const int i0 = row_lo + 4 * RPL * (tid >> 6) + RPL * (lane >> 4);  // first of this lane's rows
  const int j0 = 4 * (lane & 15);                                    // first of its 4 columns
  float* sblk = state + (static_cast<int64_t>(bh) * kHead + i0) * kHead + j0;

  float4_t S[RPL];
#pragma unroll
  for (int i = 0; i < RPL; ++i) S[i] = __builtin_nontemporal_load(reinterpret_cast<const float4_t*>(sblk + i * kHead));

  const int64_t iob = static_cast<int64_t>(bi) * T * C + h * kHead;
  // Two sets of staging registers: a chunk is requested two chunks before it is needed - eight steps are shorter
  // than a trip to memory.
  float v_stage[2][kVSlots];
  // FUSED: raw fp16 values of this thread's (token, channel) slots: r, k, a12, w12, g; and its channel's constants
  half_t raw[2][kVSlots][5];
  // RAW: the caller's r, w, k, a, b values of the slots, still in the io type
  IO rio[2][RAW ? kVSlots : 1][4];
  WT wio[2][RAW ? kVSlots : 1];
  float c_kk = 0.0f, c_a0 = 0.0f, c_ka = 0.0f, c_w0 = 0.0f, c_rk = 0.0f, c_lnw = 0.0f, c_lnb = 0.0f;
  if constexpr (FUSED) {
    const int c = h * kHead + lane;
    c_kk = h2f(fa.k_k[c]); c_a0 = h2f(fa.a0[c]); c_ka = h2f(fa.k_a[c]); c_w0 = h2f(fa.w0[c]);
    c_rk = h2f(fa.r_k[c]); c_lnw = h2f(fa.lnx_w[c]); c_lnb = h2f(fa.lnx_b[c]);
  }

  // Every load is issued unconditionally (tokens past the end repeat the last one; their steps never run): a load
  // under a branch makes the compiler's s_waitcnt accounting wait for everything in flight, the younger set too.
  auto request = [&](int t0, auto set_c) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < kVSlots; ++i) {
      const int tok = min((tid + i * NT) >> 6, kSeqChunk - 1);
      const int64_t at = iob + static_cast<int64_t>(min(t0 + tok, T - 1)) * C + lane;
      v_stage[set][i] = static_cast<float>(v[at]);
      if constexpr (FUSED) {
        raw[set][i][0] = fa.r[at]; raw[set][i][1] = fa.k[at]; raw[set][i][2] = fa.a12[at]; raw[set][i][3] = fa.w12[at];
        raw[set][i][4] = fa.g[at];
      }
      if constexpr (RAW) {
        rio[set][i][0] = ro.a[at]; rio[set][i][1] = ro.b[at]; rio[set][i][2] = ro.k[at]; rio[set][i][3] = ro.r[at];
        wio[set][i] = ro.w[at];
      }
    }
  };
  auto commit = [&](int buf, auto set_c) {
    constexpr int set = decltype(set_c)::value;
#pragma unroll
    for (int i = 0; i < kVSlots; ++i) {
      const int tok = (tid + i * NT) >> 6;  // wave-uniform: one wavefront per token, lane = channel
      if (tok < kSeqChunk) {
        vs[buf][tok][lane] = v_stage[set][i];
        if constexpr (FUSED) {
          // kk normalise, a-gate, new k, decay: the statements of kk_a_gate_kernel
          const float kv = h2f(raw[set][i][1]);
          const float u = kv * c_kk;
          const float total = wave_sum(u * u);
          const float inv = 1.0f / fmaxf(sqrtf(total), kKkEps);
          const float kk = u * inv;
          const float av = sigmoid_f(c_a0 + h2f(raw[set][i][2]));
          const half_t nk = f2h(kv * fmaf(av, c_ka, 1.0f - c_ka));
          const half_t nkk = f2h(-kk);
          const half_t kka = f2h(kk * av);
          const float wraw = round_h(h2f(raw[set][i][3]) + c_w0);
          ops[buf][tok][0][lane] = h2f(nkk);
          ops[buf][tok][1][lane] = h2f(kka);
          ops[buf][tok][2][lane] = exp2f(-0.8750387749145276f / (1.0f + exp2f(-1.4426950408889634f * wraw)));
          ops[buf][tok][3][lane] = h2f(nk);
          ops[buf][tok][4][lane] = h2f(raw[set][i][0]);
          gs[buf][tok][lane] = h2f(raw[set][i][4]);
        }
        if constexpr (RAW) {
          const float wv = static_cast<float>(wio[set][i]);
          ops[buf][tok][0][lane] = static_cast<float>(rio[set][i][0]);
          ops[buf][tok][1][lane] = static_cast<float>(rio[set][i][1]);
          ops[buf][tok][2][lane] = (ro.w_mode == RWKV_W_RAW_LOGIT) ? decay_from_logit(wv) : wv;
          ops[buf][tok][3][lane] = static_cast<float>(rio[set][i][2]);
          ops[buf][tok][4][lane] = static_cast<float>(rio[set][i][3]);
        }
      }
    }
  };

  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  request(0, Set0{});
  if (T > kSeqChunk) request(kSeqChunk, Set1{});
  commit(0, Set0{});
  __syncthreads();
  // The y rows of a finished chunk (tokens t0 .. t0+n-1, LDS buffer buf) go to memory: one wavefront per token,
  // lane = channel.  It runs in the middle of the next chunk, where its LDS and memory latencies hide behind the
  // steps; ys[buf] is next written a barrier later.  FUSED also reads the chunk's operand, v and gate rows: each
  // thread reads exactly the (token, channel) slots that it overwrites itself in the commit that follows.
  auto write_out = [&](int t0, int n, int buf) {
#pragma unroll
    for (int i = 0; i < kVSlots; ++i) {
      const int tt = (tid + i * NT) >> 6;
      if (tt < n) {
        if constexpr (FUSED) {
          // GroupNorm over the head, (r.k.r_k) v bonus, gate: the statements of lnx_rkvres_xg_kernel on the
          // fp16-rounded y
          const float yv = round_h(ys[buf][tt][lane]);
          const float mean = wave_sum(yv) * (1.0f / 64.0f);
          const float dd = yv - mean;
          const float var = wave_sum(dd * dd) * (1.0f / 64.0f);
          const float rstd = rsqrtf(var + kLnxEps);
          const float rkv = wave_sum(ops[buf][tt][4][lane] * ops[buf][tt][3][lane] * c_rk);
          const float o = (dd * rstd * c_lnw + c_lnb + rkv * vs[buf][tt][lane]) * gs[buf][tt][lane];
          y[iob + static_cast<int64_t>(t0 + tt) * C + lane] = static_cast<IO>(o);
        } else if (PARTS == 1 || (lane >= row_lo && lane < row_lo + kHead / PARTS)) {
          y[iob + static_cast<int64_t>(t0 + tt) * C + lane] = static_cast<IO>(ys[buf][tt][lane]);
        }
      }
    }
  };
  // chunk c: LDS buffer c&1, staging set c&1 - both static inside the two-chunk body
  auto run_chunk = [&](int t0, auto set_c) {
    constexpr int buf = decltype(set_c)::value;
    using Other = std::integral_constant<int, 1 - buf>;
    const bool more = t0 + kSeqChunk < T;
    request(t0 + 2 * kSeqChunk, set_c);  // this chunk's set was committed a chunk ago
    const int n = min(kSeqChunk, T - t0);
    struct StepOps {
      float4_t av, bv, dv, kv, rv;
      rows_t vv;
    };
    auto load_step = [&](int tt, StepOps& q) {
      q.av = *reinterpret_cast<const float4_t*>(&ops[buf][tt][0][j0]);
      q.bv = *reinterpret_cast<const float4_t*>(&ops[buf][tt][1][j0]);
      q.dv = *reinterpret_cast<const float4_t*>(&ops[buf][tt][2][j0]);
      q.kv = *reinterpret_cast<const float4_t*>(&ops[buf][tt][3][j0]);
      q.rv = *reinterpret_cast<const float4_t*>(&ops[buf][tt][4][j0]);
      q.vv = *reinterpret_cast<const rows_t*>(&vs[buf][tt][i0]);
    };
    // A step in two halves.  step_state carries the recurrence: row sums of S a, then the update - the only chain
    // from one token to the next.  step_out reads the new state: y = S r.
    auto step_state = [&](const StepOps& q) {
      const float4_t av = q.av, bv = q.bv, dv = q.dv, kv = q.kv;
      float sa[RPL];
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        float p = S[i].x * av.x;
        p = fmaf(S[i].y, av.y, p);
        p = fmaf(S[i].z, av.z, p);
        p = fmaf(S[i].w, av.w, p);
        sa[i] = p;
      }
#pragma unroll
      for (int i = 0; i < RPL; ++i) sa[i] = row16_sum(sa[i]);
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        const float vi = q.vv[i];
        S[i].x = fmaf(S[i].x, dv.x, fmaf(sa[i], bv.x, kv.x * vi));
        S[i].y = fmaf(S[i].y, dv.y, fmaf(sa[i], bv.y, kv.y * vi));
        S[i].z = fmaf(S[i].z, dv.z, fmaf(sa[i], bv.z, kv.z * vi));
        S[i].w = fmaf(S[i].w, dv.w, fmaf(sa[i], bv.w, kv.w * vi));
      }
    };
    auto step_out = [&](int tt, const StepOps& q) {
      const float4_t rv = q.rv;
      rows_t yy;
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        float p = S[i].x * rv.x;
        p = fmaf(S[i].y, rv.y, p);
        p = fmaf(S[i].z, rv.z, p);
        p = fmaf(S[i].w, rv.w, p);
        yy[i] = p;
      }
#pragma unroll
      for (int i = 0; i < RPL; ++i) yy[i] = row16_sum(yy[i]);
      // the 16 lanes of a row hold the same sums: the first stores them, the others store to a spare area - a
      // store under a branch would end the scheduling region here
      if constexpr (kSpare) {
        float* dst = (lane & 15) == 0 ? &ys[buf][tt][i0] : &spare[tid * RPL];
        *reinterpret_cast<rows_t*>(dst) = yy;
      } else {
        if ((lane & 15) == 0) *reinterpret_cast<rows_t*>(&ys[buf][tt][i0]) = yy;
      }
    };
    if (STRAIGHT && n == kSeqChunk) {
      // Full chunk, straight-line.  The operands of step tt+1 are read from LDS while step tt computes, and the
      // scheduling regions run from the middle of one step to the middle of the next
      // (__builtin_amdgcn_sched_barrier(0) between the halves), so that the compiler fills the latency bubbles
      // of step tt's output sums with the independent recurrence half of step tt+1.
      StepOps q[2];
      load_step(0, q[0]);
#pragma unroll
      for (int tt = 0; tt < kSeqChunk; ++tt) {
        if (tt + 1 < kSeqChunk) load_step(tt + 1, q[(tt + 1) & 1]);
        step_state(q[tt & 1]);
        __builtin_amdgcn_sched_barrier(0);
        step_out(tt, q[tt & 1]);
        if (tt == kSeqChunk / 2 - 1) {
          if (t0 > 0) write_out(t0 - kSeqChunk, kSeqChunk, buf ^ 1);
          if (more) commit(buf ^ 1, Other{});
        }
      }
    } else {
      // the last, partial chunk (and single-token calls): same step arithmetic, rolled loop
#pragma unroll 1
      for (int tt = 0; tt < n; ++tt) {
        StepOps q;
        load_step(tt, q);
        step_state(q);
        step_out(tt, q);
      }
      if (t0 > 0) write_out(t0 - kSeqChunk, kSeqChunk, buf ^ 1);
      if (more) commit(buf ^ 1, Other{});  // (only without the straight-line body: a partial chunk is the last)
    }
    __syncthreads();
  };
  for (int t0 = 0; t0 < T; t0 += 2 * kSeqChunk) {
    run_chunk(t0, Set0{});
    if (t0 + kSeqChunk < T) run_chunk(t0 + kSeqChunk, Set1{});
  }
  const int t_last = (T - 1) / kSeqChunk * kSeqChunk;
  write_out(t_last, T - t_last, (t_last / kSeqChunk) & 1);

#pragma unroll
  for (int i = 0; i < RPL; ++i) __builtin_nontemporal_store(S[i], reinterpret_cast<float4_t*>(sblk + i * kHead));
}


// ---- sequence kernel with feeders ---------------------------------------------------------------------------
// NC wavefronts own the state and do nothing but steps; NF feeders bring the operands of the next chunk of kSeqChunk tokens
// into LDS (requested SETS chunks ahead, the decay derived where the caller has logits) and take the finished y rows out.  All
// meet once per chunk, ahead of the chunk's last step, whose operands are in registers by then.  A block owns 1 / PARTS of a
// head's rows - they are independent of each other: row i needs its own sum over the columns, v_i and the per-column operands -
// a lane RPL rows x G groups of four columns.
//
// What bounds it.  Few heads (a wavefront per SIMD): a wavefront issues an instruction every 5 to 6 clocks at best and every 8.5
// where it needs the one before (16 through DPP), so the step is its instruction count, 36, times six: 0.11 us measured.  The
// staging used to stand in the same instruction stream, and five fp32 vectors per token and wavefront took the CU's LDS 170 of
// a step's 350 clocks; fp16 operands now stay fp16 in LDS (the mixed-precision multiply-add takes them as they are): 104.  Many
// heads: VALU issue, four clocks per instruction and SIMD; eight columns per lane put one of a row's four adds over lanes into the
// lane (24 instead of 28 operations per four elements).  us per call, before / now:
//   1 x 64 tokens x 12 heads, fp32 tensors 12.8 / 9.8   1 x 512 x 64, fp16 84 / 56   3 x 333 x 32 72 / 55
//   4 x 256 x 64 83.7 / 70   8 x 256 x 64 125 / 113   16 x 256 x 64 221 / 210; fp32 tensors 82 / 71, 124 / 108, 238 / 219
// The fp32 tile for more than 128 heads keeps six wavefronts per SIMD at the price of ten spilled registers: 128 tokens of 1024
// heads 108 us; five 121, four 135 (512 heads 58.3, 56.9 and 57.2).
template <typename E, int N>
struct Loose {  // N elements that are aligned like one
  typedef E type __attribute__((ext_vector_type(N), aligned(sizeof(E))));
};

// A chunk's operands in LDS.  The 16 groups of four columns of a token lie in the order in which the lanes of a row read
// them: lane e takes groups G e .. G e + G - 1, its m-th at place m * 16 / G + e, so that the lanes' pieces are neighbours.
template <typename OT>
struct SeqStage;
template <>
struct SeqStage<half_t> {  // a and b (k and r) of a group share a 16-byte piece
  half_t ab[kSeqChunk][16][8];
  half_t kr[kSeqChunk][16][8];
  float d[kSeqChunk][16][4];
  half_t v[kSeqChunk][kHead];
  __device__ __forceinline__ half_t* a_at(int t, int p) { return &ab[t][p][0]; }
  __device__ __forceinline__ half_t* b_at(int t, int p) { return &ab[t][p][4]; }
  __device__ __forceinline__ half_t* k_at(int t, int p) { return &kr[t][p][0]; }
  __device__ __forceinline__ half_t* r_at(int t, int p) { return &kr[t][p][4]; }
};
template <>
struct SeqStage<float> {
  float a[kSeqChunk][16][4], b[kSeqChunk][16][4], k[kSeqChunk][16][4], r[kSeqChunk][16][4];
  float d[kSeqChunk][16][4];
  float v[kSeqChunk][kHead];
  __device__ __forceinline__ float* a_at(int t, int p) { return &a[t][p][0]; }
  __device__ __forceinline__ float* b_at(int t, int p) { return &b[t][p][0]; }
  __device__ __forceinline__ float* k_at(int t, int p) { return &k[t][p][0]; }
  __device__ __forceinline__ float* r_at(int t, int p) { return &r[t][p][0]; }
};

// The operands of one step in a lane's registers.
template <typename OT, int G, int RPL>
struct SeqStep {
  typedef OT vec4 __attribute__((ext_vector_type(4)));
  typedef OT vec8 __attribute__((ext_vector_type(8)));
  typedef OT rows_t __attribute__((ext_vector_type(RPL)));
  vec4 a[G], b[G], k[G], r[G];
  float4_t d[G];
  rows_t v;
  __device__ __forceinline__ void load(SeqStage<OT>& st, int t, int e, int row) {
#pragma unroll
    for (int m = 0; m < G; ++m) {
      const int p = m * (16 / G) + e;
      if constexpr (sizeof(OT) == 2) {
        const vec8 ab = *reinterpret_cast<const vec8*>(st.a_at(t, p));
        const vec8 kr = *reinterpret_cast<const vec8*>(st.k_at(t, p));
        a[m] = __builtin_shufflevector(ab, ab, 0, 1, 2, 3);
        b[m] = __builtin_shufflevector(ab, ab, 4, 5, 6, 7);
        k[m] = __builtin_shufflevector(kr, kr, 0, 1, 2, 3);
        r[m] = __builtin_shufflevector(kr, kr, 4, 5, 6, 7);
      } else {
        a[m] = *reinterpret_cast<const vec4*>(st.a_at(t, p));
        b[m] = *reinterpret_cast<const vec4*>(st.b_at(t, p));
        k[m] = *reinterpret_cast<const vec4*>(st.k_at(t, p));
        r[m] = *reinterpret_cast<const vec4*>(st.r_at(t, p));
      }
      d[m] = *reinterpret_cast<const float4_t*>(&st.d[t][p][0]);
    }
    v = *reinterpret_cast<const rows_t*>(&st.v[t][row]);
  }
};

__device__ __forceinline__ void seq_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// x * y where either may be fp16.  minus_zero holds -0.0 in a register the compiler cannot see through: the mixed-precision
// multiply-add then takes fp16 operands as they are (x * y + -0.0 is x * y to the bit), where a product would convert first.
template <typename X, typename Y>
__device__ __forceinline__ float seq_product(X x, Y y, float minus_zero) {
  if constexpr (sizeof(X) == 2 || sizeof(Y) == 2) return fmaf(static_cast<float>(x), static_cast<float>(y), minus_zero);
  else return x * y;
}

template <typename IO, typename WT, int G, int RPL, int NC, int PARTS, int NF, int SETS, int WAVES, bool AHEAD>
__global__ __launch_bounds__(64 * (NC + NF), WAVES) void wkv7_feed_kernel(int T, int C, int H, float* __restrict__ state, SeqOperands<IO, WT> op,
                                                                         IO* __restrict__ y) {
  constexpr int kRows = kHead / PARTS;        // rows of the state per block
  constexpr int LPR = 16 / G;                 // lanes per row
  static_assert(NC * RPL * (64 / LPR) == kRows, "the compute wavefronts own the block's rows");
  __shared__ __align__(16) SeqStage<IO> stage[2];
  // y of a chunk: one buffer written, one read by the feeders, and the one between, whose last token is still being written
  __shared__ __align__(16) float ys[3][kSeqChunk][kRows];
  __shared__ __align__(16) float spare[kSeqChunk * kRows + 64 * RPL];  // where the idle lanes of a row store
  const int bh = blockIdx.x / PARTS;
  const int row_lo = (blockIdx.x % PARTS) * kRows;
  const int bi = bh / H;
  const int h = bh - bi * H;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int64_t base = static_cast<int64_t>(bi) * T * C + h * kHead;
  const int chunks = (T + kSeqChunk - 1) / kSeqChunk;

  if (wave >= NC) {
    // feeder f: tokens f * TPF .. of a chunk, CPF columns of one of them per lane
    constexpr int TPF = kSeqChunk / NF, LPT = 64 / TPF, CPF = kHead / LPT;
    using vec = typename Loose<IO, CPF>::type;
    using wvec = typename Loose<WT, CPF>::type;
    struct Set {
      vec a, b, k, r, v;
      wvec w;
    };
    Set set[SETS];
    const int f = wave - NC;
    const int tok = f * TPF + lane / LPT;
    const int col = (lane % LPT) * CPF;
    // (every load unconditional: tokens past the end repeat the last one, their steps never run)
    auto request = [&](Set& s, int c) {
      const int64_t at = base + static_cast<int64_t>(min(c * kSeqChunk + tok, T - 1)) * C + col;
      s.a = *reinterpret_cast<const vec*>(op.a + at);
      s.b = *reinterpret_cast<const vec*>(op.b + at);
      s.w = *reinterpret_cast<const wvec*>(op.w + at);
      s.k = *reinterpret_cast<const vec*>(op.k + at);
      s.r = *reinterpret_cast<const vec*>(op.r + at);
      s.v = *reinterpret_cast<const vec*>(op.v + at);
    };
    auto commit = [&](const Set& s, SeqStage<IO>& st) {
      constexpr int PW = CPF < 4 ? CPF : 4;  // columns of a piece
      typedef IO piece __attribute__((ext_vector_type(PW)));
      typedef float fpiece __attribute__((ext_vector_type(PW)));
#pragma unroll
      for (int g = 0; g < CPF / PW; ++g) {
        const int c = (col + g * PW) >> 2;
        const int p = (c % G) * LPR + c / G;
        const int in = (col + g * PW) & 3;
        piece a, b, k, r;
        fpiece d;
#pragma unroll
        for (int i = 0; i < PW; ++i) {
          a[i] = s.a[g * PW + i];
          b[i] = s.b[g * PW + i];
          k[i] = s.k[g * PW + i];
          r[i] = s.r[g * PW + i];
          d[i] = static_cast<float>(s.w[g * PW + i]);
        }
        if (op.w_mode == RWKV_W_RAW_LOGIT) {
#pragma unroll
          for (int i = 0; i < PW; ++i) d[i] = decay_from_logit(d[i]);
        }
        *reinterpret_cast<piece*>(st.a_at(tok, p) + in) = a;
        *reinterpret_cast<piece*>(st.b_at(tok, p) + in) = b;
        *reinterpret_cast<piece*>(st.k_at(tok, p) + in) = k;
        *reinterpret_cast<piece*>(st.r_at(tok, p) + in) = r;
        *reinterpret_cast<fpiece*>(&st.d[tok][p][in]) = d;
      }
      typedef IO store_v __attribute__((ext_vector_type(CPF)));
      *reinterpret_cast<store_v*>(&st.v[tok][col]) = s.v;
    };
    // the finished y rows of a chunk: EW neighbouring rows per lane
    auto write_out = [&](int c, int slot) {
      constexpr int EW = PARTS == 1 ? CPF : 2;
      constexpr int kPieces = kSeqChunk * kRows / EW;
      typedef float fvec __attribute__((ext_vector_type(EW)));
      using ovec = typename Loose<IO, EW>::type;
      const int n = min(kSeqChunk, T - c * kSeqChunk);
#pragma unroll
      for (int i = 0; i < (kPieces + 64 * NF - 1) / (64 * NF); ++i) {
        const int idx = f * 64 + lane + i * 64 * NF;
        const int t = idx / (kRows / EW);
        const int r = idx % (kRows / EW) * EW;
        if (t < n) {
          const fvec yv = *reinterpret_cast<const fvec*>(&ys[slot][t][r]);
          ovec o;
#pragma unroll
          for (int e = 0; e < EW; ++e) o[e] = static_cast<IO>(yv[e]);
          *reinterpret_cast<ovec*>(y + base + static_cast<int64_t>(c * kSeqChunk + t) * C + row_lo + r) = o;
        }
      }
    };
#pragma unroll
    for (int i = 0; i < SETS; ++i) request(set[i], i);
    commit(set[0], stage[0]);
    request(set[0], SETS);
    commit(set[1 % SETS], stage[1]);
    request(set[1 % SETS], SETS + 1);
    seq_barrier();  // chunks 0 and 1 are staged
    int slot = 2;   // of chunk c - 1
    // chunk c has been read (its last step runs from registers): chunk c + 2 takes its place
    auto turn = [&](int u, int c) {
      seq_barrier();
      commit(set[(u + 2) % SETS], stage[u & 1]);
      request(set[(u + 2) % SETS], c + 2 + SETS);
      if (c > 0) write_out(c - 1, slot);
      slot = slot == 2 ? 0 : slot + 1;
    };
    const int whole = chunks - chunks % SETS;
    int c0 = 0;
    for (; c0 < whole; c0 += SETS) {
#pragma unroll
      for (int u = 0; u < SETS; ++u) turn(u, c0 + u);
    }
#pragma unroll
    for (int u = 0; u < SETS - 1; ++u) {
      if (c0 + u >= chunks) break;
      turn(u, c0 + u);
    }
    seq_barrier();  // all steps are done
    write_out(chunks - 1, slot);
    return;
  }

  const int e = lane % LPR;
  const int row = RPL * ((64 / LPR) * wave + lane / LPR);  // first of this lane's rows in the block
  float* sblk = state + (static_cast<int64_t>(bh) * kHead + row_lo + row) * kHead + 4 * G * e;
  float4_t S[RPL][G];
#pragma unroll
  for (int i = 0; i < RPL; ++i)
#pragma unroll
    for (int m = 0; m < G; ++m) S[i][m] = __builtin_nontemporal_load(reinterpret_cast<const float4_t*>(sblk + i * kHead + 4 * m));

  float minus_zero = -0.0f;
  asm volatile("" : "+s"(minus_zero));
  using Step = SeqStep<IO, G, RPL>;
  typedef typename Step::vec4 vec4;
  typedef float frows __attribute__((ext_vector_type(RPL)));
  // One step of the recurrence together with the output sums of the step before it, which read the same state:
  //   y' = S r' of the step before, sa = S a, S = S d + sa b + k v
  // The sum over a row's 64 columns: four columns in a chain, then groups 2n and 2n + 1, and so on up - in the lane as far as
  // it holds them, over the lanes of the row from there - the same tree whatever G.
  // A wavefront that is alone on its SIMD waits 8 clocks for the result of the instruction before (12 where a DPP move reads
  // it), so the order is laid down here: the two chains of products alternate, the products k v stand between the DPP adds,
  // and no instruction needs one of the two before it.
  auto step = [&](const Step& q, const vec4 (&r_before)[G], float* dst) {
    float sa[RPL], out[RPL], p[RPL][G], o[RPL][G], kv[RPL][G][4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
#pragma unroll
      for (int i = 0; i < RPL; ++i)
#pragma unroll
        for (int m = 0; m < G; ++m) {
          p[i][m] = x == 0 ? seq_product(S[i][m][0], q.a[m][0], minus_zero) : fmaf(S[i][m][x], static_cast<float>(q.a[m][x]), p[i][m]);
          o[i][m] = x == 0 ? seq_product(S[i][m][0], r_before[m][0], minus_zero)
                           : fmaf(S[i][m][x], static_cast<float>(r_before[m][x]), o[i][m]);
        }
      __builtin_amdgcn_sched_barrier(0);
    }
    auto in_lane = [](const float (&t)[G]) {
      if constexpr (G == 1) return t[0];
      else if constexpr (G == 2) return t[0] + t[1];
      else return (t[0] + t[1]) + (t[2] + t[3]);
    };
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      sa[i] = in_lane(p[i]);
      out[i] = in_lane(o[i]);
    }
    constexpr int kLevels = G == 1 ? 4 : (G == 2 ? 3 : 2);
    constexpr int kProducts = RPL * G * 4;
    auto products = [&](int from, int to) {
#pragma unroll
      for (int j = from; j < to; ++j) {
        const int x = j % 4, m = j / 4 % G, i = j / (4 * G);
        kv[i][m][x] = seq_product(q.k[m][x], q.v[i], minus_zero);
        asm volatile("" : "+v"(kv[i][m][x]));  // here, not at its use
      }
    };
#pragma unroll
    for (int l = 0; l < kLevels; ++l) {
      products(l * kProducts / kLevels, (l + 1) * kProducts / kLevels);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < RPL; ++i) {
        auto add = [&](float v) {
          if (l == 0) return dpp_add<0xB1>(v);   // quad_perm [1,0,3,2]
          if (l == 1) return dpp_add<0x4E>(v);   // quad_perm [2,3,0,1]
          if (l == 2) return dpp_add<0x141>(v);  // row_half_mirror
          return dpp_add<0x140>(v);              // row_mirror
        };
        sa[i] = add(sa[i]);
        out[i] = add(out[i]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int i = 0; i < RPL; ++i)
#pragma unroll
      for (int m = 0; m < G; ++m)
#pragma unroll
        for (int x = 0; x < 4; ++x) kv[i][m][x] = fmaf(sa[i], static_cast<float>(q.b[m][x]), kv[i][m][x]);
    frows yy;
#pragma unroll
    for (int i = 0; i < RPL; ++i) yy[i] = out[i];
    *reinterpret_cast<frows*>(dst) = yy;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RPL; ++i)
#pragma unroll
      for (int m = 0; m < G; ++m)
#pragma unroll
        for (int x = 0; x < 4; ++x) S[i][m][x] = fmaf(S[i][m][x], q.d[m][x], kv[i][m][x]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto row_sums = [&](const vec4 (&x)[G], float (&sum)[RPL]) {
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      float p[G];
#pragma unroll
      for (int m = 0; m < G; ++m) {
        p[m] = seq_product(S[i][m].x, x[m][0], minus_zero);
        p[m] = fmaf(S[i][m].y, static_cast<float>(x[m][1]), p[m]);
        p[m] = fmaf(S[i][m].z, static_cast<float>(x[m][2]), p[m]);
        p[m] = fmaf(S[i][m].w, static_cast<float>(x[m][3]), p[m]);
      }
      if constexpr (G == 1) sum[i] = p[0];
      else if constexpr (G == 2) sum[i] = p[0] + p[1];
      else sum[i] = (p[0] + p[1]) + (p[2] + p[3]);
    }
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      sum[i] = dpp_add<0xB1>(sum[i]);
      sum[i] = dpp_add<0x4E>(sum[i]);
      if constexpr (LPR >= 8) sum[i] = dpp_add<0x141>(sum[i]);
      if constexpr (LPR >= 16) sum[i] = dpp_add<0x140>(sum[i]);
    }
  };
  // All lanes of a row hold its sums: the first stores them, the others store to a spare area (a store under a branch would
  // end the scheduling region).
  float* idle = &spare[lane * RPL];
  int slot = 0;
  seq_barrier();  // chunks 0 and 1 are staged
  if constexpr (AHEAD) {
    float* y_before = idle;  // where the sums of the step before go
    vec4 r_before[G];
#pragma unroll
    for (int m = 0; m < G; ++m) r_before[m] = vec4{};
    Step cur;
    cur.load(stage[0], 0, e, row_lo + row);
    for (int c = 0; c < chunks; ++c) {
      SeqStage<IO>& st = stage[c & 1];
      SeqStage<IO>& after = stage[(c & 1) ^ 1];
      float* dst = e == 0 ? &ys[slot][0][row] : idle;
      slot = slot == 2 ? 0 : slot + 1;
      const int n = T - c * kSeqChunk;
      if (n >= kSeqChunk) {
        // the operands of step t + 1 are read from LDS while step t computes
#pragma unroll
        for (int t = 0; t < kSeqChunk; ++t) {
          Step next;
          if (t + 1 < kSeqChunk) {
            next.load(st, t + 1, e, row_lo + row);
          } else {
            seq_barrier();
            next.load(after, 0, e, row_lo + row);
          }
          __builtin_amdgcn_sched_barrier(0);
          step(cur, r_before, t == 0 ? y_before : dst + (t - 1) * kRows);
#pragma unroll
          for (int m = 0; m < G; ++m) r_before[m] = cur.r[m];
          cur = next;
        }
        y_before = dst + (kSeqChunk - 1) * kRows;
      } else {  // the last, partial chunk
#pragma unroll 1
        for (int t = 0; t < n; ++t) {
          cur.load(st, t, e, row_lo + row);
          step(cur, r_before, y_before);
#pragma unroll
          for (int m = 0; m < G; ++m) r_before[m] = cur.r[m];
          y_before = dst + t * kRows;
        }
        seq_barrier();
      }
    }
    float out[RPL];  // the output sums of the last step
    row_sums(r_before, out);
    frows yy;
#pragma unroll
    for (int i = 0; i < RPL; ++i) yy[i] = out[i];
    *reinterpret_cast<frows*>(y_before) = yy;
  } else {
    // many wavefronts per SIMD: they hide each other's latencies, and registers are what limits their number
    for (int c = 0; c < chunks; ++c) {
      SeqStage<IO>& st = stage[c & 1];
      float* dst = e == 0 ? &ys[slot][0][row] : idle;
      slot = slot == 2 ? 0 : slot + 1;
      auto token = [&](int t) {
        Step q;
        q.load(st, t, e, row_lo + row);
        float sa[RPL], out[RPL];
        row_sums(q.a, sa);
#pragma unroll
        for (int i = 0; i < RPL; ++i)
#pragma unroll
          for (int m = 0; m < G; ++m)
#pragma unroll
            for (int x = 0; x < 4; ++x)
              S[i][m][x] = fmaf(S[i][m][x], q.d[m][x], fmaf(sa[i], static_cast<float>(q.b[m][x]), seq_product(q.k[m][x], q.v[i], minus_zero)));
        row_sums(q.r, out);
        frows yy;
#pragma unroll
        for (int i = 0; i < RPL; ++i) yy[i] = out[i];
        *reinterpret_cast<frows*>(dst + t * kRows) = yy;
      };
      const int n = T - c * kSeqChunk;
      if (n >= kSeqChunk) {
#pragma unroll
        for (int t = 0; t < kSeqChunk; ++t) token(t);
      } else {
#pragma unroll 1
        for (int t = 0; t < n; ++t) token(t);
      }
      seq_barrier();
    }
  }
  seq_barrier();  // all steps are done
#pragma unroll
  for (int i = 0; i < RPL; ++i)
#pragma unroll
    for (int m = 0; m < G; ++m) __builtin_nontemporal_store(S[i][m], reinterpret_cast<float4_t*>(sblk + i * kHead + 4 * m));
}

template <typename IO, typename WT, int RPL, int PARTS, bool FUSED, bool STRAIGHT>
static void launch_seq(hipStream_t st, int B, int T, int C, int H, float* state, const IO* v, IO* y, const TmixSeqArgs& fa,
                       const SeqOperands<IO, WT>& ro) {
  hipLaunchKernelGGL((wkv7_seq_kernel<IO, WT, RPL, PARTS, FUSED, STRAIGHT>), dim3(B * H * PARTS), dim3(1024 / RPL / PARTS), 0, st, T, C, H,
                     state, v, y, fa, ro);
}

template <typename IO, typename WT, int G, int RPL, int NC, int PARTS, int NF, int SETS, int WAVES, bool AHEAD>
static void launch_feed(hipStream_t st, int B, int T, int C, int H, float* state, const SeqOperands<IO, WT>& op, IO* y) {
  hipLaunchKernelGGL((wkv7_feed_kernel<IO, WT, G, RPL, NC, PARTS, NF, SETS, WAVES, AHEAD>), dim3(B * H * PARTS), dim3(64 * (NC + NF)), 0, st, T, C, H,
                     state, op, y);
}

// Which tile a call with feeders takes.  Up to 128 heads the chip has CUs to spare: a head is cut into row ranges of
// four wavefronts each, one state row per lane, and every wavefront is alone on its SIMD.  Up to 512 heads (two per CU) whole
// heads, 2 x 8 elements per lane, the next step's operands read ahead; with more heads, or fp32 operands (twice the
// registers), wavefronts are worth more than reading ahead (us per token of 16 x 64 heads, 6 per SIMD / 3 reading ahead: 0.83 /
// 1.05; of 4 x 64 heads 0.29 / 0.27, of 8 x 64 0.46 / 0.44).
constexpr int kSeqQuarterHeads = 64;
constexpr int kSeqHalfHeads = 128;
constexpr int kSeqAheadHeads = 512;

// false: few heads in flight and more than one token, so that the recurrence runs a head's row ranges on separate CUs, which
// the fused pass cannot: its GroupNorm needs whole heads
bool tmix_seq_whole_heads(int B, int T, int H) { return !(B * H <= kSeqHalfHeads && T > 1); }

// Whether a call of T tokens on `heads` = B*H heads takes the feeders.  They stage two chunks before the first step where the other
// kernel stages one, so short calls lose.  us per call, feeders / without: fp16 tensors, 12 heads 2 tokens 3.3 / 2.8, 8 tokens 3.6 /
// 3.35, 12 4.45 / 4.50; 128 heads 8 tokens 1.11 times, 16 0.99; 256 heads 8 1.12, 17 0.99; 1024 heads 3 tokens 9.9 / 7.5, 17 20.9 / 20.0,
// 32 32.4 / 32.7; fp32 tensors 256 heads 16 tokens 1.15 times, 40 1.00; 1024 heads 3 tokens 12.6 / 8.2, 32 34.6 / 34.6.  Many more than
// 1024 heads are more than one round of feeder blocks (four per CU), and the other kernel's rounds, three per CU with longer
// straight code, are the shorter ones: fp16 tensors, 256 tokens, 1088 heads 262 / 268, 1280 306 / 270, 2048 448 / 418, 4096 833 / 797; fp32
// tensors, whose staging weighs more, only for shorter calls: 1536 heads 64 tokens 91 / 86, 256 tokens 336 / 333, 2048 heads 424 / 446.
template <typename IO>
static bool feeders_pay(int heads, int T) {
  constexpr bool half = sizeof(IO) == 2;
  if (heads <= kSeqQuarterHeads) return T >= 12;
  if (heads <= kSeqHalfHeads) return T >= (half ? 16 : 20);
  if (heads <= 256) return T >= (half ? 17 : 40);
  if (heads <= 1152) return T >= (half ? 32 : 40);
  return !half && T >= 128;
}

template <typename IO, typename WT>
static int launch_recurrence(hipStream_t st, int B, int T, int C, int H, float* state, const SeqOperands<IO, WT>& op, IO* y) {
  // a model's call: above kSeqHalfHeads such go in chunks or in the fused pass, unless they are tapped and too short for chunks or off alignment
  constexpr bool kModel = !std::is_same_v<IO, WT>;
  const int heads = B * H;
  if (T == 1) {
    launch_seq<IO, WT, 4, 1, false, false>(st, B, T, C, H, state, op.v, y, TmixSeqArgs{}, op);
  } else if (!feeders_pay<IO>(heads, T) || (kModel && heads > kSeqHalfHeads)) {
    if (heads <= kSeqQuarterHeads) launch_seq<IO, WT, 1, 4, false, true>(st, B, T, C, H, state, op.v, y, TmixSeqArgs{}, op);
    else if (heads <= kSeqHalfHeads) launch_seq<IO, WT, 2, 2, false, true>(st, B, T, C, H, state, op.v, y, TmixSeqArgs{}, op);
    else launch_seq<IO, WT, 4, 1, false, true>(st, B, T, C, H, state, op.v, y, TmixSeqArgs{}, op);
  } else if (heads <= kSeqQuarterHeads) {
    launch_feed<IO, WT, 1, 1, 4, 4, 2, 2, 1, true>(st, B, T, C, H, state, op, y);
  } else if (heads <= kSeqHalfHeads) {
    launch_feed<IO, WT, 2, 1, 4, 2, 2, 4, 1, true>(st, B, T, C, H, state, op, y);
  } else if constexpr (!kModel) {
    constexpr bool kHalf = sizeof(IO) == 2;
    if (kHalf && heads <= kSeqAheadHeads) launch_feed<IO, WT, 2, 2, 4, 1, 2, 2, kHalf ? 4 : 6, kHalf>(st, B, T, C, H, state, op, y);
    else launch_feed<IO, WT, 2, 2, 4, 1, 2, 2, 6, false>(st, B, T, C, H, state, op, y);
  }
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int wkv7_seq_f16_launch(hipStream_t st, int B, int T, int C, int H, float* state, const half_t* r, const float* d,
                        const half_t* k, const half_t* a, const half_t* b, const half_t* v, half_t* y) {
  return launch_recurrence<half_t, float>(st, B, T, C, H, state, SeqOperands<half_t, float>{r, k, v, a, b, d, RWKV_W_DECAY}, y);
}

int tmix_seq_launch(hipStream_t st, int B, int T, int C, int H, float* state, const TmixSeqArgs& fa, const half_t* v,
                    half_t* y2) {
  RWKV_REQUIRE(fa.r && fa.k && fa.a12 && fa.w12 && fa.g && fa.k_k && fa.a0 && fa.k_a && fa.w0 && fa.r_k && fa.lnx_w && fa.lnx_b,
               "tmix_seq: NULL tensor");
  const SeqOperands<half_t, half_t> none = {};
  if (T == 1) launch_seq<half_t, half_t, 4, 1, true, false>(st, B, T, C, H, state, v, y2, fa, none);
  else launch_seq<half_t, half_t, 4, 1, true, true>(st, B, T, C, H, state, v, y2, fa, none);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

}  // namespace rwkv

using namespace rwkv;

extern "C" int rwkv_hip_wkv7(rwkv_stream_t s, int B, int T, int C, int H, int w_mode, int io, void* state,
                             const void* r, const void* w, const void* k, const void* v, const void* a,
                             const void* b, void* y) {
  RWKV_REQUIRE(B > 0 && T > 0 && H > 0, "wkv7: B, T, H must be positive (got %d, %d, %d)", B, T, H);
  RWKV_REQUIRE(C == H * kHead, "wkv7: C (%d) must equal H*64 (%d)", C, H * kHead);
  RWKV_REQUIRE(w_mode == RWKV_W_RAW_LOGIT || w_mode == RWKV_W_DECAY, "wkv7: bad w_mode %d", w_mode);
  RWKV_REQUIRE(state && r && w && k && v && a && b && y, "wkv7: NULL tensor");
  auto run = [&](auto type) {
    using IO = decltype(type);
    const SeqOperands<IO, IO> op = {static_cast<const IO*>(r), static_cast<const IO*>(k), static_cast<const IO*>(v),
                                    static_cast<const IO*>(a), static_cast<const IO*>(b), static_cast<const IO*>(w), w_mode};
    return launch_recurrence<IO, IO>(as_stream(s), B, T, C, H, static_cast<float*>(state), op, static_cast<IO*>(y));
  };
  if (io == RWKV_IO_F16) return run(half_t{});
  RWKV_REQUIRE(io == RWKV_IO_F32, "wkv7: bad io %d", io);
  return run(float{});
}
