// Fused element-wise / normalisation kernels of the RWKV-7 layer graph.
//
// Reference kernels restated here (same arithmetic and fp16 rounding points, re-tiled for wave64):
//   LayerNorm family ........ cuda/rwkv7_v3a_ops.cu:1272-1351 (LN, add+LN), :1800-1931 (add + last-token LN),
//                             :1933-1985 (add+LN+cmix lerp), :1987-2060 (add+LN+6 lerps)
//   token shift ............. cuda/rwkv7_fast_ops_fp16.cu:53-127 (mix6 + shift update), :393-419 (cmix mix)
//   kk / a-gate ............. cuda/rwkv7_fast_ops_fp16.cu:129-172
//   GroupNorm+rkv-res+gate .. cuda/rwkv7_fast_ops_fp16.cu:174-237
//   relu^2, add_vec, f16->f32 cuda/rwkv7_fast_ops_fp16.cu:421-485;  advance_i32 cuda/rwkv7_v3a_ops.cu:202-207
//
// The LN kernels keep the whole row in registers (one block per row, one 16-byte slice per thread: 256, 512 or
// 1024 threads by row length - decode steps have few rows, so the wavefronts of a row are the only parallelism the
// launch has: 512 threads instead of 256 with two slices each make a 4096-wide row 15-25 % faster), so a row is
// read from HBM once for the two-pass mean/variance and the normalise+lerp epilogue.
#include <algorithm>
#include <type_traits>

#include "head_ops.h"
#include "ops.h"

namespace rwkv {

constexpr int kMixSeqRows = 256;  // rows of the launch with a block per row; more: blocks of several rows
constexpr int kMixRows = 4;       // rows of a block at most
constexpr int kLnMaxThreads = 1024;  // one 8-element vector per thread -> C <= 8192



template <int MODE, int NT>
__global__ __launch_bounds__(NT) void ln_fused_kernel(LnArgs a) {
  constexpr int kLnThreads = NT;
  constexpr int kLnMaxVec = 1;
  __shared__ float red[NT / 64];
  const int row = blockIdx.x;
  const int C = a.C;
  int64_t src = static_cast<int64_t>(row) * C;
  if constexpr (MODE == kAddLastLn) src = (static_cast<int64_t>(row) * a.T + (a.T - 1)) * C;
  int64_t xsrc = src;
  if constexpr (MODE == kLnMix) {
    if (a.tokens) xsrc = a.tokens[row] * static_cast<int64_t>(C);
  }
  const int64_t dst = static_cast<int64_t>(row) * C;

  // every global load of the kernel is issued here, before the first reduction, so the block pays one
  // memory round trip instead of three
  float v[kLnMaxVec][8];
  half8_t wv[kLnMaxVec], bv[kLnMaxVec], pv[kLnMaxVec], mv[kLnMaxVec][6];
  constexpr bool kMix = (MODE == kAddLnMix || MODE == kLnMix);
  float sum = 0.0f;
#pragma unroll
  for (int i = 0; i < kLnMaxVec; ++i) {
    const int c = (i * kLnThreads + threadIdx.x) * 8;
    if (c < C) {
      // the parameter vectors first: the sum over split-K partials below waits for its loads, and loads return in
      // issue order, so anything requested after that loop would cost a second trip to memory
      wv[i] = *reinterpret_cast<const half8_t*>(a.w + c);
      bv[i] = *reinterpret_cast<const half8_t*>(a.b + c);
      if constexpr (kMix) {
        pv[i] = *reinterpret_cast<const half8_t*>(a.shift + dst + c);
        // (no branch per coefficient vector: the unused ones re-read the last one, which costs nothing, whereas a
        // load under a branch is followed by a wait for everything requested so far)
#pragma unroll
        for (int s = 0; s < 6; ++s) mv[i][s] = *reinterpret_cast<const half8_t*>(a.mu[s < a.n_mix ? s : a.n_mix - 1] + c);
      }
      const half8_t xv = *reinterpret_cast<const half8_t*>(a.x + xsrc + c);
      __builtin_amdgcn_sched_barrier(0);
      half8_t rv = {};
      if constexpr (MODE != kLn && MODE != kLnMix) {
        if (a.res_partial) {
          // (the scale vector before the partials, for the same reason; without one any valid vector is read)
          const half8_t sv8 = *reinterpret_cast<const half8_t*>((a.res_scale ? a.res_scale : a.w) + c);
          const float* pp = a.res_partial + src + c;
          float4_t s0 = *reinterpret_cast<const float4_t*>(pp);
          float4_t s1 = *reinterpret_cast<const float4_t*>(pp + 4);
          // The other partials seven (up to four splits: three) at a time, all requested before the first is added (in
          // split order, as always); past the last split the last one is read again and left out.  A plain loop over the
          // splits would wait for each partial before it asks for the next: one trip to memory per split.
          auto add_planes = [&](auto batch_c) {
            constexpr int kBatch = decltype(batch_c)::value;
            for (int base = 1; base < a.res_splits; base += kBatch) {
              float4_t q0[kBatch], q1[kBatch];
#pragma unroll
              for (int u = 0; u < kBatch; ++u) {
                const int sp = base + u < a.res_splits ? base + u : a.res_splits - 1;
                q0[u] = *reinterpret_cast<const float4_t*>(pp + sp * a.res_plane);
                q1[u] = *reinterpret_cast<const float4_t*>(pp + sp * a.res_plane + 4);
              }
              // (keeps the requests together: their only uses sit under the conditions below, and the compiler
              // would move each load down into its condition)
#pragma unroll
              for (int u = 0; u < kBatch; ++u) asm volatile("" : "+v"(q0[u]), "+v"(q1[u]));
#pragma unroll
              for (int u = 0; u < kBatch; ++u) {
                if (base + u < a.res_splits) {
                  s0 = s0 + q0[u];
                  s1 = s1 + q1[u];
                }
              }
            }
          };
          if (a.res_splits <= 4) add_planes(std::integral_constant<int, 3>{});
          else add_planes(std::integral_constant<int, 7>{});
          float scl[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) scl[e] = a.res_scale ? h2f(sv8[e]) : 1.0f;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            rv[e] = f2h(mul_f32(s0[e], scl[e]));
            rv[4 + e] = f2h(mul_f32(s1[e], scl[4 + e]));
          }
        } else {
          rv = *reinterpret_cast<const half8_t*>(a.res + src + c);
        }
      }
      if constexpr (MODE == kLn || MODE == kLnMix) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = h2f(xv[e]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[i][e] = h2f(xv[e]) + h2f(rv[e]);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) sum += v[i][e];
    }
  }
  sum = block_sum<NT / 64>(sum, red);
  const float mean = sum / static_cast<float>(C);
  float sv = 0.0f;
#pragma unroll
  for (int i = 0; i < kLnMaxVec; ++i) {
    const int c = (i * kLnThreads + threadIdx.x) * 8;
    if (c < C) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = v[i][e] - mean;
        sv = fmaf(d, d, sv);
      }
    }
  }
  sv = block_sum<NT / 64>(sv, red);
  const float rstd = rsqrtf(sv / static_cast<float>(C) + a.eps);

#pragma unroll
  for (int i = 0; i < kLnMaxVec; ++i) {
    const int c = (i * kLnThreads + threadIdx.x) * 8;
    if (c < C) {
      half8_t yv;
#pragma unroll
      for (int e = 0; e < 8; ++e) yv[e] = f2h(fmaf((v[i][e] - mean) * rstd, h2f(wv[i][e]), h2f(bv[i][e])));
      if constexpr (MODE == kAddLn || MODE == kAddLnMix) {
        half8_t xo;
#pragma unroll
        for (int e = 0; e < 8; ++e) xo[e] = f2h(v[i][e]);
        *reinterpret_cast<half8_t*>(a.x_out + dst + c) = xo;
      }
      if constexpr (MODE == kLnMix) {
        if (a.x_out) {  // the residual stream starts as the (already fp16) embedding row
          half8_t xo;
#pragma unroll
          for (int e = 0; e < 8; ++e) xo[e] = f2h(v[i][e]);
          *reinterpret_cast<half8_t*>(a.x_out + dst + c) = xo;
        }
      }
      if constexpr (kMix) {
        // lerps read the fp16-rounded LN output (rwkv7_v3a_ops.cu:1978-1983)
#pragma unroll
        for (int s = 0; s < 6; ++s) {
          if (s < a.n_mix) {
            half8_t ov;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float yf = h2f(yv[e]);
              ov[e] = f2h(fmaf(h2f(pv[i][e]) - yf, h2f(mv[i][s][e]), yf));
            }
            *reinterpret_cast<half8_t*>(a.out[s] + dst + c) = ov;
          }
        }
        *reinterpret_cast<half8_t*>(a.shift + dst + c) = yv;
        if (a.y) *reinterpret_cast<half8_t*>(a.y + dst + c) = yv;
      } else {
        *reinterpret_cast<half8_t*>(a.y + dst + c) = yv;
      }
    }
  }
}

// ---- residual add + LayerNorm + token shift over sequences (prefill chunks): one block per row (b, t) ----------
// The lerps of row t need the LayerNorm output of row t - 1, which another block computes: instead of a launch of
// its own between the two (the LN rows written and read back, 5 us of launch and ramp), the block normalises the
// previous row a second time - the same loads, the same arithmetic in the same order, so bitwise the value the
// previous row's block gets.  At t == 0 the previous output is the shift row of the state.  Blocks of other rows
// read that shift row while this launch runs, so the new one (the LN output at t == T - 1) goes to shift_next and
// the caller moves it over afterwards.
template <int NT>
__device__ __forceinline__ void block_sum2(float& a, float& b, float* scratch) {  // block_sum's order, two values
  a = wave_sum_dpp(a);
  b = wave_sum_dpp(b);
  if constexpr (NT / 64 == 1) return;
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    scratch[wave] = a;
    scratch[NT / 64 + wave] = b;
  }
  __syncthreads();
  float ta = 0.0f, tb = 0.0f;
#pragma unroll
  for (int i = 0; i < NT / 64; ++i) {
    ta += scratch[i];
    tb += scratch[NT / 64 + i];
  }
  a = ta;
  b = tb;
}

template <int NT>
__global__ __launch_bounds__(NT) void ln_mix_seq_kernel(LnArgs a) {
  __shared__ float red[2 * (NT / 64)];
  const int row = blockIdx.x;
  const int C = a.C;
  const int bi = row / a.T;
  const int t = row - bi * a.T;
  const bool live = static_cast<int>(threadIdx.x) * 8 < C;
  const int c = live ? threadIdx.x * 8 : 0;  // idle threads repeat slice 0 and store nothing
  const int64_t o = static_cast<int64_t>(row) * C + c;
  const int64_t op = t > 0 ? o - C : o;  // the previous row; at t == 0 this row again, unused

  // every load of the kernel up front, none under a per-lane branch
  const half8_t wv = *reinterpret_cast<const half8_t*>(a.w + c);
  const half8_t bv = *reinterpret_cast<const half8_t*>(a.b + c);
  const half8_t sh = *reinterpret_cast<const half8_t*>(a.shift + static_cast<int64_t>(bi) * C + c);
  half8_t mv[6];
#pragma unroll
  for (int s = 0; s < 6; ++s) mv[s] = *reinterpret_cast<const half8_t*>(a.mu[s < a.n_mix ? s : a.n_mix - 1] + c);
  const half8_t xv = *reinterpret_cast<const half8_t*>(a.x + o);
  const half8_t xp = *reinterpret_cast<const half8_t*>(a.x + op);
  half8_t rv, rp;
  if (a.res_partial) {
    const half8_t sv8 = *reinterpret_cast<const half8_t*>((a.res_scale ? a.res_scale : a.w) + c);
    const float* pp = a.res_partial + o;
    const float* pq = a.res_partial + op;
    float4_t s0 = *reinterpret_cast<const float4_t*>(pp), s1 = *reinterpret_cast<const float4_t*>(pp + 4);
    float4_t u0 = *reinterpret_cast<const float4_t*>(pq), u1 = *reinterpret_cast<const float4_t*>(pq + 4);
    // the other partials four at a time, all requested before the first is added, in split order (ln_fused_kernel)
    for (int base = 1; base < a.res_splits; base += 4) {
      float4_t q0[4], q1[4], p0[4], p1[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int64_t sp = (base + u < a.res_splits ? base + u : a.res_splits - 1) * a.res_plane;
        q0[u] = *reinterpret_cast<const float4_t*>(pp + sp);
        q1[u] = *reinterpret_cast<const float4_t*>(pp + sp + 4);
        p0[u] = *reinterpret_cast<const float4_t*>(pq + sp);
        p1[u] = *reinterpret_cast<const float4_t*>(pq + sp + 4);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) asm volatile("" : "+v"(q0[u]), "+v"(q1[u]), "+v"(p0[u]), "+v"(p1[u]));
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        if (base + u < a.res_splits) {
          s0 = s0 + q0[u]; s1 = s1 + q1[u];
          u0 = u0 + p0[u]; u1 = u1 + p1[u];
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float sl = a.res_scale ? h2f(sv8[e]) : 1.0f, sh4 = a.res_scale ? h2f(sv8[4 + e]) : 1.0f;
      rv[e] = f2h(mul_f32(s0[e], sl)); rv[4 + e] = f2h(mul_f32(s1[e], sh4));
      rp[e] = f2h(mul_f32(u0[e], sl)); rp[4 + e] = f2h(mul_f32(u1[e], sh4));
    }
  } else {
    rv = *reinterpret_cast<const half8_t*>(a.res + o);
    rp = *reinterpret_cast<const half8_t*>(a.res + op);
  }

  float v[8], vp[8];
  float sum = 0.0f, sump = 0.0f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    v[e] = h2f(xv[e]) + h2f(rv[e]);
    vp[e] = h2f(xp[e]) + h2f(rp[e]);
    if (!live) v[e] = vp[e] = 0.0f;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) sum += v[e];
#pragma unroll
  for (int e = 0; e < 8; ++e) sump += vp[e];
  block_sum2<NT>(sum, sump, red);
  const float mean = sum / static_cast<float>(C), meanp = sump / static_cast<float>(C);
  float sv = 0.0f, svp = 0.0f;
  if (live) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = v[e] - mean;
      sv = fmaf(d, d, sv);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float d = vp[e] - meanp;
      svp = fmaf(d, d, svp);
    }
  }
  block_sum2<NT>(sv, svp, red);
  const float rstd = rsqrtf(sv / static_cast<float>(C) + a.eps);
  const float rstdp = rsqrtf(svp / static_cast<float>(C) + a.eps);
  if (!live) return;

  half8_t yv, xo;
  float prev[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    // Both outputs as an fp32 fma rounded to fp16 afterwards (what the LayerNorm kernels store).  Left alone, the
    // compiler folds the conversion of the one that is not stored into the fma (v_fma_mixlo_f16: one rounding
    // instead of two), and the previous row's value then differs from what that row's own block gets in one
    // element of some ten thousand.  The same for the lerps below, against token_shift_mix_kernel.
    yv[e] = f2h_apart(fmaf((v[e] - mean) * rstd, h2f(wv[e]), h2f(bv[e])));
    const half_t yp = f2h_apart(fmaf((vp[e] - meanp) * rstdp, h2f(wv[e]), h2f(bv[e])));
    prev[e] = t > 0 ? h2f(yp) : h2f(sh[e]);
    xo[e] = f2h(v[e]);
  }
  *reinterpret_cast<half8_t*>(a.x_out + o) = xo;
  // lerps read the fp16-rounded LN output (rwkv7_v3a_ops.cu:1978-1983)
#pragma unroll
  for (int s = 0; s < 6; ++s) {
    if (s < a.n_mix) {
      half8_t ov;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float yf = h2f(yv[e]);
        ov[e] = f2h_apart(fmaf(prev[e] - yf, h2f(mv[s][e]), yf));
      }
      *reinterpret_cast<half8_t*>(a.out[s] + o) = ov;
    }
  }
  if (a.y) *reinterpret_cast<half8_t*>(a.y + o) = yv;
  if (t == a.T - 1) *reinterpret_cast<half8_t*>(a.shift_next + static_cast<int64_t>(bi) * C + c) = yv;
}

// The same for many rows: a block walks several consecutive rows, so that only the row before its first one is normalised a
// second time, and keeps the LayerNorm output of the row before in registers.  Bound by memory: against a LayerNorm and a
// token-shift launch the LN rows are neither written nor read again.  The loads of the next row are in flight during the
// reductions of this one.  Statements and order of ln_mix_seq_kernel: the same bits.  Two blocks per CU and at least two rows per
// block, at most four (three from 1536 rows on, four from 2048): us of LN1 + LN2 with 1 / 2 / 4 / 8 rows per block: 2048 rows x 4096 63.9 /
// 50.4 / 46.8 / 47.8 (two launches each 66.3), 999 x 2048 21.5 / 18.1 / 19.1 / 26.7 (25.4).  us per layer of whole prefill calls, a LayerNorm and a
// token-shift launch / this: 257 rows x 768 80.8 / 78.8, x 2048 133.2 / 130.3, x 4096 (int8) 287.9 / 285.1; 1536 x 4096 1036 / 1023.
// PLANES: split-K planes of the residual requested ahead (0: a plain fp16 residual); further ones are read in line.
template <int NT, int PLANES>
__global__ __launch_bounds__(NT) void ln_mix_rows_kernel(LnArgs a, int rows, int rows_per_block) {
  constexpr int NW = NT / 64;
  __shared__ float red[2][2][NW];  // by row parity: a buffer is written again two barriers after it was read
  const int C = a.C;
  const int first = blockIdx.x * rows_per_block;
  const int n = min(rows_per_block, rows - first);
  int bi = first / a.T;
  int t = first - bi * a.T;
  const bool live = static_cast<int>(threadIdx.x) * 8 < C;
  const int c = live ? threadIdx.x * 8 : 0;  // idle threads repeat slice 0 and store nothing
  const int wave = threadIdx.x >> 6;

  struct Raw {
    half8_t x, r;
    float4_t q[PLANES > 0 ? 2 * PLANES : 1];
  };
  auto request = [&](int row, Raw& o) {
    const int64_t at = static_cast<int64_t>(row) * C + c;
    o.x = *reinterpret_cast<const half8_t*>(a.x + at);
    if constexpr (PLANES == 0) {
      o.r = *reinterpret_cast<const half8_t*>(a.res + at);
    } else {
#pragma unroll
      for (int u = 0; u < PLANES; ++u) {
        const float* p = a.res_partial + at + (u < a.res_splits ? u : a.res_splits - 1) * a.res_plane;
        o.q[2 * u] = *reinterpret_cast<const float4_t*>(p);
        o.q[2 * u + 1] = *reinterpret_cast<const float4_t*>(p + 4);
      }
    }
  };
  const half8_t wv = *reinterpret_cast<const half8_t*>(a.w + c);
  const half8_t bv = *reinterpret_cast<const half8_t*>(a.b + c);
  half8_t mv[6];
#pragma unroll
  for (int s = 0; s < 6; ++s) mv[s] = *reinterpret_cast<const half8_t*>(a.mu[s < a.n_mix ? s : a.n_mix - 1] + c);
  half8_t sv8 = wv;
  if constexpr (PLANES > 0) {
    if (a.res_scale) sv8 = *reinterpret_cast<const half8_t*>(a.res_scale + c);
  }
  half8_t prev = *reinterpret_cast<const half8_t*>(a.shift + static_cast<int64_t>(bi) * C + c);
  Raw cur, next;
  int i = t > 0 ? -1 : 0;  // -1: the row before, for its output alone
  request(first + i, cur);
  for (; i < n; ++i) {
    request(first + min(i + 1, n - 1), next);
    half8_t rv = cur.r;
    if constexpr (PLANES > 0) {
      float4_t s0 = cur.q[0], s1 = cur.q[1];
#pragma unroll
      for (int u = 1; u < PLANES; ++u) {
        if (u < a.res_splits) {
          s0 = s0 + cur.q[2 * u];
          s1 = s1 + cur.q[2 * u + 1];
        }
      }
      for (int u = PLANES; u < a.res_splits; ++u) {
        const float* p = a.res_partial + static_cast<int64_t>(first + i) * C + c + u * a.res_plane;
        s0 = s0 + *reinterpret_cast<const float4_t*>(p);
        s1 = s1 + *reinterpret_cast<const float4_t*>(p + 4);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        rv[e] = f2h(mul_f32(s0[e], a.res_scale ? h2f(sv8[e]) : 1.0f));
        rv[4 + e] = f2h(mul_f32(s1[e], a.res_scale ? h2f(sv8[4 + e]) : 1.0f));
      }
    }
    float v[8];
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = live ? h2f(cur.x[e]) + h2f(rv[e]) : 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) sum += v[e];
    auto block_total = [&](float x, float* scratch) {  // block_sum's order
      x = wave_sum_dpp(x);
      if ((threadIdx.x & 63) == 0) scratch[wave] = x;
      __syncthreads();
      float total = 0.0f;
#pragma unroll
      for (int w = 0; w < NW; ++w) total += scratch[w];
      return total;
    };
    const float mean = block_total(sum, red[i & 1][0]) / static_cast<float>(C);
    float sq = 0.0f;
    if (live) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float d = v[e] - mean;
        sq = fmaf(d, d, sq);
      }
    }
    const float rstd = rsqrtf(block_total(sq, red[i & 1][1]) / static_cast<float>(C) + a.eps);
    half8_t yv;
#pragma unroll
    for (int e = 0; e < 8; ++e) yv[e] = f2h_apart(fmaf((v[e] - mean) * rstd, h2f(wv[e]), h2f(bv[e])));
    cur = next;
    if (i < 0) {
      prev = yv;
      continue;
    }
    if (live) {
      const int64_t o = static_cast<int64_t>(first + i) * C + c;
      half8_t xo;
#pragma unroll
      for (int e = 0; e < 8; ++e) xo[e] = f2h(v[e]);
      *reinterpret_cast<half8_t*>(a.x_out + o) = xo;
      if (a.y) *reinterpret_cast<half8_t*>(a.y + o) = yv;
      // lerps read the fp16-rounded LN output (rwkv7_v3a_ops.cu:1978-1983)
#pragma unroll
      for (int s = 0; s < 6; ++s) {
        if (s < a.n_mix) {
          half8_t ov;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float yf = h2f(yv[e]);
            ov[e] = f2h_apart(fmaf(h2f(prev[e]) - yf, h2f(mv[s][e]), yf));
          }
          *reinterpret_cast<half8_t*>(a.out[s] + o) = ov;
        }
      }
      if (t == a.T - 1) *reinterpret_cast<half8_t*>(a.shift_next + static_cast<int64_t>(bi) * C + c) = yv;
    }
    prev = yv;
    if (++t == a.T) {
      t = 0;
      ++bi;
      if (i + 1 < n) prev = *reinterpret_cast<const half8_t*>(a.shift + static_cast<int64_t>(bi) * C + c);
    }
  }
}

template <int NT>
static void ln_mix_rows_launch(hipStream_t st, int rows, const LnArgs& a) {
  const int per = std::max(2, std::min(kMixRows, rows / (2 * device_cu_count())));
  const dim3 grid(ceil_div(rows, per));
  if (!a.res_partial) hipLaunchKernelGGL((ln_mix_rows_kernel<NT, 0>), grid, dim3(NT), 0, st, a, rows, per);
  else if (a.res_splits <= 2) hipLaunchKernelGGL((ln_mix_rows_kernel<NT, 2>), grid, dim3(NT), 0, st, a, rows, per);
  else hipLaunchKernelGGL((ln_mix_rows_kernel<NT, 4>), grid, dim3(NT), 0, st, a, rows, per);
}

static int check_ln_shape(int rows, int C) {
  RWKV_REQUIRE(rows > 0, "layer norm: rows must be positive");
  RWKV_REQUIRE(C > 0 && C % 8 == 0 && C <= kLnMaxThreads * 8,
               "layer norm: C (%d) must be a multiple of 8 and at most %d", C, kLnMaxThreads * 8);
  return RWKV_OK;
}

template <int NT>
static int ln_launch_nt(hipStream_t st, int mode, int rows, const LnArgs& a) {
  switch (mode) {
    case kLn: hipLaunchKernelGGL((ln_fused_kernel<kLn, NT>), dim3(rows), dim3(NT), 0, st, a); break;
    case kAddLn: hipLaunchKernelGGL((ln_fused_kernel<kAddLn, NT>), dim3(rows), dim3(NT), 0, st, a); break;
    case kAddLastLn: hipLaunchKernelGGL((ln_fused_kernel<kAddLastLn, NT>), dim3(rows), dim3(NT), 0, st, a); break;
    case kAddLnMix: hipLaunchKernelGGL((ln_fused_kernel<kAddLnMix, NT>), dim3(rows), dim3(NT), 0, st, a); break;
    case kLnMix: hipLaunchKernelGGL((ln_fused_kernel<kLnMix, NT>), dim3(rows), dim3(NT), 0, st, a); break;
    default: set_error("bad layer-norm mode %d", mode); return RWKV_E_INVALID;
  }
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int ln_launch(hipStream_t st, int mode, int rows, const LnArgs& a) {
  if (int rc = check_ln_shape(rows, a.C)) return rc;
  if (mode == kAddLnMixSeq) {
    RWKV_REQUIRE(a.C <= 512 * 8, "layer norm + token shift over a sequence: C (%d) must be at most 4096", a.C);
    RWKV_REQUIRE(a.T >= 1 && rows % a.T == 0 && a.shift && a.shift_next && a.x_out && a.n_mix >= 1 && a.n_mix <= 6 &&
                     (a.res || a.res_partial),
                 "layer norm + token shift over a sequence: bad arguments");
    // the block of row t reads x and the residual of row t - 1 again while that row's block stores its outputs:
    // no output may share memory with an input
    RWKV_REQUIRE(a.x_out != a.x && a.y != a.x && (a.res == nullptr || (a.x_out != a.res && a.y != a.res)),
                 "layer norm + token shift over a sequence: outputs must not alias x or the residual");
    if (rows > kMixSeqRows) {
      if (a.C <= 256 * 8) ln_mix_rows_launch<256>(st, rows, a);
      else ln_mix_rows_launch<512>(st, rows, a);
    } else if (a.C <= 256 * 8) hipLaunchKernelGGL(ln_mix_seq_kernel<256>, dim3(rows), dim3(256), 0, st, a);
    else hipLaunchKernelGGL(ln_mix_seq_kernel<512>, dim3(rows), dim3(512), 0, st, a);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
  }
  if (a.C <= 256 * 8) return ln_launch_nt<256>(st, mode, rows, a);
  if (a.C <= 512 * 8) return ln_launch_nt<512>(st, mode, rows, a);
  return ln_launch_nt<1024>(st, mode, rows, a);
}

// ---- token shift: out_s = x + (prev - x) * mu_s with prev = shift[b] at t == 0, else x[b,t-1];
// then shift[b] = x[b,T-1].  One thread per (row, 8 channels); the thread of token 0 reads the old shift slice
// and then overwrites it, so no thread can overwrite a slice another one still has to read. ------------

__global__ __launch_bounds__(256) void token_shift_mix_kernel(MixArgs a) {
  const int cvecs = a.C / 8;
  const int64_t idx = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (idx >= static_cast<int64_t>(a.B) * a.T * cvecs) return;
  const int64_t row = idx / cvecs;
  const int c = static_cast<int>(idx - row * cvecs) * 8;
  const int b = static_cast<int>(row / a.T);
  const int t = static_cast<int>(row - static_cast<int64_t>(b) * a.T);
  const int64_t o = row * a.C + c;
  const half8_t cur = *reinterpret_cast<const half8_t*>(a.x + o);
  const half8_t prev = (t == 0) ? *reinterpret_cast<const half8_t*>(a.shift + static_cast<int64_t>(b) * a.C + c)
                                : *reinterpret_cast<const half8_t*>(a.x + o - a.C);
  for (int s = 0; s < a.n_mix; ++s) {
    const half8_t mu = *reinterpret_cast<const half8_t*>(a.mu[s] + c);
    half8_t ov;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float cf = h2f(cur[e]);
      ov[e] = f2h(cf + (h2f(prev[e]) - cf) * h2f(mu[e]));
    }
    *reinterpret_cast<half8_t*>(a.out[s] + o) = ov;
  }
  // the thread that read the old shift slice replaces it with the last token's slice: no other thread touches it
  if (t == 0) {
    const half8_t last = (a.T == 1) ? cur : *reinterpret_cast<const half8_t*>(a.x + o + static_cast<int64_t>(a.T - 1) * a.C);
    *reinterpret_cast<half8_t*>(a.shift + static_cast<int64_t>(b) * a.C + c) = last;
  }
}

int token_shift_mix_launch(hipStream_t st, const MixArgs& a) {
  RWKV_REQUIRE(a.B > 0 && a.T > 0 && a.C > 0 && a.C % 8 == 0, "token shift: bad shape B=%d T=%d C=%d", a.B, a.T, a.C);
  RWKV_REQUIRE(a.n_mix >= 1 && a.n_mix <= 6, "token shift: n_mix %d out of range", a.n_mix);
  const int64_t n = static_cast<int64_t>(a.B) * a.T * (a.C / 8);
  hipLaunchKernelGGL(token_shift_mix_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, a);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

// ---- kk normalise + a-gate, GroupNorm + rkv residual + gate: 16 lanes per (row, head), four channels per lane ------------
// Both read and write a few fp16 rows once: with one channel per lane their requests were 128 bytes per wavefront and the
// sums six trips through LDS each.  Four channels per lane make requests of 512 bytes and keep the sums in the registers of a DPP row;
// eight would halve the blocks of a 128-row chunk, which are two per CU.  us, before -> now: 999 rows x 32 heads 12.5 and 9.7
// -> 9.4 and 5.8; 128 rows x 64 heads 5.2 and 4.6 -> 5.3 and 4.7 (launch and latency).
// kk / a-gate of fewer than 12 heads per CU keeps one channel per lane: its chain of divisions and exponentials, four times as
// long with four of them, is then all there is (kk_a_gate_few_kernel; us, back to back, four channels / one: 17 rows x 64 heads 2.24 / 2.05,
// 64 x 32 2.30 / 2.14, 96 x 32 2.29 / 2.35, 128 x 64 2.84 / 3.26).

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

template <bool VEC>
__global__ __launch_bounds__(256) void kk_a_gate_kernel(KkArgs p) {
  const int64_t rh = static_cast<int64_t>(blockIdx.x) * 16 + (threadIdx.x >> 4);
  if (rh >= p.rows_heads) return;  // whole groups of 16 lanes
  const int h = static_cast<int>(rh % p.H);
  const int64_t idx = rh * kHead + 4 * (threadIdx.x & 15);
  const int c = h * kHead + 4 * (threadIdx.x & 15);
  const half4_t k4 = load4<VEC>(p.k + idx), a4 = load4<VEC>(p.a12 + idx);
  const half4_t kk4 = load4<VEC>(p.k_k + c), a04 = load4<VEC>(p.a0 + c), ka4 = load4<VEC>(p.k_a + c);
  half4_t w4 = {}, w04 = {};
  if (p.d32 || p.w_sum16) {
    w4 = load4<VEC>(p.w12 + idx);
    w04 = load4<VEC>(p.w0 + c);
  }
  const HeadGate o = head_gate(k4, a4, w4, kk4, a04, ka4, w04);
  if (p.new_k) store4<VEC>(p.new_k + idx, o.new_k);
  if (p.neg_kk) store4<VEC>(p.neg_kk + idx, o.neg_kk);
  if (p.kka) store4<VEC>(p.kka + idx, o.kka);
  if (p.d32) {
    float4_t d;
#pragma unroll
    for (int e = 0; e < 4; ++e) d[e] = head_decay(o.w_sum[e]);
    *reinterpret_cast<float4_t*>(p.d32 + idx) = d;
  }
  if (p.w_sum16) store4<VEC>(p.w_sum16 + idx, o.w_sum);
}

constexpr int kKkFewHeads = 12;  // per CU

// one wavefront per (row, head), lane = channel; few enough heads for 32-bit indices
__global__ __launch_bounds__(256) void kk_a_gate_few_kernel(KkArgs p) {
  const int rh = static_cast<int>(blockIdx.x * 4 + (threadIdx.x >> 6));
  if (rh >= static_cast<int>(p.rows_heads)) return;
  const int lane = threadIdx.x & 63;
  const int idx = rh * kHead + lane;
  const int c = rh % p.H * kHead + lane;
  const float kv = h2f(p.k[idx]);
  const float u = kv * h2f(p.k_k[c]);
  const float total = wave_sum(u * u);
  const float inv = 1.0f / fmaxf(sqrtf(total), kKkEps);
  const float kk = u * inv;
  const float av = sigmoid_f(h2f(p.a0[c]) + h2f(p.a12[idx]));
  const float ka = h2f(p.k_a[c]);
  const half_t nk = f2h(kv * fmaf(av, ka, 1.0f - ka));
  const half_t nkk = f2h(-kk);
  const half_t kka = f2h(kk * av);
  if (p.new_k) p.new_k[idx] = nk;
  if (p.neg_kk) p.neg_kk[idx] = nkk;
  if (p.kka) p.kka[idx] = kka;
  if (p.d32 || p.w_sum16) {
    const half_t ws = f2h(h2f(p.w12[idx]) + h2f(p.w0[c]));  // rwkv7_add_vec_launch rounding point
    if (p.d32) p.d32[idx] = exp2f(-0.8750387749145276f / (1.0f + exp2f(-1.4426950408889634f * h2f(ws))));
    if (p.w_sum16) p.w_sum16[idx] = ws;
  }
}

int kk_a_gate_launch(hipStream_t st, const KkArgs& p) {
  RWKV_REQUIRE(p.rows_heads > 0 && p.H > 0, "kk_a_gate: bad shape");
  RWKV_REQUIRE(p.w_sum16 == nullptr || (p.w12 && p.w0), "kk_a_gate: the rounded decay logit needs w12 and w0");
  RWKV_REQUIRE(reinterpret_cast<uintptr_t>(p.d32) % 16 == 0, "kk_a_gate: the decay must be 16-byte aligned");
  if (p.rows_heads < kKkFewHeads * device_cu_count()) {
    hipLaunchKernelGGL(kk_a_gate_few_kernel, dim3(ceil_div(p.rows_heads, 4)), dim3(256), 0, st, p);
    RWKV_LAUNCH_CHECK();
    return RWKV_OK;
  }
  const uintptr_t bits = reinterpret_cast<uintptr_t>(p.k) | reinterpret_cast<uintptr_t>(p.a12) | reinterpret_cast<uintptr_t>(p.k_k) |
                         reinterpret_cast<uintptr_t>(p.a0) | reinterpret_cast<uintptr_t>(p.k_a) | reinterpret_cast<uintptr_t>(p.w12) |
                         reinterpret_cast<uintptr_t>(p.w0) | reinterpret_cast<uintptr_t>(p.new_k) |
                         reinterpret_cast<uintptr_t>(p.neg_kk) | reinterpret_cast<uintptr_t>(p.kka) |
                         reinterpret_cast<uintptr_t>(p.w_sum16);
  const dim3 grid(ceil_div(p.rows_heads, 16));
  if (bits % 8 == 0) hipLaunchKernelGGL(kk_a_gate_kernel<true>, grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL(kk_a_gate_kernel<false>, grid, dim3(256), 0, st, p);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

template <bool VEC>
__global__ __launch_bounds__(256) void lnx_rkvres_xg_kernel(int64_t rows_heads, int H, const half_t* __restrict__ y,
                                                            const half_t* __restrict__ r, const half_t* __restrict__ k,
                                                            const half_t* __restrict__ v, const half_t* __restrict__ r_k,
                                                            const half_t* __restrict__ lnw, const half_t* __restrict__ lnb,
                                                            const half_t* __restrict__ g, half_t* out) {
  const int64_t rh = static_cast<int64_t>(blockIdx.x) * 16 + (threadIdx.x >> 4);
  if (rh >= rows_heads) return;  // whole groups of 16 lanes
  const int h = static_cast<int>(rh % H);
  const int64_t idx = rh * kHead + 4 * (threadIdx.x & 15);
  const int c = h * kHead + 4 * (threadIdx.x & 15);
  const half4_t y4 = load4<VEC>(y + idx), r4 = load4<VEC>(r + idx), k4 = load4<VEC>(k + idx), v4 = load4<VEC>(v + idx),
                g4 = load4<VEC>(g + idx);
  const half4_t rk4 = load4<VEC>(r_k + c), lw4 = load4<VEC>(lnw + c), lb4 = load4<VEC>(lnb + c);
  float yv[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) yv[e] = h2f(y4[e]);
  store4<VEC>(out + idx, head_output(yv, r4, k4, v4, g4, rk4, lw4, lb4));
}

// ---- small element-wise kernels ---------------------------------------------------------------------
__global__ __launch_bounds__(256) void relu_square_kernel(int64_t n, const half_t* __restrict__ x, half_t* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  const float v = fmaxf(h2f(x[i]), 0.0f);
  out[i] = f2h(v * v);
}

__global__ __launch_bounds__(256) void add_vec_kernel(int64_t n, int C, const half_t* __restrict__ x,
                                                      const half_t* __restrict__ vec, half_t* __restrict__ out) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  out[i] = f2h(h2f(x[i]) + h2f(vec[i % C]));
}

__global__ __launch_bounds__(256) void f16_to_f32_kernel(int64_t n, const half_t* __restrict__ src, float* __restrict__ dst) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= n) return;
  dst[i] = h2f(src[i]);
}

__global__ __launch_bounds__(256) void advance_i32_kernel(int n, int amount, int* __restrict__ x) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) x[i] += amount;
}

// gather embedding rows for T > 1: out[row] = table[tokens[row]]
__global__ __launch_bounds__(256) void embed_gather_kernel(int C, const int64_t* __restrict__ tokens,
                                                           const half_t* __restrict__ table, half_t* __restrict__ out) {
  const int row = blockIdx.x;
  const int64_t src = tokens[row] * static_cast<int64_t>(C);
  for (int c = threadIdx.x * 8; c < C; c += 256 * 8)
    *reinterpret_cast<half8_t*>(out + static_cast<int64_t>(row) * C + c) = *reinterpret_cast<const half8_t*>(table + src + c);
}

int embed_gather_launch(hipStream_t st, int rows, int C, const int64_t* tokens, const half_t* table, half_t* out) {
  hipLaunchKernelGGL(embed_gather_kernel, dim3(rows), dim3(256), 0, st, C, tokens, table, out);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int lnx_launch(hipStream_t st, int64_t rows_heads, int H, const half_t* y, const half_t* r, const half_t* k,
               const half_t* v, const half_t* r_k, const half_t* lnw, const half_t* lnb, const half_t* g, half_t* out) {
  const uintptr_t bits = reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(r) | reinterpret_cast<uintptr_t>(k) |
                         reinterpret_cast<uintptr_t>(v) | reinterpret_cast<uintptr_t>(r_k) | reinterpret_cast<uintptr_t>(lnw) |
                         reinterpret_cast<uintptr_t>(lnb) | reinterpret_cast<uintptr_t>(g) | reinterpret_cast<uintptr_t>(out);
  const dim3 grid(ceil_div(rows_heads, 16));
  if (bits % 8 == 0)
    hipLaunchKernelGGL(lnx_rkvres_xg_kernel<true>, grid, dim3(256), 0, st, rows_heads, H, y, r, k, v, r_k, lnw, lnb, g, out);
  else
    hipLaunchKernelGGL(lnx_rkvres_xg_kernel<false>, grid, dim3(256), 0, st, rows_heads, H, y, r, k, v, r_k, lnw, lnb, g, out);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int add_vec_launch(hipStream_t st, int rows, int C, const half_t* x, const half_t* vec, half_t* out) {
  const int64_t n = static_cast<int64_t>(rows) * C;
  hipLaunchKernelGGL(add_vec_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, C, x, vec, out);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int advance_launch(hipStream_t st, int n, int amount, int* x) {
  hipLaunchKernelGGL(advance_i32_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, st, n, amount, x);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

}  // namespace rwkv

using namespace rwkv;

#define H16(p) static_cast<const half_t*>(p)
#define H16M(p) static_cast<half_t*>(p)

extern "C" {

int rwkv_hip_layer_norm(rwkv_stream_t s, int rows, int C, const void* x, const void* w, const void* b, void* y,
                        float eps) {
  RWKV_REQUIRE(x && w && b && y, "layer_norm: NULL tensor");
  LnArgs a = {};
  a.x = H16(x); a.w = H16(w); a.b = H16(b); a.y = H16M(y); a.C = C; a.T = 1; a.eps = eps;
  return ln_launch(as_stream(s), kLn, rows, a);
}

int rwkv_hip_add_layer_norm(rwkv_stream_t s, int rows, int C, const void* x, const void* res, const void* w,
                            const void* b, void* x_out, void* y, float eps) {
  RWKV_REQUIRE(x && res && w && b && x_out && y, "add_layer_norm: NULL tensor");
  LnArgs a = {};
  a.x = H16(x); a.res = H16(res); a.w = H16(w); a.b = H16(b); a.x_out = H16M(x_out); a.y = H16M(y);
  a.C = C; a.T = 1; a.eps = eps;
  return ln_launch(as_stream(s), kAddLn, rows, a);
}

int rwkv_hip_add_last_layer_norm(rwkv_stream_t s, int B, int T, int C, const void* x, const void* res, const void* w,
                                 const void* b, void* y, float eps) {
  RWKV_REQUIRE(x && res && w && b && y && T > 0, "add_last_layer_norm: bad arguments");
  LnArgs a = {};
  a.x = H16(x); a.res = H16(res); a.w = H16(w); a.b = H16(b); a.y = H16M(y); a.C = C; a.T = T; a.eps = eps;
  return ln_launch(as_stream(s), kAddLastLn, B, a);
}

int rwkv_hip_token_shift_mix(rwkv_stream_t s, int B, int T, int C, int n_mix, const void* x, void* shift,
                             const void* const* mu_host, void* const* out_host) {
  RWKV_REQUIRE(x && shift && mu_host && out_host, "token_shift_mix: NULL tensor");
  RWKV_REQUIRE(n_mix >= 1 && n_mix <= 6, "token_shift_mix: n_mix %d out of range", n_mix);
  MixArgs a = {};
  a.x = H16(x); a.shift = H16M(shift); a.B = B; a.T = T; a.C = C; a.n_mix = n_mix;
  for (int i = 0; i < n_mix; ++i) {
    RWKV_REQUIRE(mu_host[i] && out_host[i], "token_shift_mix: NULL tensor");
    a.mu[i] = H16(mu_host[i]);
    a.out[i] = H16M(out_host[i]);
  }
  return token_shift_mix_launch(as_stream(s), a);
}

int rwkv_hip_add_layer_norm_cmix_mix(rwkv_stream_t s, int rows, int C, const void* x, const void* res, void* shift,
                                     const void* w, const void* b, const void* mu_k, void* x_out, void* mixed,
                                     float eps) {
  RWKV_REQUIRE(x && res && shift && w && b && mu_k && x_out && mixed, "add_layer_norm_cmix_mix: NULL tensor");
  LnArgs a = {};
  a.x = H16(x); a.res = H16(res); a.w = H16(w); a.b = H16(b); a.x_out = H16M(x_out); a.shift = H16M(shift);
  a.mu[0] = H16(mu_k); a.out[0] = H16M(mixed); a.n_mix = 1; a.C = C; a.T = 1; a.eps = eps;
  return ln_launch(as_stream(s), kAddLnMix, rows, a);
}

int rwkv_hip_add_layer_norm_tmix_mix6(rwkv_stream_t s, int rows, int C, const void* x, const void* res, void* shift,
                                      const void* w, const void* b, const void* const* mu6_host, void* x_out,
                                      void* const* out6_host, float eps) {
  RWKV_REQUIRE(x && res && shift && w && b && mu6_host && x_out && out6_host, "add_layer_norm_tmix_mix6: NULL tensor");
  LnArgs a = {};
  a.x = H16(x); a.res = H16(res); a.w = H16(w); a.b = H16(b); a.x_out = H16M(x_out); a.shift = H16M(shift);
  for (int i = 0; i < 6; ++i) {
    RWKV_REQUIRE(mu6_host[i] && out6_host[i], "add_layer_norm_tmix_mix6: NULL tensor");
    a.mu[i] = H16(mu6_host[i]);
    a.out[i] = H16M(out6_host[i]);
  }
  a.n_mix = 6; a.C = C; a.T = 1; a.eps = eps;
  return ln_launch(as_stream(s), kAddLnMix, rows, a);
}

int rwkv_hip_kk_a_gate(rwkv_stream_t s, int rows, int C, int H, const void* k, const void* k_k, const void* a0,
                       const void* a12, const void* k_a, void* new_k, void* neg_kk, void* kka) {
  RWKV_REQUIRE(rows > 0 && H > 0 && C == H * kHead, "kk_a_gate: C (%d) must equal H*64", C);
  RWKV_REQUIRE(k && k_k && a0 && a12 && k_a && new_k && neg_kk && kka, "kk_a_gate: NULL tensor");
  KkArgs p = {};
  p.k = H16(k); p.k_k = H16(k_k); p.a0 = H16(a0); p.a12 = H16(a12); p.k_a = H16(k_a);
  p.new_k = H16M(new_k); p.neg_kk = H16M(neg_kk); p.kka = H16M(kka);
  p.rows_heads = static_cast<int64_t>(rows) * H; p.H = H;
  return kk_a_gate_launch(as_stream(s), p);
}

int rwkv_hip_lnx_rkvres_xg(rwkv_stream_t s, int rows, int C, int H, const void* y, const void* r, const void* k,
                           const void* v, const void* r_k, const void* lnw, const void* lnb, const void* g,
                           void* out) {
  RWKV_REQUIRE(rows > 0 && H > 0 && C == H * kHead, "lnx_rkvres_xg: C (%d) must equal H*64", C);
  RWKV_REQUIRE(y && r && k && v && r_k && lnw && lnb && g && out, "lnx_rkvres_xg: NULL tensor");
  return lnx_launch(as_stream(s), static_cast<int64_t>(rows) * H, H, H16(y), H16(r), H16(k), H16(v), H16(r_k),
                    H16(lnw), H16(lnb), H16(g), H16M(out));
}

int rwkv_hip_relu_square(rwkv_stream_t s, int64_t n, const void* x, void* out) {
  RWKV_REQUIRE(n > 0 && x && out, "relu_square: bad arguments");
  hipLaunchKernelGGL(relu_square_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, as_stream(s), n, H16(x), H16M(out));
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int rwkv_hip_add_vec(rwkv_stream_t s, int rows, int C, const void* x, const void* vec, void* out) {
  RWKV_REQUIRE(rows > 0 && C > 0 && x && vec && out, "add_vec: bad arguments");
  return add_vec_launch(as_stream(s), rows, C, H16(x), H16(vec), H16M(out));
}

int rwkv_hip_f16_to_f32(rwkv_stream_t s, int64_t n, const void* src, void* dst) {
  RWKV_REQUIRE(n > 0 && src && dst, "f16_to_f32: bad arguments");
  hipLaunchKernelGGL(f16_to_f32_kernel, dim3(ceil_div(n, 256)), dim3(256), 0, as_stream(s), n, H16(src),
                     static_cast<float*>(dst));
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int rwkv_hip_advance_i32(rwkv_stream_t s, int n, int amount, void* x) {
  RWKV_REQUIRE(n > 0 && x, "advance_i32: bad arguments");
  return advance_launch(as_stream(s), n, amount, static_cast<int*>(x));
}

}  // extern "C"
