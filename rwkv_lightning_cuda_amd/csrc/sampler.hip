// Sampler: repetition penalty, temperature, softmax, top-k / top-p threshold, inverse-CDF draw, penalty update.
//
// Reference: src/utils/sampling.cu:205-471 (with penalties), :613-848 (without), argument
// normalisation :492-512, sf() :139-142.  Same pipeline and the same threshold definition: the
// largest probability value t (searched by bisection on the IEEE bit pattern, :294-362) such that
// {p >= t} still holds at least top_k entries or at least top_p mass; entries equal to t are scaled by
// `comp` so the kept set has exactly top_k entries / top_p mass (:393-404).
//
// gfx950 re-design: rows with a small top_k take three launches (sample_stats_kernel and on, below).  Otherwise one 1024-thread
// block (16 wavefronts) per row; each thread owns a fixed set of entries -
// for rows of up to 65536 entries the float4 t, t + 1024, ..., loaded once (coalesced) and kept in registers
// through the softmax, the bisection and the draw; for larger rows a contiguous slice that stays in `probs` -
// so the draw is a single inverse-CDF walk with one uniform number over a fixed order of the row; block
// reductions are wave64 butterflies (DPP and row swaps, no LDS) + one LDS exchange; a bisection step skips the
// slots whose largest entry lies below its threshold; top_k == 1 (greedy, what top_p == 0 normalises to) skips the
// bisection.  Randomness is counter-based Philox4x32-10 keyed by (seed; row, step) instead of a
// per-row cuRAND state seeded from the wall clock (src/rwkv_sampler.cpp:14-19), so a run is reproducible.
#include <cfloat>
#include <type_traits>

#include "ops.h"

namespace rwkv {

constexpr int kSampleThreads = 1024;
constexpr int kSampleWaves = kSampleThreads / 64;

__device__ __forceinline__ float sf(float x) {
  const float y = isnan(x) ? 0.0f : x;
  return isinf(y) ? copysignf(FLT_MAX, y) : y;
}

constexpr int kBracket = 256;  // entries between the two ends of the bisection that one wavefront takes over (four per lane)

struct BlockRed {
  float f[kSampleWaves];
  unsigned u[kSampleWaves];
  float bracket[kBracket];
};

template <typename Op>
__device__ __forceinline__ float block_reduce_f(float v, Op op, float* buf) {
  v = wave_reduce_dpp(v, op);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) buf[threadIdx.x >> 6] = v;
  __syncthreads();
  float r = buf[0];
#pragma unroll
  for (int i = 1; i < kSampleWaves; ++i) r = op(r, buf[i]);
  return r;
}

__device__ __forceinline__ unsigned block_sum_u(unsigned v, unsigned* buf) {
  v = wave_reduce_dpp(v, [](unsigned x, unsigned y) { return x + y; });
  __syncthreads();
  if ((threadIdx.x & 63) == 0) buf[threadIdx.x >> 6] = v;
  __syncthreads();
  unsigned r = 0;
#pragma unroll
  for (int i = 0; i < kSampleWaves; ++i) r += buf[i];
  return r;
}

// exclusive prefix over threads (thread order), total returned through *total
__device__ __forceinline__ float block_exclusive_scan(float v, float* buf, float* total) {
  float inc = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const float n = __shfl_up(inc, off, 64);
    if ((threadIdx.x & 63) >= off) inc += n;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 63) buf[threadIdx.x >> 6] = inc;
  __syncthreads();
  float base = 0.0f, tot = 0.0f;
#pragma unroll
  for (int i = 0; i < kSampleWaves; ++i) {
    if (i < static_cast<int>(threadIdx.x >> 6)) base += buf[i];
    tot += buf[i];
  }
  *total = tot;
  return base + inc - v;
}

struct Philox {
  uint32_t c[4];
};
__device__ __forceinline__ Philox philox4x32_10(uint64_t seed, uint64_t ctr_lo, uint64_t ctr_hi) {
  uint32_t k0 = static_cast<uint32_t>(seed), k1 = static_cast<uint32_t>(seed >> 32);
  Philox p = {{static_cast<uint32_t>(ctr_lo), static_cast<uint32_t>(ctr_lo >> 32), static_cast<uint32_t>(ctr_hi),
               static_cast<uint32_t>(ctr_hi >> 32)}};
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * p.c[0];
    const uint64_t p1 = static_cast<uint64_t>(0xCD9E8D57u) * p.c[2];
    const uint32_t n0 = static_cast<uint32_t>(p1 >> 32) ^ p.c[1] ^ k0;
    const uint32_t n1 = static_cast<uint32_t>(p1);
    const uint32_t n2 = static_cast<uint32_t>(p0 >> 32) ^ p.c[3] ^ k1;
    const uint32_t n3 = static_cast<uint32_t>(p0);
    p.c[0] = n0; p.c[1] = n1; p.c[2] = n2; p.c[3] = n3;
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  return p;
}

struct SampleArgs {
  const float* logits;
  float* penalties;  // may be NULL
  float* probs;
  int* out;
  int V;
  float presence, frequency, decay, log2_inv_temp;
  int top_k;
  float top_p;
  uint64_t seed, step;
};

__device__ __forceinline__ float penalised(float logit, float penalty, float log2_inv_temp) {
  return sf((sf(logit) - penalty) * log2_inv_temp);
}

// how much of each of the n_eq entries at the threshold is kept, so that the kept set has top_k entries or top_p mass
__device__ __forceinline__ float tie_share(const SampleArgs& a, float thr, unsigned n_eq, unsigned n_gt, float p_gt) {
  float comp = fminf(sf((a.top_p - p_gt) / (thr * n_eq)), 1.0f);
  comp = fminf(sf(static_cast<float>(a.top_k - static_cast<int>(n_gt)) / n_eq), comp);
  return fmaxf(comp, 0.0f);
}

// uniform in (0,1]: never selects a zero-mass prefix
__device__ __forceinline__ float uniform_of_row(const SampleArgs& a, int b) {
  const Philox rnd = philox4x32_10(a.seed, static_cast<uint64_t>(b), a.step);
  return (static_cast<float>(rnd.c[0] >> 8) + 1.0f) * (1.0f / 16777216.0f);
}

// count and mass of one bisection step through one LDS exchange (the same sums, in the same order, as
// block_sum_u and block_reduce_f one after the other)
__device__ __forceinline__ void block_count_mass(unsigned& c, float& m, BlockRed& red) {
  c = wave_reduce_dpp(c, [](unsigned x, unsigned y) { return x + y; });
  m = wave_reduce_dpp(m, [](float x, float y) { return x + y; });
  __syncthreads();
  if ((threadIdx.x & 63) == 0) {
    red.u[threadIdx.x >> 6] = c;
    red.f[threadIdx.x >> 6] = m;
  }
  __syncthreads();
  unsigned rc = 0;
  float rm = red.f[0];
#pragma unroll
  for (int i = 0; i < kSampleWaves; ++i) rc += red.u[i];
#pragma unroll
  for (int i = 1; i < kSampleWaves; ++i) rm += red.f[i];
  c = rc;
  m = rm;
}

constexpr int kSampleRegVecs = 16;  // float4 per thread held in registers: rows of up to 65536 entries

// REG: a thread's slice of the row (up to 16 float4) stays in registers from the first load to the draw, so
// the softmax, the ~30 bisection steps and the tie count touch no memory; `probs` is not written.  Larger
// rows keep the slice in `probs` (L2) and re-read it in every pass.  Same arithmetic in the same order.
template <bool REG>
__device__ __forceinline__ int sample_row(const SampleArgs& a, int b, BlockRed& red, int& s_pick) {
  const int t = threadIdx.x;
  const int V = a.V;
  const float* logits = a.logits + static_cast<int64_t>(b) * V;
  const float* pen = a.penalties ? a.penalties + static_cast<int64_t>(b) * V : nullptr;
  float* probs = a.probs + static_cast<int64_t>(b) * V;
  // contiguous slice per thread, in units of 4 floats
  const int V4 = V / 4;
  const int per = (V4 + kSampleThreads - 1) / kSampleThreads;
  const int i0 = min(t * per, V4);
  const int i1 = min(i0 + per, V4);
  // REG: thread t owns the float4 t, t + 1024, ... (every load of a wavefront is one contiguous KiB); the draw
  // walks the kept entries thread by thread, a fixed permutation of the row, which leaves every entry its probability.
  const int n = REG ? (t < V4 ? min((V4 - t + kSampleThreads - 1) / kSampleThreads, kSampleRegVecs) : 0) : i1 - i0;
  auto fmax_op = [](float x, float y) { return fmaxf(x, y); };
  auto fmin_op = [](float x, float y) { return fminf(x, y); };
  auto fadd_op = [](float x, float y) { return x + y; };

  float4_t vals[REG ? kSampleRegVecs : 1];
  // f(q, i): q = position in the slice, i = float4 index in the row
  auto for_each = [&](auto&& f) {
    if constexpr (REG) {
#pragma unroll
      for (int q = 0; q < kSampleRegVecs; ++q)
        if (q < n) f(q, q * kSampleThreads + t);
    } else {
      for (int i = i0; i < i1; ++i) f(0, i);
    }
  };
  auto get = [&](int q, int i) -> float4_t {
    if constexpr (REG) return vals[q];
    else return reinterpret_cast<const float4_t*>(probs)[i];
  };
  auto put = [&](int q, int i, const float4_t& v) {
    if constexpr (REG) vals[q] = v;
    else reinterpret_cast<float4_t*>(probs)[i] = v;
  };

  // 1. penalised, temperature-scaled logits in base-2 units; row maximum and its lowest index
  if constexpr (REG) {
#pragma unroll
    for (int q = 0; q < kSampleRegVecs; ++q)  // all loads of the slice in flight together
      if (q < n) vals[q] = reinterpret_cast<const float4_t*>(logits)[q * kSampleThreads + t];
  }
  float maxu = -INFINITY;
  int maxi = 0x7fffffff;
  for_each([&](int q, int i) {
    float4_t l;
    if constexpr (REG) l = vals[q];
    else l = reinterpret_cast<const float4_t*>(logits)[i];
    float4_t p = {0.0f, 0.0f, 0.0f, 0.0f};
    if (pen) p = reinterpret_cast<const float4_t*>(pen)[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      l[j] = penalised(l[j], p[j], a.log2_inv_temp);
      if (l[j] > maxu) {
        maxu = l[j];
        maxi = i * 4 + j;
      }
    }
    put(q, i, l);
  });
  const float gmax = block_reduce_f(maxu, fmax_op, red.f);
  int pick = -1;

  if (a.top_k == 1) {
    // greedy: lowest index among the maxima (the reference draws uniformly among exact ties)
    unsigned cand = (maxu == gmax) ? static_cast<unsigned>(maxi) : 0x7fffffffu;
    cand = wave_reduce_dpp(cand, [](unsigned x, unsigned y) { return min(x, y); });
    __syncthreads();
    if ((t & 63) == 0) red.u[t >> 6] = cand;
    __syncthreads();
    unsigned best = red.u[0];
#pragma unroll
    for (int i = 1; i < kSampleWaves; ++i) best = min(best, red.u[i]);
    pick = static_cast<int>(best);
  } else {
    // 2.-3. softmax
    float den = 0.0f;
    for_each([&](int q, int i) {
      const float4_t l = get(q, i);
      const float4_t e = {exp2f(l[0] - gmax), exp2f(l[1] - gmax), exp2f(l[2] - gmax), exp2f(l[3] - gmax)};
      den += e[0] + e[1] + e[2] + e[3];
      if constexpr (REG) put(q, i, e);  // registers keep the exponentials for the division below
    });
    den = block_reduce_f(den, fadd_op, red.f);
    float pmax = -INFINITY, pmin = INFINITY;
    for_each([&](int q, int i) {
      float4_t l = get(q, i);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        l[j] = (REG ? l[j] : exp2f(l[j] - gmax)) / den;
        pmax = fmaxf(pmax, l[j]);
        pmin = fminf(pmin, l[j]);
      }
      put(q, i, l);
    });
    const bool bisect = a.top_k < V || a.top_p < 1.0f;  // (else the loop below does not run: no threshold to find)
    // REG: the largest probability among the 256 entries that this wavefront holds in slot q (bit pattern; the same
    // in every lane).  A bisection step whose threshold lies above it has nothing to count there.
    unsigned slot_max[REG ? kSampleRegVecs : 1];
    if constexpr (REG) {
#pragma unroll
      for (int q = 0; q < kSampleRegVecs; ++q) slot_max[q] = 0xffffffffu;
    }
    if (REG && bisect) {
#pragma unroll
      for (int q = 0; q < kSampleRegVecs; ++q) {
        float mx = 0.0f;
        if (q < n) mx = fmaxf(fmaxf(vals[q][0], vals[q][1]), fmaxf(vals[q][2], vals[q][3]));
        mx = wave_reduce_dpp(mx, fmax_op);
        slot_max[q] = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, mx)));
      }
    }
    pmax = block_reduce_f(pmax, fmax_op, red.f);
    pmin = block_reduce_f(pmin, fmin_op, red.f);

    // 4. threshold by bisection on the bit pattern
    unsigned left = __float_as_uint(pmin), right = __float_as_uint(pmax) + 1u;
    unsigned cnt = static_cast<unsigned>(V);
    float mass = 1.0f;
    unsigned cnt_right = 0;  // count and mass of the entries at or above `right`
    float mass_right = 0.0f;
    auto go_on = [&] { return (cnt > static_cast<unsigned>(a.top_k) || mass > a.top_p) && left < right - 1u; };
    auto step = [&](unsigned mid, unsigned c, float m) {
      if (c < static_cast<unsigned>(a.top_k) && m < a.top_p) {
        right = mid;
        cnt_right = c;
        mass_right = m;
      } else {
        left = mid;
        cnt = c;
        mass = m;
      }
    };
    // Row in registers: a step over the whole row is a block exchange and up to 64 comparisons per thread, and about 30 of
    // them find the threshold.  Once no more than kBracket entries lie between the ends these alone go through the rest,
    // every wavefront for itself, without a barrier; 512 instead of 256 measured the same.  us per call, rows of 65536 logits
    // ~ N(0, 9), whole-row steps only / this: top-p 0.9 1 row 98 / 67, 64 rows 104 / 70; top-p 0.6 94 / 61, 97 / 63; top-k
    // 400 and top-p 0.8 61 / 56, 76 / 60.  The picks of 30000 compared draws are the same.
    while (go_on() && !(REG && cnt - cnt_right <= static_cast<unsigned>(kBracket))) {
      const unsigned mid = left + (right - left) / 2u;
      const float thr = __uint_as_float(mid);
      unsigned c = 0;
      float m = 0.0f;
      if constexpr (REG) {
        // (probabilities are not negative: their order is the order of their bit patterns, which the bisection
        // itself relies on; the comparison of two wavefront-wide values is a scalar one)
        const unsigned mid_u = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(mid)));
#pragma unroll
        for (int q = 0; q < kSampleRegVecs; ++q) {
          if (slot_max[q] >= mid_u) {
            if (q < n) {
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (vals[q][j] >= thr) {
                  ++c;
                  m += vals[q][j];
                }
            }
          }
        }
      } else {
        for_each([&](int q, int i) {
          const float4_t l = get(q, i);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (l[j] >= thr) {
              ++c;
              m += l[j];
            }
        });
      }
      block_count_mass(c, m, red);
      step(mid, c, m);
    }
    if constexpr (REG) {
      if (go_on()) {  // (the same in every thread)
        const float lo = __uint_as_float(left), hi = __uint_as_float(right);
        const unsigned left_u = static_cast<unsigned>(__builtin_amdgcn_readfirstlane(static_cast<int>(left)));
        int mine = 0;
#pragma unroll
        for (int q = 0; q < kSampleRegVecs; ++q)
          if (slot_max[q] >= left_u && q < n)
#pragma unroll
            for (int j = 0; j < 4; ++j) mine += vals[q][j] >= lo && vals[q][j] < hi ? 1 : 0;
        // (at most kBracket of them: whole numbers, exact in fp32; thread order, so that the sums below repeat)
        float total;
        int at = static_cast<int>(block_exclusive_scan(static_cast<float>(mine), red.f, &total));
        const int inside = min(static_cast<int>(total), kBracket);
        if (mine > 0) {
#pragma unroll
          for (int q = 0; q < kSampleRegVecs; ++q)
            if (q < n)
#pragma unroll
              for (int j = 0; j < 4; ++j)
                if (vals[q][j] >= lo && vals[q][j] < hi && at < kBracket) red.bracket[at++] = vals[q][j];
        }
        __syncthreads();
        constexpr int kRounds = kBracket / 64;
        float e[kRounds];
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
          const int i = r * 64 + (t & 63);
          e[r] = i < inside ? red.bracket[i] : -1.0f;  // past the end: below every threshold
        }
        // every wavefront for itself, all with the same sums
        const unsigned cnt_above = cnt_right;
        const float mass_above = mass_right;
        while (go_on()) {
          const unsigned mid = left + (right - left) / 2u;
          const float thr = __uint_as_float(mid);
          unsigned c = 0;
          float m = 0.0f;
#pragma unroll
          for (int r = 0; r < kRounds; ++r) {
            c += static_cast<unsigned>(__popcll(__ballot(e[r] >= thr)));
            m += e[r] >= thr ? e[r] : 0.0f;
          }
          step(mid, cnt_above + c, mass_above + wave_reduce_dpp(m, fadd_op));
        }
      }
    }
    const float thr = __uint_as_float(left);

    // 5. tie compensation
    unsigned eqk = 0, gtk = 0;
    float gtp = 0.0f;
    for_each([&](int q, int i) {
      const float4_t l = get(q, i);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (l[j] == thr) ++eqk;
        if (l[j] > thr) {
          ++gtk;
          gtp += l[j];
        }
      }
    });
    const unsigned n_eq = block_sum_u(eqk, red.u);
    const unsigned n_gt = block_sum_u(gtk, red.u);
    const float p_gt = block_reduce_f(gtp, fadd_op, red.f);
    float comp = 1.0f;
    if (n_eq > 0) comp = tie_share(a, thr, n_eq, n_gt, p_gt);

    // 6. inverse-CDF draw over the kept set, thread by thread
    const float mine = gtp + (thr * eqk) * comp;
    float total;
    const float before = block_exclusive_scan(mine, red.f, &total);
    const float target = uniform_of_row(a, b) * total;
    if (t == 0) s_pick = -1;
    __syncthreads();
    if (mine > 0.0f && target > before && target <= before + mine) {
      float cum = before;
      int found = -1, last = -1;
      for_each([&](int q, int i) {
        const float4_t l = get(q, i);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float w = (l[j] < thr) ? 0.0f : (l[j] == thr ? l[j] * comp : l[j]);
          if (w > 0.0f && found < 0) {
            cum += w;
            last = i * 4 + j;
            if (cum >= target) found = last;
          }
        }
      });
      if (found < 0) found = last;  // rounding inside the slice: its last kept entry
      atomicMax(&s_pick, found);
    }
    __syncthreads();
    const bool fallback = s_pick < 0;  // rounding between slices left the target past every interval
    __syncthreads();
    if (fallback && mine > 0.0f) {
      int last = -1;
      for_each([&](int q, int i) {
        const float4_t l = get(q, i);
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (l[j] > thr || (l[j] == thr && comp > 0.0f)) last = i * 4 + j;
      });
      atomicMax(&s_pick, last);
    }
    __syncthreads();
    pick = s_pick < 0 ? 0 : s_pick;
  }

  return pick;
}

// 7. penalty update (sampling.cu:461-470) of one float4 of the row
__device__ __forceinline__ float4_t decayed_penalty(float4_t p, int i, int pick, const SampleArgs& a) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float add = (pick != i * 4 + j) ? 0.0f : (p[j] == 0.0f ? a.presence : a.frequency);
    p[j] = fmaf(p[j], a.decay, add);
  }
  return p;
}

template <bool REG>
__global__ __launch_bounds__(kSampleThreads) void sample_kernel(SampleArgs a) {
  __shared__ BlockRed red;
  __shared__ int s_pick;
  const int b = blockIdx.x;
  const int pick = sample_row<REG>(a, b, red, s_pick);
  if (threadIdx.x == 0) a.out[b] = pick;
  if (!a.penalties) return;
  float4_t* pen = reinterpret_cast<float4_t*>(a.penalties + static_cast<int64_t>(b) * a.V);
  // (rows in registers: one piece at a time, so that the first store does not wait for a second load.  us, 1 / 64 rows of 65536
  // without filters, 1 / 2 / 4 / 16 pieces: 34.8 / 35.0 / 35.3 / 35.7 and 37.7 / 38.1 / 38.2 / 38.5)
#pragma unroll(REG ? 1 : 4)
  for (int i = threadIdx.x; i < a.V / 4; i += kSampleThreads) pen[i] = decayed_penalty(pen[i], i, pick, a);
}

// ---- top-k rows in three launches ------------------------------------------------------------------------------------
// One block per row has one CU to move the row through and to do its arithmetic on (0.4 us per VALU operation and row of
// 65536 entries), and at 64 rows three quarters of the chip idle.  With a top_k of at most kSplitMaxTopK the kept set is known to
// lie among a few hundred entries before any probability is:
//   sample_stats_kernel  the whole chip reads the rows: per 64 entries (a slot) the largest penalised logit, per 4096 entries
//                        their maximum and the sum of their exponentials below it;
//   sample_pick_kernel   one block per row: a value that at least top_k slot maxima reach bounds the top_k-th largest entry from
//                        below, so only those slots (top_k and a few) are read again, and of them only the entries above it
//                        compete: softmax, threshold, ties and draw of sample_row over these, in the order sample_row walks the
//                        row in (13.3 of the 23.5 us of 64 rows of 65536, top-k 50, top-p 0.6; 20.8 with sample_row's bisection).  A row with more than kMaxCandidates of them (equal logits) goes through sample_row itself;
//   sample_decay_kernel  the penalty rows, by the whole chip again.
// Against the one-block kernel the sum of the exponentials and the masses are added in another order (fp32 both), no more.
// Rows of 65536, penalties, top-k 50, top-p 0.6, one block per row / this: 1 row 53.4 / 17.6 us, 64 rows 66-70 / 23.7,
// 128 rows 70.9 / 36.3; 8 rows, top-k 200, top-p 0.8: 64.5 / 24.1.  The same rows masked down to 20 entries: 64 rows 75.1 /
// 20.4.  Rows of equal logits, which pay for the launches on top of sample_row, lose: 1 row 87 / 95, 256 rows 112 / 143.
// The slot maxima and the parts' sums lie in `probs`.
constexpr int kSlot = 64;
constexpr int kPartEntries = 4096;
constexpr int kPartThreads = 256;
constexpr int kSplitMaxTopK = 256;
constexpr int kMaxCandidates = 1024;  // one per thread
constexpr int kFewCandidates = 128;   // up to here the threshold is searched among the candidates in order of value
constexpr int kMaxSlots = kSampleRegVecs * kSampleThreads * 4 / kSlot;
static_assert(kMaxSlots == kSampleThreads, "one slot per thread, sixteen per lane of a wavefront");

// top_k slot maxima have to bound the kept set well (twice as many slots), one block has to hold a row's slots, and the greedy
// pick of top_k == 1 compares logits, not probabilities.
inline bool sample_split_ok(int V, int top_k) {
  return top_k >= 2 && top_k <= kSplitMaxTopK && V <= kMaxSlots * kSlot && V / kSlot >= 2 * top_k;
}

__global__ __launch_bounds__(kPartThreads) void sample_stats_kernel(SampleArgs a) {
  constexpr int kVecs = kPartEntries / 4 / kPartThreads;
  __shared__ float red[kPartThreads / 64];
  const int b = blockIdx.x;
  const int part = blockIdx.y, parts = gridDim.y;
  const int t = threadIdx.x;
  const int V4 = a.V / 4;
  const int n_slots = (a.V + kSlot - 1) / kSlot;
  const float4_t* logits = reinterpret_cast<const float4_t*>(a.logits + static_cast<int64_t>(b) * a.V);
  const float4_t* pen = a.penalties ? reinterpret_cast<const float4_t*>(a.penalties + static_cast<int64_t>(b) * a.V) : nullptr;
  float* stats = a.probs + static_cast<int64_t>(b) * a.V;
  float4_t l[kVecs], p[kVecs];
#pragma unroll
  for (int q = 0; q < kVecs; ++q) l[q] = logits[min(part * (kPartEntries / 4) + q * kPartThreads + t, V4 - 1)];
#pragma unroll
  for (int q = 0; q < kVecs; ++q) p[q] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  if (pen) {
#pragma unroll
    for (int q = 0; q < kVecs; ++q) p[q] = pen[min(part * (kPartEntries / 4) + q * kPartThreads + t, V4 - 1)];
  }
  auto fmax_op = [](float x, float y) { return fmaxf(x, y); };
  float top = -INFINITY;
#pragma unroll
  for (int q = 0; q < kVecs; ++q) {
    const bool live = part * (kPartEntries / 4) + q * kPartThreads + t < V4;
#pragma unroll
    for (int j = 0; j < 4; ++j) l[q][j] = live ? penalised(l[q][j], p[q][j], a.log2_inv_temp) : -INFINITY;
    float m = fmaxf(fmaxf(l[q][0], l[q][1]), fmaxf(l[q][2], l[q][3]));
    m = fmaxf(m, __builtin_bit_cast(float, lane_xor_dpp<8>(__builtin_bit_cast(int, m))));
    m = fmaxf(m, __builtin_bit_cast(float, lane_xor_dpp<4>(__builtin_bit_cast(int, m))));
    m = fmaxf(m, __builtin_bit_cast(float, lane_xor_dpp<2>(__builtin_bit_cast(int, m))));
    m = fmaxf(m, __builtin_bit_cast(float, lane_xor_dpp<1>(__builtin_bit_cast(int, m))));
    const int slot = part * (kPartEntries / kSlot) + (q * kPartThreads + t) / 16;
    if ((t & 15) == 0 && slot < n_slots) stats[slot] = m;
    top = fmaxf(top, m);
  }
  top = wave_reduce_dpp(top, fmax_op);
  if ((t & 63) == 0) red[t >> 6] = top;
  __syncthreads();
  top = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float sum = 0.0f;
#pragma unroll
  for (int q = 0; q < kVecs; ++q)
    sum += (exp2f(l[q][0] - top) + exp2f(l[q][1] - top)) + (exp2f(l[q][2] - top) + exp2f(l[q][3] - top));
  sum = wave_reduce_dpp(sum, [](float x, float y) { return x + y; });
  __syncthreads();
  if ((t & 63) == 0) red[t >> 6] = sum;
  __syncthreads();
  if (t == 0) {
    stats[n_slots + part] = top;
    stats[n_slots + parts + part] = (red[0] + red[1]) + (red[2] + red[3]);
  }
}
static_assert(kPartThreads == 256, "sample_stats_kernel adds up four wavefronts");

// order of finite floats as unsigned integers, and back
__device__ __forceinline__ unsigned order_key(float x) {
  const unsigned u = __float_as_uint(x);
  return static_cast<int>(u) < 0 ? ~u : u | 0x80000000u;
}
__device__ __forceinline__ float from_order_key(unsigned k) {
  return __uint_as_float(static_cast<int>(k) < 0 ? k & 0x7fffffffu : ~k);
}

__global__ __launch_bounds__(kSampleThreads) void sample_pick_kernel(SampleArgs a, int parts) {
  __shared__ BlockRed red;
  __shared__ int s_pick;
  __shared__ __align__(16) unsigned counts[2][kSampleWaves];
  __shared__ int slots[kMaxSlots];
  __shared__ int n_cand;
  __shared__ __align__(16) unsigned cand_at[kMaxCandidates];
  __shared__ __align__(16) float cand[kMaxCandidates];
  __shared__ unsigned sorted_at[kMaxCandidates];
  __shared__ float sorted[kMaxCandidates], by_value[kFewCandidates];
  const int b = blockIdx.x;
  const int t = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int lane = t & 63;
  const int V4 = a.V / 4;
  const int n_slots = (a.V + kSlot - 1) / kSlot;
  const unsigned top_k = static_cast<unsigned>(a.top_k);
  const float* stats = a.probs + static_cast<int64_t>(b) * a.V;
  auto fmax_op = [](float x, float y) { return fmaxf(x, y); };
  auto fmin_op = [](float x, float y) { return fminf(x, y); };
  auto fadd_op = [](float x, float y) { return x + y; };
  auto umin_op = [](unsigned x, unsigned y) { return min(x, y); };

  // every wavefront: the parts, and all slot maxima (sixteen per lane)
  const int part = min(lane, parts - 1);
  const float part_max = stats[n_slots + part];
  const float part_sum = lane < parts ? stats[n_slots + parts + part] : 0.0f;
  unsigned key[kMaxSlots / 64];
#pragma unroll
  for (int i = 0; i < kMaxSlots / 64; ++i) key[i] = order_key(stats[min(i * 64 + lane, n_slots - 1)]);
  const float my_slot_max = stats[min(t, n_slots - 1)];
  const float gmax = wave_reduce_dpp(part_max, fmax_op);
  const float den = wave_reduce_dpp(part_sum * exp2f(part_max - gmax), fadd_op);

  // a value that at least top_k slot maxima reach, and hardly more: sixteen thresholds at a time, one per wavefront
  unsigned low_key = 0xffffffffu;
#pragma unroll
  for (int i = 0; i < kMaxSlots / 64; ++i) {
    low_key = min(low_key, key[i]);
    if (i * 64 + lane >= n_slots) key[i] = 0;  // (below every threshold; a lane past the end repeated the last slot)
  }
  unsigned lo = wave_reduce_dpp(low_key, umin_op);
  unsigned hi = order_key(gmax) + 1u;
  unsigned reach = static_cast<unsigned>(n_slots);  // maxima at or above lo
  const unsigned enough = top_k + max(top_k / 4u, 16u);
  // Entries 150 octaves below the maximum have probability zero: they never carry weight.  Where fewer than top_k slots reach
  // higher than that - a row masked down to a few entries - there is nothing to search for, and the zeros need not compete one
  // by one; that they are there the threshold search below has to know: it then starts at zero with a count above any top_k.
  const float zero_u = gmax - 150.0f;
  const unsigned zero_key = order_key(zero_u);
  if (lo < zero_key) {
    unsigned c = 0;
#pragma unroll
    for (int i = 0; i < kMaxSlots / 64; ++i) c += static_cast<unsigned>(__popcll(__ballot(key[i] >= zero_key)));
    reach = c;
    if (c >= top_k) lo = zero_key;
  }
  for (int it = 0; reach > enough && hi - lo > 1u; it ^= 1) {
    const unsigned apart = max((hi - lo) / 17u, 1u);
    auto threshold = [&](int w) { return lo + apart * (w + 1); };
    const unsigned mine = threshold(wave);
    unsigned c = 0;
#pragma unroll
    for (int i = 0; i < kMaxSlots / 64; ++i) c += static_cast<unsigned>(__popcll(__ballot(key[i] >= mine)));
    if (lane == 0) counts[it][wave] = c;
    __syncthreads();
    // (counts fall from one threshold to the next: the first `held` of them are held by top_k maxima)
    const unsigned cw = counts[it][lane & (kSampleWaves - 1)];
    const int held = __popcll(__ballot(lane < kSampleWaves && cw >= top_k));
    const unsigned below = lo;
    if (held > 0) {
      lo = threshold(held - 1);
      reach = static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(cw), held - 1));
    }
    if (held < kSampleWaves) hi = min(hi, below + apart * (held + 1));
  }
  // (two logits this close may round to the same probability, and entries of one probability share its fate)
  const float bound_u = from_order_key(lo) - 4e-6f;
  const bool zeros_below = bound_u < zero_u;
  const float floor_u = fmaxf(bound_u, zero_u);

  // the slots that reach it, then their entries that do
  if (t == 0) n_cand = 0;
  cand_at[t] = 0xffffffffu;  // past the last candidate: behind every position, below every value
  cand[t] = -INFINITY;
  const bool chosen = t < n_slots && my_slot_max >= floor_u;
  const uint64_t mask = __ballot(chosen);
  if (lane == 0) red.u[wave] = static_cast<unsigned>(__popcll(mask));
  __syncthreads();
  int first = 0, n_chosen = 0;
#pragma unroll
  for (int w = 0; w < kSampleWaves; ++w) {
    if (w < wave) first += static_cast<int>(red.u[w]);
    n_chosen += static_cast<int>(red.u[w]);
  }
  if (chosen) slots[first + __popcll(mask & ((1ull << lane) - 1ull))] = t;
  __syncthreads();
  const float4_t* logits = reinterpret_cast<const float4_t*>(a.logits + static_cast<int64_t>(b) * a.V);
  const float4_t* pen = a.penalties ? reinterpret_cast<const float4_t*>(a.penalties + static_cast<int64_t>(b) * a.V) : nullptr;
  for (int s = t >> 4; s < n_chosen; s += kSampleThreads / 16) {
    // (more candidates than fit: the row goes another way, whatever the rest of them is)
    if (s >= kSampleThreads / 16 && *static_cast<volatile int*>(&n_cand) > kMaxCandidates) break;
    const int i = slots[s] * (kSlot / 4) + (t & 15);
    if (i >= V4) continue;
    const float4_t l = logits[i];
    float4_t p = {0.0f, 0.0f, 0.0f, 0.0f};
    if (pen) p = pen[i];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float u = penalised(l[j], p[j], a.log2_inv_temp);
      if (u >= floor_u) {
        const int at = atomicAdd(&n_cand, 1);
        if (at < kMaxCandidates) {
          cand[at] = u;
          // where sample_row's draw meets the entry: thread i % 1024, its slice's float4 i / 1024, element j
          cand_at[at] = static_cast<unsigned>(((i % kSampleThreads) * kSampleRegVecs + i / kSampleThreads) * 4 + j);
        }
      }
    }
  }
  __syncthreads();
  const int n = n_cand;
  int pick = 0;
  if (n > kMaxCandidates) {
    pick = sample_row<true>(a, b, red, s_pick);
  } else {
    auto rank_candidates = [&](auto few_c) {
      constexpr bool kFew = decltype(few_c)::value;
      const unsigned at = cand_at[t];
      const float u = cand[t];
      int rank = 0, larger = 0;
      // sixteen at a time: the reads of a trip are in flight together (one by one they took 2.1 us for 55 candidates)
      for (int i0 = 0; i0 < n; i0 += 16) {
        uint4_t where[4];
        float4_t value[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          where[q] = *reinterpret_cast<const uint4_t*>(&cand_at[i0 + 4 * q]);
          if constexpr (kFew) value[q] = *reinterpret_cast<const float4_t*>(&cand[i0 + 4 * q]);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          rank += where[i / 4][i % 4] < at ? 1 : 0;
          if constexpr (kFew) {
            const float x = value[i / 4][i % 4];
            larger += x > u || (x == u && i0 + i < t) ? 1 : 0;
          }
        }
      }
      const float prob = exp2f(u - gmax) / den;
      sorted_at[rank] = at;
      sorted[rank] = prob;
      if constexpr (kFew) by_value[larger] = prob;  // (not increasing: the exponential is monotone)
    };
    if (t < n) {
      if (n <= kFewCandidates) rank_candidates(std::true_type{});
      else rank_candidates(std::false_type{});
    }
    __syncthreads();
    if (wave != 0) return;
    // one wavefront, up to two or up to sixteen entries per lane: steps 4 to 6 of sample_row without a barrier
    auto draw = [&](auto rounds_c) {
      constexpr int kRounds = decltype(rounds_c)::value;
      const int rounds = (n + 63) / 64;
      constexpr bool kFew = kRounds * 64 <= kFewCandidates;
      float p[kRounds];
      float pmin = INFINITY, pmax = -INFINITY, mass = 0.0f;
#pragma unroll
      for (int r = 0; r < kRounds; ++r) {
        p[r] = -1.0f;  // past the end: below every threshold
        if (r < rounds && r * 64 + lane < n) {
          p[r] = sorted[r * 64 + lane];
          pmin = fminf(pmin, p[r]);
          if constexpr (!kFew) pmax = fmaxf(pmax, p[r]);
          mass += p[r];
        }
      }
      pmin = wave_reduce_dpp(pmin, fmin_op);
      if constexpr (!kFew) pmax = wave_reduce_dpp(pmax, fmax_op);
      mass = wave_reduce_dpp(mass, fadd_op);
      unsigned cnt = zeros_below ? static_cast<unsigned>(V4) * 4u : static_cast<unsigned>(n);
      // entries at or above v, and their mass
      auto reach_of = [&](float v, unsigned& c, float& m) {
        c = 0;
        m = 0.0f;
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
          if (r < rounds) {
            c += static_cast<unsigned>(__popcll(__ballot(p[r] >= v)));
            m += p[r] >= v ? p[r] : 0.0f;
          }
        }
        m = wave_reduce_dpp(m, fadd_op);
      };
      // The threshold of sample_row's bisection is the largest value that still leaves top_k entries or top_p mass at or above it,
      // and that changes only at an entry: instead of some 25 halvings of the bit pattern (0.3 us each; a row that needs them all
      // held up the launch) the entries in order of value are halved, 6 or 7 times for 50 to 100 of them, with the same sums at each.
      // More candidates keep sample_row's bisection: ranking them by value, whose pairs grow with their square, costs more than it
      // saves (us, 64 rows of 65536, ranked / bisected: 125 to 160 candidates of rows as flat as N(0, 9) 30.2 / 27.5, of N(0, 100) 30.0 /
      // 31.7; top_k 200, top_p 0.8 41.4 / 31.9; top_k 256 48.4 / 32.3).
      float thr = zeros_below ? 0.0f : pmin;
      bool fits = false;  // the kept set has top_k entries or top_p mass as it is
      if constexpr (kFew) {
        if (cnt > top_k || mass > a.top_p) {
          int low = 0, high = n;  // entries from `high` on leave enough, those before `low` do not
          while (low < high) {
            const int mid = (low + high) / 2;
            unsigned c;
            float m;
            reach_of(by_value[mid], c, m);
            if (c < top_k && m < a.top_p) {
              low = mid + 1;
            } else {
              high = mid;
              cnt = c;
              mass = m;
            }
          }
          if (high < n) thr = by_value[high];
          fits = cnt <= top_k && mass <= a.top_p;
        }
      } else {
        unsigned left = __float_as_uint(thr), right = __float_as_uint(pmax) + 1u;
        while ((cnt > top_k || mass > a.top_p) && left < right - 1u) {
          const unsigned mid = left + (right - left) / 2u;
          unsigned c;
          float m;
          reach_of(__uint_as_float(mid), c, m);
          if (c < top_k && m < a.top_p) {
            right = mid;
          } else {
            left = mid;
            cnt = c;
            mass = m;
          }
        }
        thr = __uint_as_float(left);
      }
      unsigned n_eq = 0, n_gt = 0;
      float p_gt = 0.0f;
#pragma unroll
      for (int r = 0; r < kRounds; ++r) {
        if (r < rounds) {
          n_eq += static_cast<unsigned>(__popcll(__ballot(p[r] == thr)));
          n_gt += static_cast<unsigned>(__popcll(__ballot(p[r] > thr)));
          p_gt += p[r] > thr ? p[r] : 0.0f;
        }
      }
      p_gt = wave_reduce_dpp(p_gt, fadd_op);
      float comp = 1.0f;
      if (n_eq > 0 && !fits) comp = tie_share(a, thr, n_eq, n_gt, p_gt);
      // running sums of the kept weights in the draw's order, then the first that reaches the target
      float total = 0.0f;
      float cum[kRounds];
#pragma unroll
      for (int r = 0; r < kRounds; ++r) {
        cum[r] = 0.0f;
        if (r < rounds) {
          p[r] = p[r] < thr ? 0.0f : (p[r] == thr ? p[r] * comp : p[r]);
          float inc = p[r];
#pragma unroll
          for (int off = 1; off < 64; off <<= 1) {
            const float below = __shfl_up(inc, off, 64);
            if (lane >= off) inc += below;
          }
          cum[r] = total + inc;
          total = __shfl(cum[r], 63, 64);
        }
      }
      const float target = uniform_of_row(a, b) * total;
      int found = -1, last = -1;
#pragma unroll
      for (int r = 0; r < kRounds; ++r) {
        if (r < rounds) {
          const uint64_t kept = __ballot(p[r] > 0.0f);
          const uint64_t hit = __ballot(p[r] > 0.0f && cum[r] >= target);
          if (hit != 0 && found < 0) found = r * 64 + __ffsll(static_cast<unsigned long long>(hit)) - 1;
          if (kept != 0) last = r * 64 + 63 - __clzll(static_cast<long long>(kept));
        }
      }
      if (found < 0) found = last;  // rounding left the target past the last sum
      if (found >= 0) {
        const unsigned at = sorted_at[found];
        const int i = static_cast<int>((at >> 2) % kSampleRegVecs) * kSampleThreads + static_cast<int>(at >> 2) / kSampleRegVecs;
        pick = i * 4 + static_cast<int>(at & 3u);
      }
    };
    if (n <= kFewCandidates) draw(std::integral_constant<int, kFewCandidates / 64>{});
    else draw(std::integral_constant<int, kMaxCandidates / 64>{});
  }
  if (t == 0) a.out[b] = pick;
}

__global__ __launch_bounds__(kPartThreads) void sample_decay_kernel(SampleArgs a) {
  constexpr int kVecs = kPartEntries / 4 / kPartThreads;
  const int b = blockIdx.x;
  const int first = blockIdx.y * (kPartEntries / 4) + threadIdx.x;
  const int V4 = a.V / 4;
  float4_t* pen = reinterpret_cast<float4_t*>(a.penalties + static_cast<int64_t>(b) * a.V);
  const int pick = a.out[b];
  float4_t p[kVecs];
#pragma unroll
  for (int q = 0; q < kVecs; ++q) p[q] = pen[min(first + q * kPartThreads, V4 - 1)];
#pragma unroll
  for (int q = 0; q < kVecs; ++q) {
    const int i = first + q * kPartThreads;
    if (i < V4) pen[i] = decayed_penalty(p[q], i, pick, a);
  }
}

// One 1024-thread block per row; 16-byte loads, eight in flight per thread (the row is 256 KiB at V = 65536 and
// the kernel is pure load latency).  Lowest index among equal maxima.
constexpr int kArgmaxThreads = 1024;

// next / history (may be null): the picked id also becomes the row's next input token and an entry of the caller's
// list of generated tokens - what a greedy decode loop would otherwise launch a second kernel for.
__global__ __launch_bounds__(kArgmaxThreads) void argmax_kernel(int V, const float* __restrict__ logits, int* __restrict__ out,
                                                               int64_t* __restrict__ next, int* __restrict__ history) {
  __shared__ float bv[kArgmaxThreads / 64];
  __shared__ int bi[kArgmaxThreads / 64];
  const float* row = logits + static_cast<int64_t>(blockIdx.x) * V;
  float best = -INFINITY;
  int idx = 0x7fffffff;
  auto take = [&](float v, int i) {
    if (v > best || (v == best && i < idx)) {
      best = v;
      idx = i;
    }
  };
  const bool vec_ok = (reinterpret_cast<uintptr_t>(row) & 15) == 0;
  const int V4 = vec_ok ? V / 4 : 0;
  constexpr int kBatch = 8;
  for (int base = 0; base < V4; base += kArgmaxThreads * kBatch) {
    float4_t q[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int i = base + u * kArgmaxThreads + threadIdx.x;
      q[u] = float4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
      if (i < V4) q[u] = reinterpret_cast<const float4_t*>(row)[i];
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int i = (base + u * kArgmaxThreads + threadIdx.x) * 4;
      if (i < V4 * 4) {
        take(q[u].x, i);
        take(q[u].y, i + 1);
        take(q[u].z, i + 2);
        take(q[u].w, i + 3);
      }
    }
  }
  for (int i = V4 * 4 + threadIdx.x; i < V; i += kArgmaxThreads) take(row[i], i);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(best, off, 64);
    const int oi = __shfl_xor(idx, off, 64);
    if (ov > best || (ov == best && oi < idx)) {
      best = ov;
      idx = oi;
    }
  }
  if ((threadIdx.x & 63) == 0) {
    bv[threadIdx.x >> 6] = best;
    bi[threadIdx.x >> 6] = idx;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int i = 1; i < kArgmaxThreads / 64; ++i)
      if (bv[i] > best || (bv[i] == best && bi[i] < idx)) {
        best = bv[i];
        idx = bi[i];
      }
    const int pick = idx == 0x7fffffff ? 0 : idx;
    out[blockIdx.x] = pick;
    if (next) next[blockIdx.x] = pick;
    if (history) history[blockIdx.x] = pick;
  }
}

int argmax_launch(hipStream_t st, int B, int V, const float* logits, int* out, int64_t* next, int* history) {
  hipLaunchKernelGGL(argmax_kernel, dim3(B), dim3(kArgmaxThreads), 0, st, V, logits, out, next, history);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

}  // namespace rwkv

using namespace rwkv;

extern "C" {

int rwkv_hip_sample(rwkv_stream_t s, int B, int V, const void* logits, void* penalties, void* probs, void* out,
                    double presence, double frequency, double decay, double temperature, int top_k, double top_p,
                    uint64_t seed, uint64_t step) {
  // same argument checks as the reference (src/utils/sampling.cu:492-512)
  RWKV_REQUIRE(V > 0 && V <= 1048576 && V % 4 == 0,
               "Vocabulary size must be multiple of 4, and no larger than 1048576, got %d", V);
  RWKV_REQUIRE(B > 0, "B must be positive, got %d", B);
  RWKV_REQUIRE(temperature >= 0.001 && temperature <= 1000.0, "Temperature outside range, got %f", temperature);
  RWKV_REQUIRE(logits && probs && out, "sample: NULL tensor");
  if (top_k <= 0 || top_k > V) top_k = V;
  if (top_p < 0 || top_p > 1) top_p = 1;
  if (top_p == 0) {
    top_k = 1;
    top_p = 1;
  }
  SampleArgs a;
  a.logits = static_cast<const float*>(logits);
  a.penalties = static_cast<float*>(penalties);
  a.probs = static_cast<float*>(probs);
  a.out = static_cast<int*>(out);
  a.V = V;
  a.presence = static_cast<float>(presence);
  a.frequency = static_cast<float>(frequency);
  a.decay = static_cast<float>(decay);
  a.log2_inv_temp = static_cast<float>(1.44269504088896340736 / temperature);
  a.top_k = top_k;
  a.top_p = static_cast<float>(top_p);
  a.seed = seed;
  a.step = step;
  // The three launches keep their sums in `probs` while the logits and penalties are still being read and other rows' picks are
  // written.  The one-block kernel does not touch the scratch of a row it holds in registers: a caller whose scratch reaches
  // into one of these stays there.
  const int64_t row_bytes = static_cast<int64_t>(B) * V * 4;
  const auto apart = [&](const void* other, int64_t bytes) {
    const char* p = static_cast<const char*>(probs);
    const char* q = static_cast<const char*>(other);
    return !other || p + row_bytes <= q || q + bytes <= p;
  };
  if (sample_split_ok(V, top_k) && apart(logits, row_bytes) && apart(penalties, row_bytes) && apart(out, static_cast<int64_t>(B) * 4)) {
    const int parts = ceil_div(V, kPartEntries);
    hipLaunchKernelGGL(sample_stats_kernel, dim3(B, parts), dim3(kPartThreads), 0, as_stream(s), a);
    hipLaunchKernelGGL(sample_pick_kernel, dim3(B), dim3(kSampleThreads), 0, as_stream(s), a, parts);
    if (penalties) hipLaunchKernelGGL(sample_decay_kernel, dim3(B, parts), dim3(kPartThreads), 0, as_stream(s), a);
  } else if (V / 4 <= kSampleRegVecs * kSampleThreads) {
    hipLaunchKernelGGL(sample_kernel<true>, dim3(B), dim3(kSampleThreads), 0, as_stream(s), a);
  } else {
    hipLaunchKernelGGL(sample_kernel<false>, dim3(B), dim3(kSampleThreads), 0, as_stream(s), a);
  }
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int rwkv_hip_argmax(rwkv_stream_t s, int B, int V, const void* logits, void* out) {
  RWKV_REQUIRE(B > 0 && V > 0 && logits && out, "argmax: bad arguments");
  return argmax_launch(as_stream(s), B, V, static_cast<const float*>(logits), static_cast<int*>(out));
}

}  // extern "C"
