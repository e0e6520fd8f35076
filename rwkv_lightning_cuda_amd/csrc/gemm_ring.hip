// Packed-weight MFMA GEMM for batched decode and prefill chunks (up to some hundred rows; any number of rows of int4 codes):
// X through a ring of LDS stages that feeder wavefronts fill with direct-to-LDS loads, weights through registers.
//
// Reference: as gemm_stream.hip (cuda/rwkv7_v3a_ops.cu:2235-2368).
//
// What bounds it.  256 CUs that stream the weights once take 12.8 us for 67 MB (6.5 TB/s and 2 us of launch); every block also
// needs its rows of X, out of L2, and the two add up: 15.4 us with 64 rows of X per CU (512 KB), 19.3 with 128, whatever
// the number of loads in flight.  So a block (a) reads every weight byte once - up to 64 rows no two blocks share weights -
// and (b) has no other traffic: 12 wavefronts, one block per CU (two of the tiles of 32 rows and 128 k, 64 KB of LDS each).
//   * Four feeders only move X: 16-byte direct-to-LDS loads (no registers, no ds_write), seven stages ahead - three where a
//     stage is 32 KB - waits by count.  A separate wavefront counts X alone: in the wavefronts that also load weights, loads return in order and every
//     wait for X (L2) would be one for older weights (HBM).
//   * Eight workers multiply.  A worker owns NB bands of 32 columns and 1 / KG of each stage's k; its weights come as whole
//     1 KiB pieces, non-temporally, one to three stages ahead (what the registers hold).  KG groups of workers share the k of a stage, so that 64 columns still
//     occupy eight wavefronts; their sums meet in LDS once, at the end, in group order.
//   * One barrier per stage for all twelve, placed before the last MFMA step, whose fragments are in registers by then: the
//     first fragments of the next stage are read under that step's products.
// LDS rows are 256 or 512 bytes apart with the 16-byte pieces of row r permuted by r & 15, so that the 32 rows a fragment
// read touches hit different banks; a direct-to-LDS load writes lane after lane, so the permutation is in the addresses it
// reads from.
//
// Measured (us per launch, back to back on weights that are not in any cache, this / the register-staged tiles before it):
//   int8, 16384 x 4096:  17 rows 14.9 / 19.9, 64 rows 21.0 / 24.3, 128 rows 26.4 / 30.8, 256 rows 41.9 / 47.6
//   int8, 12288 x 4096:  64 rows 18.6 / 28.2, 128 rows 23.7 / 35.4      int8, 4096 x 4096: 64 rows 11.2 / 14.4, 128 rows 11.5 / 17.1
//   int8, 4096 x 16384 (K split, reduce launch included): 64 rows 24.8 / 28.0, 128 rows 32.9 / 39.6
//   fp16, 16384 x 4096:  64 rows 27.4 / 35.1, 256 rows 45.0 / 54.3      int4, 16384 x 4096: 64 rows 20.6 / 24.0, 2048 rows 335 / 429
// Wavefront timestamps of the 64-row launch (21 us): 2.1 us between launches, 1.2 to the first weight request, 1.8 until the
// first stage of X has arrived, 13.4 of streaming (the 67 MB alone: 10.3), 1.7 for the groups' sums and the stores.
#include "gemm_stream.h"

namespace rwkv {

namespace {

constexpr int kRingFeeders = 4;     // wavefronts that load X
constexpr int kRingWorkers = 8;     // wavefronts that multiply
constexpr int kRingThreads = 64 * (kRingFeeders + kRingWorkers);

// A block: 32 * MT rows, WP * NB bands of 32 columns (NB per worker), KC k per stage shared out between KG workers.
template <int MT, int NB, int WP, int KC>
struct RingTile {
  static constexpr int BM = 32 * MT, BN = 32 * NB * WP;
  static constexpr int KG = kRingWorkers / WP;
  static constexpr int KW = KC / KG;           // k per worker and stage
  static constexpr int kRowBytes = KC * 2;
  static constexpr int kStageBytes = BM * kRowBytes;
  static constexpr int kStages = kStageBytes >= 32768 ? 4 : 8;
  static constexpr int kRedLd = BN + 4;
  static constexpr int kRedBytes = KG * BM * kRedLd * 4;
  static constexpr int kLdsBytes = kStages * kStageBytes > kRedBytes ? kStages * kStageBytes : kRedBytes;
  static constexpr int kLoads = kStageBytes / 1024 / kRingFeeders;  // direct-to-LDS loads per feeder and stage
  static_assert(KW == 32 || KW == 64, "a worker takes one or two 32-k groups of a stage");
  static_assert(kLoads >= 1, "at least one load per feeder");
};

// Everything a wavefront wrote to or read from LDS is done, then the block meets.  Loads from memory stay in flight.
__device__ __forceinline__ void ring_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// One stage's weights of a worker: one band x KW k, as loaded.
template <int FMT, int KC, int KW>
struct RingWeights {
  static constexpr int GPW = KW / 32;  // groups of 32 k
  static constexpr int ND = GPW * (FMT == RWKV_FMT_F16 ? 8 : (FMT == RWKV_FMT_W8 ? 4 : 2));
  uint32_t d[ND];
  half_t sc;
  uint32_t zb;

  __device__ __forceinline__ void put(int at, const uint4_t& v) {
    d[at] = v[0]; d[at + 1] = v[1]; d[at + 2] = v[2]; d[at + 3] = v[3];
  }
  // k32: the 32-k group of the matrix where the worker's share begins; wband: the band's first piece of this lane
  __device__ __forceinline__ void request(const StreamArgs& g, const StreamProblem& pr, int k32, const uint4_t* wband, int n) {
    if constexpr (FMT == RWKV_FMT_W8) {
#pragma unroll
      for (int i = 0; i < GPW; ++i) put(i * 4, __builtin_nontemporal_load(wband + static_cast<int64_t>(k32 + i) * 64));
    } else if constexpr (FMT == RWKV_FMT_F16) {
#pragma unroll
      for (int i = 0; i < 2 * GPW; ++i) put(i * 4, __builtin_nontemporal_load(wband + (static_cast<int64_t>(k32) * 2 + i) * 64));
    } else {
      static_assert(KW == 64, "a worker of int4 codes takes whole pieces");
      put(0, __builtin_nontemporal_load(wband + static_cast<int64_t>(k32 >> 1) * 64));
      const int q = n * pr.group_n + (k32 >> 2) * pr.group_k;
      sc = pr.scale[q];
      zb = pr.zp[q];
    }
  }
  __device__ __forceinline__ half8_t fragment(int st, half2_t zbias) const {
    if constexpr (FMT == RWKV_FMT_F16) {
      const uint4_t v = {d[st * 4], d[st * 4 + 1], d[st * 4 + 2], d[st * 4 + 3]};
      return __builtin_bit_cast(half8_t, v);
    } else if constexpr (FMT == RWKV_FMT_W8) {
      return expand_w8(d[st * 2], d[st * 2 + 1]);
    } else {
      return expand_w4(d[st], zbias);
    }
  }
};

// 16-byte piece of a staged row that lane half h meets in MFMA step st of group kg's share
template <int FMT, int KW>
__device__ __forceinline__ int ring_x_piece(int st, int kg, int h) {
  if constexpr (FMT == RWKV_FMT_W4) {
    return kg * 8 + h * 4 + st;
  } else {
    return kg * (KW / 8) + (st >> 1) * 4 + h * 2 + (st & 1);
  }
}

template <int FMT, int MT, int NB, int WP, int KC>
__device__ __forceinline__ void ring_work(const StreamArgs& g, const StreamProblem& pr, int col_block, int kbeg, int nstages,
                                          unsigned char* lds, int worker, int lane) {
  using T = RingTile<MT, NB, WP, KC>;
  using W = RingWeights<FMT, KC, T::KW>;
  constexpr int NS = T::KW / 16;  // MFMA steps per stage
  constexpr int kRegs = W::ND * NB;
  constexpr int D = FMT == RWKV_FMT_W4 && MT == 4 ? 3 : (kRegs <= 8 ? 4 : (kRegs <= 16 ? 3 : 2));  // register sets in the ring of weights
  const int j = lane & 31;
  const int h = lane >> 5;
  const int kg = worker / WP;
  const int wp = worker % WP;
  constexpr int G = FMT == RWKV_FMT_W4 ? 64 : 32;
  constexpr int PIECES = FMT == RWKV_FMT_F16 ? 2 : 1;
  const uint4_t* wband[NB];
  int n[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int band_here = (col_block * WP + wp) * NB + nb;
    const int band = band_here * 32 < pr.N ? band_here : pr.N / 32 - 1;  // past the last band: repeat it (columns not stored)
    wband[nb] = pr.wp + static_cast<int64_t>(band) * (g.K / G) * (PIECES * 64) + lane;
    n[nb] = band * 32 + j;
  }
  const int last = nstages - 1;
  const int k32 = (kbeg + kg * T::KW) >> 5;

  W w[D][NB];
  auto request = [&](int u, int c) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) w[u][nb].request(g, pr, k32 + (c < last ? c : last) * (KC / 32), wband[nb], n[nb]);
  };
#pragma unroll
  for (int i = 0; i < D - 1; ++i) request(i, i);

  float16_t acc[NB][MT];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[nb][mt][v] = 0.0f;
  int xoff[NS];
#pragma unroll
  for (int st = 0; st < NS; ++st) xoff[st] = j * T::kRowBytes + ((ring_x_piece<FMT, T::KW>(st, kg, h) ^ (j & 15)) << 4);
  auto load_a = [&](const unsigned char* xs, int st, half8_t (&dst)[MT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) dst[mt] = *reinterpret_cast<const half8_t*>(xs + xoff[st] + mt * 32 * T::kRowBytes);
  };

  int slot = 0;
  half8_t a[2][MT];
  auto stage = [&](int u, int c) {
    request((u + D - 1) % D, c + D - 1);
    const unsigned char* xs = lds + slot * T::kStageBytes;
    slot = slot + 1 == T::kStages ? 0 : slot + 1;
    const unsigned char* xs_next = lds + slot * T::kStageBytes;
    if constexpr (FMT == RWKV_FMT_W4) {
      // a worker's share of a stage lies in one 128-group: its sums on their own, folded with the group's scale, two row
      // tiles at a time (one tile's folds under the other's products)
      static_assert(NB == 1, "int4 tiles have one band per worker");
      const W& wc = w[u % D][0];
      uint32_t sr = __builtin_bit_cast(unsigned short, wc.sc), zr = wc.zb;
      asm volatile("" : "+v"(sr), "+v"(zr));  // converted here, below the requests of this stage
      const float scf = h2f(__builtin_bit_cast(half_t, static_cast<unsigned short>(sr)));
      const half_t zf = static_cast<half_t>(1024.0f + static_cast<float>(zr));
      const half2_t zbias = half2_t{zf, zf};
      constexpr int MP = MT >= 2 ? 2 : 1;
#pragma unroll
      for (int m0 = 0; m0 < MT; m0 += MP) {
        float16_t part[MP];
#pragma unroll
        for (int m = 0; m < MP; ++m)
#pragma unroll
          for (int v = 0; v < 16; ++v) part[m][v] = 0.0f;
#pragma unroll
        for (int st = 0; st < NS; ++st) {
          const half8_t b = wc.fragment(st, zbias);
#pragma unroll
          for (int m = 0; m < MP; ++m) {
            const half8_t ax = *reinterpret_cast<const half8_t*>(xs + xoff[st] + (m0 + m) * 32 * T::kRowBytes);
            part[m] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ax, b, part[m], 0, 0, 0);
          }
        }
#pragma unroll
        for (int m = 0; m < MP; ++m)
#pragma unroll
          for (int v = 0; v < 16; ++v) acc[0][m0 + m][v] = fmaf(part[m][v], scf, acc[0][m0 + m][v]);
      }
    } else {
      // a[0] holds step 0 already: the fragments of the next step - behind the last step, of the next stage's first - are
      // read while the current one multiplies.  The stage ends one step early: with the last step's fragments in
      // registers nobody reads it any more.
#pragma unroll
      for (int st = 0; st < NS; ++st) {
        if (st + 1 == NS) ring_barrier();
        if (st + 1 < NS) load_a(xs, st + 1, a[(st + 1) & 1]);
        else load_a(xs_next, 0, a[(st + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const half8_t b = w[u % D][nb].fragment(st, half2_t{});
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[nb][mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b, a[st & 1][mt], acc[nb][mt], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (FMT == RWKV_FMT_W4) ring_barrier();
  };
  static_assert(NS % 2 == 0, "the fragment sets alternate");

  ring_barrier();  // stage 0 has landed
  if constexpr (FMT != RWKV_FMT_W4) load_a(lds, 0, a[0]);
  // whole rounds of D stages as one basic block (with exits between them the compiler waits for every load in flight
  // at the head of each round), the stages left over with exits
  const int whole = nstages - nstages % D;
  int c0 = 0;
  for (; c0 < whole; c0 += D) {
#pragma unroll
    for (int u = 0; u < D; ++u) stage(u, c0 + u);
  }
  if (c0 < nstages) {
#pragma unroll
    for (int u = 0; u < D - 1; ++u) {
      if (c0 + u >= nstages) break;
      stage(u, c0 + u);
    }
  }

  // The group's sums into its plane.  A worker may still be reading the ring when another is here: they meet first (the
  // feeders with them).
  ring_barrier();
  float* red = reinterpret_cast<float*>(lds) + kg * T::BM * T::kRedLd;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int col = (wp * NB + nb) * 32;
      if constexpr (FMT == RWKV_FMT_W4) {  // lane j: column j, registers run along the rows
#pragma unroll
        for (int v = 0; v < 16; ++v) red[(mt * 32 + 8 * (v >> 2) + 4 * h + (v & 3)) * T::kRedLd + col + j] = acc[nb][mt][v];
      } else {  // lane j: row j, registers run along the columns
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4_t*>(red + (mt * 32 + j) * T::kRedLd + col + 8 * q + 4 * h) =
              float4_t{acc[nb][mt][4 * q], acc[nb][mt][4 * q + 1], acc[nb][mt][4 * q + 2], acc[nb][mt][4 * q + 3]};
      }
    }
}

template <int MT, int NB, int WP, int KC>
__device__ __forceinline__ void ring_feed(const StreamArgs& g, const StreamProblem& pr, int m0, int kbeg, int nstages,
                                          unsigned char* lds, int feeder, int lane) {
  using T = RingTile<MT, NB, WP, KC>;
  constexpr int S = T::kStages, PER = T::kLoads;
  constexpr int LPR = T::kRowBytes / 16;  // lanes (16-byte pieces) per row
  constexpr int RPL = 64 / LPR;           // rows per load
  // load i of feeder f: rows RPL (i * kRingFeeders + f) and following.  LDS receives lane after lane, so the swizzle that
  // keeps the fragment reads conflict-free is in the source: lane p of row r fetches piece p ^ (r & 15).
  uint32_t off[PER];
  const int rows = g.M - m0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int r = (i * kRingFeeders + feeder) * RPL + lane / LPR;
    const int row = r < rows ? r : rows - 1;  // rows past M repeat the last one (not stored)
    off[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(g.K) * 2u + (((lane % LPR) ^ (r & 15)) << 4);
  }
  const char* x0 = reinterpret_cast<const char*>(pr.x + static_cast<int64_t>(m0) * g.K + kbeg);
  auto request = [&](int c, int slot) {
    const char* src = x0 + c * T::kRowBytes;
    unsigned char* dst = lds + slot * T::kStageBytes + feeder * 1024;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + off[i]),
                                       (__attribute__((address_space(3))) void*)(dst + i * (kRingFeeders * 1024)), 16, 0, 0);
  };
  // Barrier c: stage c + 1 has landed and stage c has been read; stage c + S - 1 goes where stage c - 1 was.
#pragma unroll
  for (int c = 0; c < S - 1; ++c)
    if (c < nstages) request(c, c);
  if (nstages >= S - 1) wait_loads<PER * (S - 2)>();
  else wait_loads<0>();
  ring_barrier();  // stage 0 has landed
  int slot = S - 1;
  for (int c = 0; c < nstages; ++c) {
    if (c + S - 1 < nstages) {
      request(c + S - 1, slot);
      wait_loads<PER * (S - 2)>();
    } else {
      wait_loads<0>();
    }
    slot = slot + 1 == S ? 0 : slot + 1;
    ring_barrier();
  }
  ring_barrier();  // the ring is free
}

// One block of one problem: X staging and products, then the groups' planes added up in group order, scale and epilogue.
template <int FMT, int MT, int NB, int WP, int KC>
__device__ __forceinline__ void ring_block(const StreamArgs& g, const StreamProblem& pr, int row_tile, int col_block, int split,
                                           unsigned char* lds) {
  using T = RingTile<MT, NB, WP, KC>;
  const int m0 = row_tile * T::BM;
  const int kbeg = split * g.k_per_split;
  const int nstages = g.k_per_split / KC;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;

  // this thread's columns of the epilogue; their int8 scales are requested now (in the epilogue they would cost the block
  // a trip to memory)
  constexpr int kPieces = T::BN / 8;
  const int piece = threadIdx.x % kPieces;
  const int col = col_block * T::BN + piece * 8;
  const bool partial_out = g.splits > 1;
  half8_t scale_h;
#pragma unroll
  for (int e = 0; e < 8; ++e) scale_h[e] = static_cast<half_t>(1.0f);
  if (FMT == RWKV_FMT_W8 && !partial_out) scale_h = *reinterpret_cast<const half8_t*>(pr.scale + (col < pr.N ? col : pr.N - 8));

  if (wave >= kRingWorkers) {
    ring_feed<MT, NB, WP, KC>(g, pr, m0, kbeg, nstages, lds, wave - kRingWorkers, lane);
    ride_along_copy(g.copy, g.col_blocks * g.splits, 64 * kRingFeeders);  // (a block past the last pair has left)
  } else {
    ring_work<FMT, MT, NB, WP, KC>(g, pr, col_block, kbeg, nstages, lds, wave, lane);
  }
  __syncthreads();

  const float* red = reinterpret_cast<const float*>(lds);
  float* part_out = partial_out ? pr.partial + static_cast<int64_t>(split) * g.M * pr.N : nullptr;
  if (col >= pr.N) return;
  for (int row = threadIdx.x / kPieces; row < T::BM && m0 + row < g.M; row += kRingThreads / kPieces) {
    float val[8];
#pragma unroll
    for (int q = 0; q < T::KG; ++q) {
      const float4_t lo = *reinterpret_cast<const float4_t*>(red + (q * T::BM + row) * T::kRedLd + piece * 8);
      const float4_t hi = *reinterpret_cast<const float4_t*>(red + (q * T::BM + row) * T::kRedLd + piece * 8 + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        val[e] = q == 0 ? lo[e] : val[e] + lo[e];
        val[4 + e] = q == 0 ? hi[e] : val[4 + e] + hi[e];
      }
    }
    if (!partial_out) {
#pragma unroll
      for (int e = 0; e < 8; ++e) val[e] = finish_value(mul_f32(val[e], h2f(scale_h[e])), g.epilogue);
    }
    const int64_t o = static_cast<int64_t>(m0 + row) * pr.N + col;
    if (partial_out || g.out_f32) {
      float* dst = partial_out ? part_out + o : static_cast<float*>(pr.y) + o;
      *reinterpret_cast<float4_t*>(dst) = float4_t{val[0], val[1], val[2], val[3]};
      *reinterpret_cast<float4_t*>(dst + 4) = float4_t{val[4], val[5], val[6], val[7]};
    } else {
      half8_t hv;
#pragma unroll
      for (int e = 0; e < 8; ++e) hv[e] = f2h(val[e]);
      *reinterpret_cast<half8_t*>(static_cast<half_t*>(pr.y) + o) = hv;
    }
  }
}

// grid = 8 x row tiles x groups of eight (column block, K split) pairs: the workgroups of one pair differ in y only and run
// on the same XCD (linear id & 7), whose L2 they share the weights through; consecutive pairs are the splits of one column
// block, so that an XCD's workgroups ask for a part of X only.
// MIXED: fp16 problems beside int8 / int4 ones (the LoRA rank-ins beside the projections) take half as many columns per
// block, so that every block of the launch streams about the same bytes.
template <int FMT, bool MIXED, int MT, int NB, int WP, int KC>
__global__ __launch_bounds__(kRingThreads, 1) void gemm_ring_kernel(StreamArgs g) {
  using T = RingTile<MT, NB, WP, KC>;
  constexpr int NB2 = NB > 1 ? NB / 2 : 1, WP2 = NB > 1 ? WP : WP / 2;
  constexpr int kLds2 = MIXED ? RingTile<MT, NB2, MIXED ? WP2 : WP, KC>::kLdsBytes : 0;
  __shared__ __align__(1024) unsigned char lds[T::kLdsBytes > kLds2 ? T::kLdsBytes : kLds2];
  const int pair = blockIdx.z * 8 + blockIdx.x;
  if (pair >= g.col_blocks * g.splits) return;
  const int split = pair & (g.splits - 1);
  const int col_all = pair >> (31 - __builtin_clz(g.splits));
  int pi = 0, first = 0;
#pragma unroll
  for (int i = 0; i + 1 < kMaxProblems; ++i) {  // (unused entries lie behind the last block)
    const int end = g.block_end[i];
    pi = col_all >= end ? i + 1 : pi;
    first = col_all >= end ? end : first;
  }
  const StreamProblem& pr = g.p[pi];
  if constexpr (MIXED) {
    if (pr.fmt == RWKV_FMT_F16) {
      ring_block<RWKV_FMT_F16, MT, NB2, WP2, KC>(g, pr, blockIdx.y, col_all - first, split, lds);
      return;
    }
  }
  ring_block<FMT, MT, NB, WP, KC>(g, pr, blockIdx.y, col_all - first, split, lds);
}

template <int MT, int NB, int WP, int KC, int FMT, bool MIXED>
void launch(hipStream_t st, const StreamArgs& g) {
  const dim3 grid(8, g.row_tiles, ceil_div(g.col_blocks * g.splits, 8));
  hipLaunchKernelGGL((gemm_ring_kernel<FMT, MIXED, MT, NB, WP, KC>), grid, dim3(kRingThreads), 0, st, g);
}

constexpr int key_of(int mt, int nb, int wp, int kc, int fmt, bool mixed) {
  return ((((mt * 4 + nb) * 8 + wp) * 4 + kc / 128) * 4 + fmt) * 2 + (mixed ? 1 : 0);
}

struct RingEntry {
  int key;
  void (*launch)(hipStream_t, const StreamArgs&);
};
#define RING(MT, NB, WP, KC, FMT, MIXED) {key_of(MT, NB, WP, KC, FMT, MIXED), launch<MT, NB, WP, KC, FMT, MIXED>}
constexpr RingEntry kRingTable[] = {
    RING(1, 1, 2, 128, RWKV_FMT_W8, false), RING(1, 1, 2, 128, RWKV_FMT_F16, false), RING(1, 1, 2, 256, RWKV_FMT_W4, false),
    RING(1, 1, 2, 256, RWKV_FMT_W8, true),  RING(1, 1, 2, 256, RWKV_FMT_W4, true),   RING(2, 1, 2, 256, RWKV_FMT_W8, false),
    RING(2, 1, 2, 256, RWKV_FMT_F16, false), RING(2, 1, 2, 256, RWKV_FMT_W4, false), RING(2, 1, 2, 256, RWKV_FMT_W8, true),
    RING(2, 1, 2, 256, RWKV_FMT_W4, true),  RING(2, 2, 2, 128, RWKV_FMT_W8, false),  RING(2, 2, 2, 128, RWKV_FMT_F16, false),
    RING(2, 2, 2, 128, RWKV_FMT_W8, true),  RING(4, 1, 2, 128, RWKV_FMT_W8, false),  RING(4, 1, 2, 128, RWKV_FMT_F16, false),
    RING(4, 1, 4, 128, RWKV_FMT_W8, false),  RING(4, 1, 4, 128, RWKV_FMT_F16, false),
    RING(4, 1, 4, 128, RWKV_FMT_W4, false), RING(2, 1, 4, 128, RWKV_FMT_W4, false),  RING(2, 1, 4, 128, RWKV_FMT_W4, true),
    RING(1, 1, 4, 128, RWKV_FMT_W4, false), RING(1, 1, 4, 128, RWKV_FMT_W8, false), RING(1, 1, 4, 128, RWKV_FMT_F16, false),
    RING(4, 1, 4, 128, RWKV_FMT_W8, true),   RING(4, 1, 4, 128, RWKV_FMT_W4, true)};
#undef RING

const RingEntry* find_ring(const RingShape& s, int fmt, bool mixed) {
  const int key = key_of(s.mt, s.nb, s.wp, s.kc, fmt, mixed);
  for (const RingEntry& e : kRingTable)
    if (e.key == key) return &e;
  return nullptr;
}

}  // namespace

bool gemm_ring_has(const RingShape& s, int fmt, bool mixed) { return find_ring(s, fmt, mixed) != nullptr; }

int gemm_ring_launch(hipStream_t st, const RingShape& s, int fmt, bool mixed, const StreamArgs& g) {
  const RingEntry* e = find_ring(s, fmt, mixed);
  RWKV_REQUIRE(e != nullptr, "gemm_ring: no tile of %d x 32 rows and %d x 32 columns for format %d", s.mt, s.nb * s.wp, fmt);
  e->launch(st, g);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

}  // namespace rwkv
