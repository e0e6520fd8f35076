// Weight-streaming MFMA GEMM Y[M,N] = X[M,K] . W[N,K]^T over weights stored in an MFMA-native packed order.
// This is the path of prefill chunks and of batched decode, from 5 rows on (from 3 for int8 / int4 rows of 4096 and more).
//
// Reference: the cuBLAS / cuBLASLt calls behind rwkv7_v3a_linear_f16_orig_launch and
// rwkv7_v3a_linear_f16_orig_lt_cfg_launch (cuda/rwkv7_v3a_ops.cu:2235-2368): fp16 in, fp32 accumulate, fp16
// (or fp32) out.  The arithmetic there lives in a closed library; the contract is the textbook GEMM.
//
// Packed order.  v_mfma_f32_32x32x16_f16 takes, from lane l = j + 32h, 8 fp16 values of row j of each
// operand for 8 of the 16 k of the step; any assignment of k to (h, step) is valid as long as both operands
// use the same one.  A packed matrix is cut into tiles of 32 rows x G k (G = 32 for fp16 and int8 codes, 64
// for int4 codes); inside a tile lane (j, h) owns the KR = G/2 consecutive k [h*KR, h*KR + KR) of row j, and
// the tile is stored as 64 lanes x 16 bytes (x 2 pieces for fp16), tiles of one 32-row band consecutive
// along k.  A wavefront therefore streams one band with 1 KiB fully coalesced loads and feeds the pieces
// to the matrix core after an exact in-register expansion of the codes, without any transpose or LDS
// traffic for the weights; every weight byte leaves HBM once per 32*MT rows of X.
//
// Three kernels stream that order.  gemm_ring.hip: up to a few hundred rows (all rows for int4 codes), where the product is
// bound by the weights' and X's way into the CUs.  gemm_tile.hip: many rows, bound by the matrix core and the chip's power.  Here: a
// 64 x 256 tile of int8 codes between the two.  With more than one K split each block writes an fp32 partial tile and a second small kernel sums the partials in split order (a
// fixed order: results do not depend on scheduling) and applies scale and epilogue - or the LayerNorm kernel that consumes
// the result does (DeferredReduce).
#include <algorithm>
#include <climits>
#include <cstring>

#include "gemm_stream.h"

namespace rwkv {

template <int FMT>
struct PackTraits;
template <>
struct PackTraits<RWKV_FMT_F16> {
  static constexpr int KR = 16, PIECES = 2;
};
template <>
struct PackTraits<RWKV_FMT_W8> {
  static constexpr int KR = 16, PIECES = 1;
};
template <>
struct PackTraits<RWKV_FMT_W4> {
  static constexpr int KR = 32, PIECES = 1;
};

bool linear_packed_supported(int fmt, int M, int N, int K) {
  if (fmt != RWKV_FMT_F16 && fmt != RWKV_FMT_W8 && fmt != RWKV_FMT_W4) return false;
  return M >= 1 && N >= 32 && N % 32 == 0 && K >= 256 && K % 256 == 0;
}

// ---- packing: a permutation of the 16-byte pieces of the row-major codes ---------------------------------------------
__global__ __launch_bounds__(256) void pack_weights_kernel(int fmt, int N, int K, const uint4_t* __restrict__ src,
                                                           uint4_t* __restrict__ dst, int64_t n_pieces) {
  const int64_t p = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (p >= n_pieces) return;
  const int G = fmt == RWKV_FMT_W4 ? 64 : 32;
  const int KR = G / 2;
  const int pieces = fmt == RWKV_FMT_F16 ? 2 : 1;
  const int lane = static_cast<int>(p & 63);
  int64_t q = p >> 6;
  const int i = static_cast<int>(q % pieces);
  q /= pieces;
  const int KG = K / G;
  const int kg = static_cast<int>(q % KG);
  const int nt = static_cast<int>(q / KG);
  const int row = nt * 32 + (lane & 31);
  const int k = kg * G + (lane >> 5) * KR + i * 8;
  // elements per 16-byte piece: 8 (fp16), 16 (int8), 32 (int4)
  const int per = fmt == RWKV_FMT_F16 ? 8 : (fmt == RWKV_FMT_W8 ? 16 : 32);
  dst[p] = src[(static_cast<int64_t>(row) * K + k) / per];
}

int pack_weights_launch(hipStream_t st, int fmt, int N, int K, const void* w, void* packed) {
  RWKV_REQUIRE(linear_packed_supported(fmt, 16, N, K), "pack_weights: unsupported shape N=%d K=%d fmt=%d", N, K, fmt);
  RWKV_REQUIRE(w && packed && w != packed, "pack_weights: bad pointers");
  const int per = fmt == RWKV_FMT_F16 ? 8 : (fmt == RWKV_FMT_W8 ? 16 : 32);
  const int64_t n_pieces = static_cast<int64_t>(N) * K / per;
  hipLaunchKernelGGL(pack_weights_kernel, dim3(static_cast<unsigned>((n_pieces + 255) / 256)), dim3(256), 0, st, fmt,
                     N, K, static_cast<const uint4_t*>(w), static_cast<uint4_t*>(packed), n_pieces);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

// ---- the GEMM ---------------------------------------------------------------------------------------------------------

// The 64 x 256 tile: 32 * MT rows, chunks of KC k, four wavefronts, int8 codes.
struct Tile {
  using P = PackTraits<RWKV_FMT_W8>;
  static constexpr int MT = 2, KC = 128;
  static constexpr int BM = 32 * MT;
  static constexpr int G = 2 * P::KR;
  static constexpr int GROUPS = KC / G;
  static constexpr int NW = GROUPS * P::PIECES;     // weight pieces per lane per chunk and band
  static constexpr int STEPS = P::KR / 8;           // MFMA steps per group
  static constexpr int XSTRIDE = KC + 8;            // fp16 per staged row: 16-byte pad keeps b128 reads conflict-free
  static constexpr int GT = 256;                    // threads of the block
  static constexpr int XV = BM * (KC / 8) / GT;     // 16-byte vectors of X per thread per chunk
  static constexpr int kTileHalfs = BM * XSTRIDE;   // one staged X tile
};

// One chunk's slice of X held by a thread between request and its store to LDS.
struct XRegs {
  using T = Tile;
  static constexpr int KC = T::KC;
  uint4_t xv[T::XV];

  // vector i of the thread's slice
  __device__ __forceinline__ void request_one(int i, const StreamArgs& g, const StreamProblem& pr, int tid, int m0, int kc) {
    const int idx = tid + i * T::GT;
    const int r = idx / (KC / 8);
    const int c = (idx % (KC / 8)) * 8;
    // rows past M repeat the last row (their sums are never stored): a load under a per-lane branch, or merged
    // with a default value, makes the compiler drain every load in flight at the head of the chunk loop
    const int row = m0 + r < g.M ? m0 + r : g.M - 1;
    xv[i] = *reinterpret_cast<const uint4_t*>(pr.x + static_cast<int64_t>(row) * g.K + kc + c);
  }
  __device__ __forceinline__ void store_one(int i, int tid, half_t* xs) const {
    const int idx = tid + i * T::GT;
    const int r = idx / (KC / 8);
    const int c = (idx % (KC / 8)) * 8;
    *reinterpret_cast<uint4_t*>(xs + r * T::XSTRIDE + c) = xv[i];
  }

  __device__ __forceinline__ void request(const StreamArgs& g, const StreamProblem& pr, int tid, int m0, int kc) {
#pragma unroll
    for (int i = 0; i < T::XV; ++i) request_one(i, g, pr, tid, m0, kc);
  }

  __device__ __forceinline__ void store_x(int tid, half_t* xs) const {
#pragma unroll
    for (int i = 0; i < T::XV; ++i) store_one(i, tid, xs);
  }
};

// One chunk's weight pieces held by a lane between request and use.
struct WRegs {
  using T = Tile;
  uint4_t w[T::NW];

  // piece i of the chunk at kc
  __device__ __forceinline__ void request_piece(int i, int kc, const uint4_t* wband) {
    w[i] = wband[static_cast<int64_t>(kc / T::G) * (T::P::PIECES * 64) + i * 64];
  }
  __device__ __forceinline__ void request(int kc, const uint4_t* wband) {
#pragma unroll
    for (int i = 0; i < T::NW; ++i) request_piece(i, kc, wband);
  }
};

// ---- some hundred rows of int8 weights: 64 rows x 256 columns per block, two bands per wavefront ----------------------
// A wavefront keeps two 32-column bands (wave w: bands w and w + 4 of the block), so each X fragment it reads from LDS feeds two
// MFMAs.  One weight set per band, each piece requested again for the next chunk right after its last use (six MFMA steps ahead),
// and one set of X, requested during the first half of a chunk's steps and stored during the second: 168 registers and nine spilled,
// three wavefronts per SIMD, whose MFMAs fill each other's gaps.  (us per launch, 178 registers and two wavefronts / this: 65536 x 768, 160 rows
// 34.0 / 31.7, 600 rows 90.6 / 85.6; 32768 x 1024, 320 rows 37.7 / 34.1; 65536 x 2048, 192 rows 64.1 / 62.4; 16384 x 4096, 600 rows 102.5 /
// 96.7, 320 rows, about a block per CU, 60.6 / 62.1.)
__device__ __forceinline__ void stream_block_wide(const StreamArgs& g, const StreamProblem& pr, int row_tile, int col_block,
                                                  int split, half_t* xs) {
  using T = Tile;
  using P = T::P;
  constexpr int MT = T::MT, KC = T::KC, BM = T::BM, NB = 2;

  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int j = lane & 31;
  const int h = lane >> 5;
  const int m0 = row_tile * BM;
  const int kbeg = split * g.k_per_split;
  const int nchunks = g.k_per_split / KC;

  bool active[NB];
  int n[NB];
  const uint4_t* wband[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    const int band_here = col_block * (4 * NB) + nb * 4 + wave;
    active[nb] = band_here * 32 < pr.N;
    const int band = active[nb] ? band_here : pr.N / 32 - 1;  // past the last band: repeat it, store nothing
    n[nb] = band * 32 + j;
    wband[nb] = pr.wp + (static_cast<int64_t>(band) * (g.K / T::G)) * (P::PIECES * 64) + lane;
  }
  half_t scale_h[NB];  // the columns' int8 scales, requested before the main loop (in the epilogue: 1.2 us per launch)
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) scale_h[nb] = pr.scale[n[nb]];

  float16_t acc[NB][MT];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[nb][mt][v] = 0.0f;

  constexpr int NK = T::GROUPS * T::STEPS;        // MFMA steps of a chunk
  WRegs w[NB];
  XRegs xq;
  const int last = nchunks - 1;
  xq.request(g, pr, tid, m0, kbeg);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) w[nb].request(kbeg, wband[nb]);
  xq.store_x(tid, xs);
  __syncthreads();
  static_assert(T::XV % (NK / 2) == 0 && T::STEPS == 2 && T::NW == T::GROUPS,
                "a whole number of X vectors per MFMA step, two steps per weight piece");
  constexpr int XPS = T::XV / (NK / 2);  // X vectors requested (first half of the steps) or stored (second half) per step
  auto chunk = [&](int u, int c) {
    const half_t* tile = xs + (u & 1) * T::kTileHalfs;
    half_t* tile_next = xs + ((u + 1) & 1) * T::kTileHalfs;
    const int knext = kbeg + (c + 1 <= last ? c + 1 : c) * KC;  // past the end: the current chunk again (in cache)
    const half_t* xlane = tile + j * T::XSTRIDE + h * P::KR;
    half8_t a[2][MT];
    auto load_a = [&](int ks, half8_t (&dst)[MT]) {
      const half_t* xa = xlane + (ks / T::STEPS) * T::G + 8 * (ks % T::STEPS);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) dst[mt] = *reinterpret_cast<const half8_t*>(xa + mt * 32 * T::XSTRIDE);
    };
    load_a(0, a[0]);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks) {
      const int gi = ks / T::STEPS;
      const int st = ks % T::STEPS;
      if (ks + 1 < NK) load_a(ks + 1, a[(ks + 1) & 1]);
#pragma unroll
      for (int i = 0; i < XPS; ++i) {
        if (ks < NK / 2) {
          xq.request_one(XPS * ks + i, g, pr, tid, m0, knext);
        } else {
          xq.store_one(XPS * (ks - NK / 2) + i, tid, tile_next);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        const uint4_t piece = w[nb].w[gi];
        const half8_t b = st == 0 ? expand_w8(piece[0], piece[1]) : expand_w8(piece[2], piece[3]);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nb][mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[ks & 1][mt], b, acc[nb][mt], 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if (st == T::STEPS - 1) {  // piece gi has been expanded for the last time: the next chunk's takes its place
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) w[nb].request_piece(gi, knext, wband[nb]);
      }
    }
    __syncthreads();
  };
  const int whole = nchunks - nchunks % 2;
  int c0 = 0;
  for (; c0 < whole; c0 += 2) {
    chunk(0, c0);
    chunk(1, c0 + 1);
  }
  if (c0 < nchunks) chunk(0, c0);

  // output: one 128-column half of the tile at a time through LDS (the X tiles are free), written in 16/32-byte
  // pieces along the rows
  constexpr int kStageLd = 128 + 8;
  static_assert(BM * kStageLd * 4 <= 2 * T::kTileHalfs * 2, "epilogue tile exceeds the LDS tiles");
  float* stage = reinterpret_cast<float*>(xs);
  const bool partial_out = g.splits > 1;
  float* part_out = partial_out ? pr.partial + static_cast<int64_t>(split) * g.M * pr.N : nullptr;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    if (nb > 0) __syncthreads();  // the previous half has been read
    const float scl = partial_out ? 1.0f : h2f(scale_h[nb]);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const float sum = acc[nb][mt][v];
        const int row = mt * 32 + 8 * (v >> 2) + 4 * h + (v & 3);
        stage[row * kStageLd + wave * 32 + j] = partial_out ? sum : finish_value(mul_f32(sum, scl), g.epilogue);
      }
    __syncthreads();
    const int col0 = col_block * (128 * NB) + nb * 128;
    for (int idx = tid; idx < BM * 16; idx += 256) {
      const int row = idx >> 4;
      const int piece = idx & 15;
      const int col = col0 + piece * 8;
      if (m0 + row >= g.M || col >= pr.N) continue;
      const float4_t lo = *reinterpret_cast<const float4_t*>(stage + row * kStageLd + piece * 8);
      const float4_t hi = *reinterpret_cast<const float4_t*>(stage + row * kStageLd + piece * 8 + 4);
      const int64_t o = static_cast<int64_t>(m0 + row) * pr.N + col;
      if (partial_out || g.out_f32) {
        float* dst = partial_out ? part_out + o : static_cast<float*>(pr.y) + o;
        *reinterpret_cast<float4_t*>(dst) = lo;
        *reinterpret_cast<float4_t*>(dst + 4) = hi;
      } else {
        half8_t hv;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          hv[e] = f2h(lo[e]);
          hv[4 + e] = f2h(hi[e]);
        }
        *reinterpret_cast<half8_t*>(static_cast<half_t*>(pr.y) + o) = hv;
      }
    }
  }
}

__global__ __launch_bounds__(256, 3) void gemm_stream_wide_kernel(StreamArgs g) {
  __shared__ __align__(16) half_t xs[2 * Tile::kTileHalfs];
  ride_along_copy(g.copy, gridDim.x, blockDim.x);
  const int id = blockIdx.x;
  const int row_tile = (id >> 3) % g.row_tiles;
  const int pair = (id / (8 * g.row_tiles)) * 8 + (id & 7);
  if (pair >= g.col_blocks * g.splits) return;
  const int col_all = pair % g.col_blocks;
  const int split = pair / g.col_blocks;
  int pi = 0;
  while (pi + 1 < g.n_problems && col_all >= g.block_end[pi]) ++pi;
  const int col_block = col_all - (pi > 0 ? g.block_end[pi - 1] : 0);
  stream_block_wide(g, g.p[pi], row_tile, col_block, split, xs);
}

// int4 scales and zero points by group: the 32 columns of a band then lie in one piece of 64 (32) bytes, where the rows of
// [N][K/128] put every column in a cache line of its own (K = 16384, 17 / 64 / 256 rows: 19.4 / 25.8 / 57.9 -> 16.2 / 23.1 /
// 53.9 us per 4096-column product).  Load time only.
__global__ __launch_bounds__(256) void transpose_groups_kernel(int N, int groups, const half_t* __restrict__ scale,
                                                               const uint8_t* __restrict__ zp, half_t* __restrict__ scale_t,
                                                               uint8_t* __restrict__ zp_t) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<int64_t>(N) * groups) return;
  const int n = static_cast<int>(i % N);
  const int q = static_cast<int>(i / N);
  scale_t[i] = scale[static_cast<int64_t>(n) * groups + q];
  zp_t[i] = zp[static_cast<int64_t>(n) * groups + q];
}

int transpose_groups_launch(hipStream_t st, int N, int groups, const half_t* scale, const uint8_t* zp, half_t* scale_t,
                            uint8_t* zp_t) {
  RWKV_REQUIRE(N > 0 && groups > 0 && scale && zp && scale_t && zp_t, "transpose_groups: bad arguments");
  const unsigned blocks = static_cast<unsigned>((static_cast<int64_t>(N) * groups + 255) / 256);
  hipLaunchKernelGGL(transpose_groups_kernel, dim3(blocks), dim3(256), 0, st, N, groups, scale, zp, scale_t, zp_t);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

struct ReduceProblem {
  const float4_t* partial;
  const half_t* scale;  // NULL unless the problem's weights are int8 codes
  void* y;
  int N4;
};
struct ReduceArgs {
  ReduceProblem p[kMaxProblems];
  int block_end[kMaxProblems];
  int n_problems;
  int M, splits, epilogue, out_f32;
};

// y = finish(scale * sum over splits of partial), four columns per thread; blocks run over all problems.
__global__ __launch_bounds__(256) void splitk_reduce_kernel(ReduceArgs g) {
  int pi = 0;
  while (pi + 1 < g.n_problems && static_cast<int>(blockIdx.x) >= g.block_end[pi]) ++pi;
  const ReduceProblem& pr = g.p[pi];
  const int64_t plane4 = static_cast<int64_t>(g.M) * pr.N4;
  const int64_t i = static_cast<int64_t>(blockIdx.x - (pi > 0 ? g.block_end[pi - 1] : 0)) * 256 + threadIdx.x;
  if (i >= plane4) return;
  const float4_t* partial = pr.partial;
  // the scale first (without one: any readable vector), then the partials four at a time, each group requested
  // whole before its first member is added, in split order; past the last split the last one is read again and
  // left out - no load waits for an earlier one
  const half4_t sv = *reinterpret_cast<const half4_t*>(pr.scale ? pr.scale + (i % pr.N4) * 4
                                                                : reinterpret_cast<const half_t*>(partial));
  float4_t sum = partial[i];
  for (int base = 1; base < g.splits; base += 4) {
    float4_t q[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) q[u] = partial[(base + u < g.splits ? base + u : g.splits - 1) * plane4 + i];
    // (keeps the four requests together: the compiler would move each load down into the condition of its use)
#pragma unroll
    for (int u = 0; u < 4; ++u) asm volatile("" : "+v"(q[u]));
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (base + u < g.splits) sum = sum + q[u];
  }
  float4_t scl = {1.0f, 1.0f, 1.0f, 1.0f};
  if (pr.scale) scl = float4_t{h2f(sv[0]), h2f(sv[1]), h2f(sv[2]), h2f(sv[3])};
  float4_t val;
#pragma unroll
  for (int c = 0; c < 4; ++c) val[c] = finish_value(mul_f32(sum[c], scl[c]), g.epilogue);
  if (g.out_f32) {
    static_cast<float4_t*>(pr.y)[i] = val;
  } else {
    half4_t o;
#pragma unroll
    for (int c = 0; c < 4; ++c) o[c] = f2h(val[c]);
    static_cast<half4_t*>(pr.y)[i] = o;
  }
}

struct StreamConfig {
  RingShape ring = {0, 0, 0, 0};  // mt == 0: another tile
  int wide_rows = 0;              // of 256 columns: 64 (int8 only), 128 or 256 rows
  int fmt = RWKV_FMT_F16;         // ring: the launch's format
  bool mixed = false;             // ring: fp16 problems beside it
  int splits = 1;
  float us = 1e30f;               // estimate
  bool is_ring() const { return ring.mt > 0; }
  int rows() const { return is_ring() ? 32 * ring.mt : wide_rows; }
  int cols(int problem_fmt) const {
    if (!is_ring()) return 256;
    const int bn = 32 * ring.nb * ring.wp;
    return mixed && problem_fmt == RWKV_FMT_F16 ? bn / 2 : bn;
  }
  int k_step() const { return is_ring() ? ring.kc : 128; }
};

// Blocks that occupy the 256 CUs well enough without a K split.
constexpr int kFilledBlocks = 200;
// Rows from which the tiles of 256 columns, whose wavefronts feed two MFMAs from every X fragment they read from LDS, are looked at.
constexpr int kWideMinRows = 160;

// Estimated microseconds of a launch: what the choice between tiles and K splits goes by.  Fitted to sweeps of every tile and
// split over 5 .. 3000 rows x the matrices of the presets (768 .. 65536 columns, 768 .. 16384 k, three formats: 969 launches).
// Its pick takes the best one's time in half of them; in geometric mean 1.04 (int8), 1.02 (fp16), 1.01 (int4 scales by row)
// and 1.03 (by group) times, in one of ten more than 1.16 / 1.09 / 1.02 / 1.13 times (before the tiles of 128 and 256 rows).
//   ring: a fixed part (launch, first stage, epilogue); the bytes of the busiest CU at what a CU takes in while all of them
//   stream (94 GB/s; 130 while half of the chip idles); what of the HBM stream of the weights does not hide behind that; the
//   products; per further round of blocks its start and end, which a second block hides where two fit a CU.
//   64 x 256: bound by the matrix core; rounds past the second overlap.
//   128 and 256 x 256: a fixed part, then per stage of 64 k and round of blocks a time that grows with the blocks that run - the clock the
//   chip holds goes down with them - but not less than the stage's weights take at 4 TB/s out of HBM, where few row tiles share them
//   (fp16, 4096 x 16384, 160 .. 255 rows: tiles 56 .. 65 us, ring 46 .. 50); 128 rows: the start and end of every further round, 256
//   rows of fp16: a clock that goes on falling over full rounds (65536 x 4096, 512 rows 287 us, blocks of 128 rows 260).
//   K splits: their fp32 planes and, where no consumer sums them, the reduce launch; a consumer's block waits longer the more
//   planes it asks for (0.15 us each; with 0 / 0.4 decode steps of 5 .. 16 rows are 1-4 % slower, 7.2B and 1.5B int8).
//   int4 scales and zero points as [N][K/128] (group_rows): a cache line each per column and stage, of which the stage uses a few
//   bytes.  Two bytes per code of what a CU takes in, 1.5 with stages of 256 k; up to 2048 k a column's lie in 48 bytes.
// From 160 rows on, int8 and fp16, the pick takes 1.010 times the best one's time in geometric mean, in one call of twenty more than
// 1.08 times (every tile and split measured over 14 matrices of the presets' sizes, 552 launches of 160 .. 2048 rows).
static float estimate_us(const StreamConfig& c, int M, int K, int n_problems, const int* Ns, const int* fmts, bool deferred,
                         bool group_rows) {
  constexpr int kCus = 256;
  const int bm = c.rows();
  int blocks = 0, bn_max = 0;
  float block_bytes = 0.0f, w_bytes = 0.0f, n_total = 0.0f, f16_blocks = 0.0f;
  for (int i = 0; i < n_problems; ++i) {
    const int bn = c.cols(fmts[i]);
    const float per = fmts[i] == RWKV_FMT_F16 ? 2.0f : (fmts[i] == RWKV_FMT_W8 ? 1.0f : 0.55f);
    blocks += ceil_div(Ns[i], bn);
    if (fmts[i] == RWKV_FMT_F16) f16_blocks += ceil_div(Ns[i], bn);
    const float lines = group_rows && K > 2048 && fmts[i] == RWKV_FMT_W4 ? (c.k_step() == 128 ? 2.0f : 1.5f) : 0.0f;
    block_bytes = std::max(block_bytes, bn * (per + lines) + bm * 2.0f);
    bn_max = std::max(bn_max, bn);
    w_bytes += per * Ns[i];
    n_total += Ns[i];
  }
  const float k_block = static_cast<float>(K) / c.splits;
  const float f16_share = f16_blocks / blocks;
  blocks *= c.splits;
  // (each eighth pair of column block and split goes to the same XCD, whose 32 CUs run all its row tiles: twelve pairs of 18
  // row tiles leave four XCDs with 36 blocks.  Launches of several problems have too many pairs for it to matter.)
  if (n_problems == 1) blocks = ceil_div(blocks, 8) * 8;
  blocks *= ceil_div(M, bm);
  block_bytes *= k_block;
  w_bytes *= static_cast<float>(K);
  const int full = blocks / kCus, rest = blocks % kCus;
  const int rounds = full + (rest > 0 ? 1 : 0);
  float us;
  if (c.is_ring()) {
    us = 6.0f + 0.42f * w_bytes / 6.5e6f;
    us += full * block_bytes / 94e3f;
    if (rest > 0) us += block_bytes / (130e3f - 36e3f * std::max(0, rest - 128) / 128.0f);
    const float gflop = 2e-9f * bm * bn_max * k_block * kCus;
    const bool two_per_cu = c.ring.mt == 1 && c.ring.kc == 128;
    const bool wide_ring = c.ring.mt == 4 || c.ring.wp == 4;
    us += rounds * gflop * (c.fmt == RWKV_FMT_W4 ? (wide_ring ? 0.73f : 0.57f) : (c.ring.mt == 4 && c.fmt == RWKV_FMT_W8 ? 0.55f : (c.ring.nb == 2 ? 0.37f : (c.ring.mt == 1 && c.ring.wp == 4 ? 0.30f : 0.28f))));
    us += (two_per_cu ? 1.5f : 4.5f) * (rounds - 1);
  } else if (c.wide_rows > 64) {
    const float stage_bytes = 64.0f * 256.0f * (1.0f + f16_share) / ceil_div(M, bm);  // of weights, per block: the row tiles share them
    auto round_us = [&](int running) {
      const float stage = c.wide_rows == 256 ? 1.08f + 0.0027f * running + f16_share * (0.22f - 0.0006f * running) : 0.58f + 0.0013f * running;
      return std::max(stage, running * stage_bytes / 4.0e6f) * k_block / 64.0f;
    };
    us = (c.wide_rows == 256 ? 10.0f : 11.0f) + full * round_us(kCus) + (rest > 0 ? round_us(rest) : 0.0f) +
         (c.wide_rows == 256 ? f16_share * 0.3f * k_block / 64.0f * std::max(0, full - 1) : 6.0f * (rounds - 1));
  } else {
    const float part = std::max(1.0f, blocks * 1.05f / kCus);
    us = 1.09f * (7.0f + 34.0f * (part - 0.15f * std::max(0.0f, part - 2.0f)) * k_block / 4096.0f);
  }
  if (c.splits > 1) us += (deferred ? 0.35f + 0.15f * c.splits : 2.6f) + c.splits * M * n_total * (deferred ? 6.0f : 8.0f) / 5e6f;
  return us;
}

// Whether the planes of a K split may be left to the launch's consumer.  Inside a model the choice of tile and split goes by this
// alone and not by whether this call leaves them: a product has the same sums either way.  (linear_packed has no consumer and
// goes by the reduce launch it pays for.)
static bool sums_at_consumer(int n_problems, int epilogue, int out_f32) {
  return n_problems == 1 && epilogue == RWKV_EPI_NONE && !out_f32;
}

// wide: tiles of 256 columns are looked at (launch_config)
static StreamConfig search_config(int M, int K, int n_problems, const int* Ns, const int* fmts, bool deferred, bool group_rows,
                                  int max_splits, bool wide) {
  bool any[3] = {false, false, false};
  for (int i = 0; i < n_problems; ++i) any[fmts[i]] = true;
  StreamConfig best;
  auto consider = [&](StreamConfig c) {
    for (c.splits = 1; c.splits == 1 || (c.splits <= max_splits && K % (c.splits * c.k_step()) == 0); c.splits *= 2) {
      c.us = estimate_us(c, M, K, n_problems, Ns, fmts, deferred, group_rows);
      if (c.us < best.us) best = c;
    }
  };
  StreamConfig c;
  c.fmt = any[RWKV_FMT_W8] ? RWKV_FMT_W8 : (any[RWKV_FMT_W4] ? RWKV_FMT_W4 : RWKV_FMT_F16);
  c.mixed = c.fmt != RWKV_FMT_F16 && any[RWKV_FMT_F16];
  for (const RingShape& shape : kRingShapes) {
    if (!gemm_ring_has(shape, c.fmt, c.mixed)) continue;
    c.ring = shape;
    consider(c);
  }
  if (wide && M >= kWideMinRows && !any[RWKV_FMT_W4]) {
    c.ring = RingShape{0, 0, 0, 0};
    for (c.wide_rows = 128; c.wide_rows <= 256; c.wide_rows *= 2) consider(c);
    if (!any[RWKV_FMT_F16] && K <= 4096 && M <= 1024) {
      c.wide_rows = 64;
      consider(c);
    }
  }
  return best;
}

// The search over tiles and splits takes 1 to 6 us of host time, and a decode step asks for about ten choices before its first
// launch: each thread keeps the latest by all that they depend on (us per step, searching / kept: 1.5B shape fp16 4 rows
// 1270 / 1236, int8 13 rows 1189 / 1158; 7.2B shape int8 8 rows 2239 / 2198; 0.1B shape fp16 8 rows 460 / 447).
static StreamConfig choose_config(int M, int K, int n_problems, const int* Ns, const int* fmts, bool deferred, bool group_rows,
                                  int max_splits, bool wide) {
  struct Entry {
    int key[5 + 2 * kMaxProblems];
    bool used;
    StreamConfig config;
  };
  constexpr unsigned kSets = 32, kWays = 4;
  static thread_local Entry table[kSets][kWays];
  static thread_local unsigned oldest[kSets];
  int key[5 + 2 * kMaxProblems] = {M, K, n_problems, (deferred ? 1 : 0) + (group_rows ? 2 : 0) + (wide ? 4 : 0), max_splits};
  for (int i = 0; i < n_problems; ++i) {
    key[5 + 2 * i] = Ns[i];
    key[6 + 2 * i] = fmts[i];
  }
  uint32_t hash = 0;
  for (int i = 0; i < 5 + 2 * n_problems; ++i) hash = (hash ^ static_cast<uint32_t>(key[i])) * 0x9e3779b1u + (hash >> 15);
  const unsigned set = (hash >> 16) % kSets;
  for (const Entry& e : table[set])
    if (e.used && memcmp(e.key, key, sizeof key) == 0) return e.config;
  Entry& e = table[set][oldest[set]];
  oldest[set] = (oldest[set] + 1) % kWays;
  e.config = search_config(M, K, n_problems, Ns, fmts, deferred, group_rows, max_splits, wide);
  memcpy(e.key, key, sizeof key);
  e.used = true;
  return e.config;
}

// The operator: a K split is an offer, not a need, for int4 codes, from 513 rows on, where blocks of 32 x 32 alone occupy the chip and
// where K has no power of two of whole 512s (1024s up to 32 rows, and up to 64 rows of K up to 2048): such a call runs without a
// workspace too, with the split that fits.  Elsewhere a workspace too small for the split is an error.
static bool split_is_an_offer(int fmt, int M, int64_t N, int K) {
  return fmt == RWKV_FMT_W4 || M > 512 || K % (M <= 32 || (M <= 64 && K <= 2048) ? 1024 : 512) != 0 || ceil_div(M, 32) * (N / 32) >= kFilledBlocks;
}

// The format is not known here: the largest that any of the choices would need.
size_t linear_packed_workspace_bytes(int M, int N, int K) {
  int splits = 1;
  for (const int fmt : {RWKV_FMT_W8, RWKV_FMT_W4, RWKV_FMT_F16})
    splits = std::max(splits, choose_config(M, K, 1, &N, &fmt, false, fmt == RWKV_FMT_W4, 32, split_is_an_offer(fmt, M, N, K)).splits);
  return splits > 1 ? static_cast<size_t>(splits) * M * N * sizeof(float) : 0;
}

// int8 and int4 matrices side by side have no launch in common: f is called with the problems of each format.
template <typename F>
static int for_each_launch(int n_problems, const PackedProblem* problems, F&& f) {
  bool any[3] = {false, false, false};
  for (int i = 0; i < n_problems; ++i) any[problems[i].fmt] = true;
  if (!(any[RWKV_FMT_W8] && any[RWKV_FMT_W4])) return f(n_problems, problems);
  for (const int fmt : {RWKV_FMT_W8, RWKV_FMT_W4, RWKV_FMT_F16}) {
    PackedProblem part[kMaxProblems];
    int n = 0;
    for (int i = 0; i < n_problems; ++i)
      if (problems[i].fmt == fmt) part[n++] = problems[i];
    const int rc = n > 0 ? f(n, part) : RWKV_OK;
    if (rc != RWKV_OK) return rc;
  }
  return RWKV_OK;
}

size_t linear_packed_multi_workspace_bytes(int M, int K, int n_problems, const PackedProblem* problems, int epilogue, int out_f32) {
  size_t bytes = 0;
  for_each_launch(n_problems, problems, [&](int n, const PackedProblem* part) -> int {
    int Ns[kMaxProblems], fmts[kMaxProblems];
    int64_t n_total = 0;
    bool group_rows = false;
    for (int i = 0; i < n; ++i) {
      n_total += Ns[i] = part[i].N;
      fmts[i] = part[i].fmt;
      group_rows = group_rows || (fmts[i] == RWKV_FMT_W4 && !part[i].groups_first);
    }
    const int splits = choose_config(M, K, n, Ns, fmts, sums_at_consumer(n, epilogue, out_f32), group_rows, 32, true).splits;
    if (splits > 1) bytes = std::max(bytes, static_cast<size_t>(splits) * M * n_total * sizeof(float));
    return RWKV_OK;
  });
  return bytes;
}

// (0.9: a second launch's start and end are a guess.  7.2B shape int8, ms per chunk, together / apart: 260 rows 9.76 / 9.28, 340
// rows 10.53 / 10.30, 384 rows 10.42 / 10.56; 1.5B shape: 516 rows 4.79 / 4.86, 640 rows 5.23 / 5.18, 1200 rows 8.73 / 8.53)
bool linear_packed_apart(int M, int K, int n_first, int n_problems, const PackedProblem* problems) {
  int Ns[kMaxProblems], fmts[kMaxProblems];
  for (int i = 0; i < n_problems; ++i) {
    Ns[i] = problems[i].N;
    fmts[i] = problems[i].fmt;
    if (i < n_first && fmts[i] != RWKV_FMT_W8) return false;
  }
  const float together = choose_config(M, K, n_problems, Ns, fmts, false, false, 32, true).us;
  const float apart = choose_config(M, K, n_first, Ns, fmts, false, false, 32, true).us +
                      choose_config(M, K, n_problems - n_first, Ns + n_first, fmts + n_first, false, false, 32, true).us;
  return apart < 0.9f * together;
}

static int packed_launch(hipStream_t st, int M, int K, int n_problems, const PackedProblem* problems, int epilogue, int out_f32,
                         void* workspace, size_t workspace_bytes, bool fit_splits, bool at_consumer, bool op, DeferredReduce* defer,
                         const RowCopy* copy);

// What a launch with this workspace takes: no more K splits than fit it where they are an offer or the caller says so (fit_splits).  A
// model's launches look at every tile, the operator (op) at those of 256 columns only where a split is an offer.  Elsewhere fewer than
// 200 blocks of 32 x 32 leave them a handful of blocks, which want a split, and a call that runs without a workspace must go on to.
static StreamConfig launch_config(int M, int K, int n_problems, const int* Ns, const int* fmts, bool at_consumer, bool group_rows,
                                  size_t workspace_bytes, bool fit_splits, bool op) {
  int64_t n_total = 0;
  for (int i = 0; i < n_problems; ++i) n_total += Ns[i];
  const size_t plane = static_cast<size_t>(M) * n_total * sizeof(float);
  const bool offer = split_is_an_offer(fmts[0], M, n_total, K);
  const int max_splits = offer || fit_splits ? static_cast<int>(std::min<size_t>(32, workspace_bytes / plane)) : 32;
  return choose_config(M, K, n_problems, Ns, fmts, at_consumer, group_rows, max_splits, !op || offer);
}

static int require_supported(int M, int K, int n_problems, const PackedProblem* problems) {
  RWKV_REQUIRE(n_problems >= 1 && n_problems <= kMaxProblems, "linear_packed: %d problems (1..%d allowed)", n_problems,
               kMaxProblems);
  for (int i = 0; i < n_problems; ++i)
    RWKV_REQUIRE(linear_packed_supported(problems[i].fmt, M, problems[i].N, K), "linear_packed: unsupported shape M=%d N=%d K=%d fmt=%d",
                 M, problems[i].N, K, problems[i].fmt);
  return RWKV_OK;
}

int linear_packed_multi(hipStream_t st, int M, int K, int n_problems, const PackedProblem* problems, int epilogue,
                        int out_f32, void* workspace, size_t workspace_bytes, DeferredReduce* defer, const RowCopy* copy) {
  if (const int rc = require_supported(M, K, n_problems, problems)) return rc;
  return for_each_launch(n_problems, problems, [&](int n, const PackedProblem* part) {
    // (several problems take no more K splits than fit the workspace)
    const int rc = packed_launch(st, M, K, n, part, epilogue, out_f32, workspace, workspace_bytes, n_problems > 1,
                                 sums_at_consumer(n, epilogue, out_f32), false, n == n_problems ? defer : nullptr, copy);
    copy = nullptr;  // the rows ride on the first launch
    return rc;
  });
}

static int packed_launch(hipStream_t st, int M, int K, int n_problems, const PackedProblem* problems, int epilogue, int out_f32,
                         void* workspace, size_t workspace_bytes, bool fit_splits, bool at_consumer, bool op, DeferredReduce* defer,
                         const RowCopy* copy) {
  StreamArgs g;
  ReduceArgs r;
  if (copy) {
    RWKV_REQUIRE(copy->n >= 0 && copy->n % 8 == 0 && (copy->n == 0 || (copy->src && copy->dst)), "linear_packed: bad row copy");
    g.copy = *copy;
  }
  g.n_problems = r.n_problems = n_problems;
  g.M = r.M = M;
  g.K = K;
  g.epilogue = r.epilogue = epilogue;
  g.out_f32 = r.out_f32 = out_f32;
  int Ns[kMaxProblems], fmts[kMaxProblems];
  int64_t n_total = 0;
  bool group_rows = false;
  for (int i = 0; i < n_problems; ++i) {
    n_total += Ns[i] = problems[i].N;
    fmts[i] = problems[i].fmt;
    group_rows = group_rows || (fmts[i] == RWKV_FMT_W4 && !problems[i].groups_first);
  }
  const size_t plane = static_cast<size_t>(M) * n_total * sizeof(float);
  const StreamConfig cfg = launch_config(M, K, n_problems, Ns, fmts, at_consumer, group_rows, workspace ? workspace_bytes : 0, fit_splits,
                                         op);
  int col_blocks = 0;
  for (int i = 0; i < n_problems; ++i) {
    const PackedProblem& q = problems[i];
    RWKV_REQUIRE(q.x && q.packed && q.y, "linear_packed: NULL tensor");
    RWKV_REQUIRE(q.fmt == RWKV_FMT_F16 || q.scale, "linear_packed: quantised weights need a scale tensor");
    RWKV_REQUIRE(q.fmt != RWKV_FMT_W4 || q.zp, "linear_packed: W4 weights need a zero-point tensor");
    col_blocks += ceil_div(q.N, cfg.cols(q.fmt));
    g.block_end[i] = col_blocks;
    const int groups = K / 128;
    const bool by_group = q.groups_first;
    g.p[i] = StreamProblem{q.x, static_cast<const uint4_t*>(q.packed), q.scale, q.zp, q.y, nullptr, q.N, q.fmt,
                           by_group ? 1 : groups, by_group ? q.N : 1};
  }
  g.splits = r.splits = cfg.splits;
  g.k_per_split = K / g.splits;
  if (g.splits > 1) {
    const size_t need = g.splits * plane;
    RWKV_REQUIRE(workspace && workspace_bytes >= need, "linear_packed: workspace of %zu bytes needed, got %zu", need,
                 workspace_bytes);
    float* at = static_cast<float*>(workspace);
    int red_blocks = 0;
    for (int i = 0; i < n_problems; ++i) {
      g.p[i].partial = at;
      const int64_t plane4 = static_cast<int64_t>(M) * problems[i].N / 4;
      red_blocks += static_cast<int>((plane4 + 255) / 256);
      r.block_end[i] = red_blocks;
      r.p[i] = ReduceProblem{reinterpret_cast<const float4_t*>(at),
                             problems[i].fmt == RWKV_FMT_W8 ? problems[i].scale : nullptr, problems[i].y, problems[i].N / 4};
      at += static_cast<size_t>(g.splits) * M * problems[i].N;
    }
  }
  RWKV_REQUIRE(g.k_per_split % cfg.k_step() == 0, "linear_packed: K slice %d is not a whole number of %d-chunks", g.k_per_split,
               cfg.k_step());
  for (int i = n_problems - 1; i < kMaxProblems; ++i) g.block_end[i] = INT_MAX;
  g.row_tiles = ceil_div(M, cfg.rows());
  g.col_blocks = col_blocks;
  if (cfg.is_ring()) {
    const int rc = gemm_ring_launch(st, cfg.ring, cfg.fmt, cfg.mixed, g);
    if (rc != RWKV_OK) return rc;
  } else if (cfg.wide_rows > 64) {
    const int rc = gemm_tile_launch(st, cfg.wide_rows, g);
    if (rc != RWKV_OK) return rc;
  } else {
    hipLaunchKernelGGL(gemm_stream_wide_kernel, dim3(g.row_tiles * ceil_div(col_blocks * g.splits, 8) * 8), dim3(256), 0, st, g);
    RWKV_LAUNCH_CHECK();
  }
  if (defer) *defer = DeferredReduce{};
  if (g.splits == 1) return RWKV_OK;
  if (defer) {
    RWKV_REQUIRE(sums_at_consumer(n_problems, epilogue, out_f32),
                 "linear_packed: a deferred reduce takes one problem, fp16 output and no epilogue");
    defer->partial = g.p[0].partial;
    defer->scale = problems[0].fmt == RWKV_FMT_W8 ? problems[0].scale : nullptr;
    defer->plane = static_cast<int64_t>(M) * problems[0].N;
    defer->splits = g.splits;
    return RWKV_OK;
  }
  hipLaunchKernelGGL(splitk_reduce_kernel, dim3(r.block_end[n_problems - 1]), dim3(256), 0, st, r);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

int linear_packed(hipStream_t st, int fmt, int M, int N, int K, const half_t* x, const void* packed, const half_t* scale,
                  const uint8_t* zp, int epilogue, int out_f32, void* y, void* workspace, size_t workspace_bytes) {
  const PackedProblem q = {packed, scale, zp, x, y, N, fmt};
  if (const int rc = require_supported(M, K, 1, &q)) return rc;
  return packed_launch(st, M, K, 1, &q, epilogue, out_f32, workspace, workspace_bytes, false, false, true, nullptr, nullptr);
}

}  // namespace rwkv

using namespace rwkv;

extern "C" {

int rwkv_hip_pack_weights(rwkv_stream_t s, int fmt, int N, int K, const void* w, void* packed) {
  return pack_weights_launch(as_stream(s), fmt, N, K, w, packed);
}

int rwkv_hip_linear_packed_workspace(int M, int N, int K, size_t* bytes) {
  RWKV_REQUIRE(bytes && M > 0 && N > 0 && K > 0, "linear_packed_workspace: bad arguments");
  *bytes = linear_packed_workspace_bytes(M, N, K);
  return RWKV_OK;
}

int rwkv_hip_linear_packed_plan(int M, int K, int n_problems, const int* N, const int* fmt, size_t workspace_bytes, int* tile_rows,
                                int* tile_cols, int* splits, int* apart) {
  RWKV_REQUIRE(M > 0 && K > 0 && N && fmt && tile_rows && tile_cols && splits, "linear_packed_plan: bad arguments");
  RWKV_REQUIRE(n_problems >= 1 && n_problems <= kMaxProblems, "linear_packed_plan: %d problems (1..%d allowed)", n_problems, kMaxProblems);
  for (int i = 0; i < n_problems; ++i)
    RWKV_REQUIRE(linear_packed_supported(fmt[i], M, N[i], K) && (n_problems == 1 || fmt[i] != RWKV_FMT_W4),
                 "linear_packed_plan: unsupported shape M=%d N=%d K=%d fmt=%d", M, N[i], K, fmt[i]);
  const bool several = n_problems > 1;
  const StreamConfig c = launch_config(M, K, n_problems, N, fmt, false, fmt[0] == RWKV_FMT_W4, workspace_bytes, several, !several);
  *tile_rows = c.rows();
  *tile_cols = c.cols(c.fmt);
  *splits = c.splits;
  if (apart) {
    PackedProblem p[kMaxProblems] = {};
    int first = 0;  // the leading int8 matrices
    for (int i = 0; i < n_problems; ++i) {
      p[i].N = N[i];
      p[i].fmt = fmt[i];
      if (first == i && fmt[i] == RWKV_FMT_W8) ++first;
    }
    *apart = first > 0 && first < n_problems && linear_packed_apart(M, K, first, n_problems, p) ? 1 : 0;
  }
  return RWKV_OK;
}

int rwkv_hip_linear_packed(rwkv_stream_t s, int fmt, int M, int N, int K, const void* x, const void* packed,
                           const void* scale, const void* zp, int epilogue, int out_f32, void* y, void* workspace,
                           size_t workspace_bytes) {
  RWKV_REQUIRE(epilogue == RWKV_EPI_NONE || epilogue == RWKV_EPI_RELU_SQUARE, "linear_packed: bad epilogue %d", epilogue);
  return linear_packed(as_stream(s), fmt, M, N, K, static_cast<const half_t*>(x), packed,
                       static_cast<const half_t*>(scale), static_cast<const uint8_t*>(zp), epilogue, out_f32, y, workspace,
                       workspace_bytes);
}

}  // extern "C"
