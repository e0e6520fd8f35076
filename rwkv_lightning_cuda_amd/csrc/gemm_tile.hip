// Packed-weight MFMA GEMM for many rows of int8 and fp16 weights: blocks of 256 or 128 rows x 256 columns, X and the weights through a
// ring of LDS stages that every wavefront fills with direct-to-LDS loads.
//
// Reference: as gemm_stream.hip (cuda/rwkv7_v3a_ops.cu:2235-2368).
//
// What bounds it: the power the chip may draw.  At 2048 rows the 256-row blocks take 2610 clocks per stage of 64 k - 2048 of them the
// matrix core's - at 1.6 GHz; half as many blocks, alone on half the CUs, as many clocks at 2.1-2.3 GHz.  So a block moves as few bytes
// per product as its registers allow:
//   * Eight wavefronts, two per SIMD, each 128 (64) rows x 64 columns of accumulators: an X fragment out of LDS feeds two MFMAs, a
//     weight fragment four (two).  Wavefronts of 256 x 64, one per SIMD, expand every int8 code once instead of twice and read a tenth
//     less from LDS, and were slower (16384 x 4096, 2048 rows: 250 us against 237): nothing fills their waits.
//   * X and weights go from memory to LDS without passing through registers, two or three stages ahead, and weights arrive in the
//     order in which the matrix core reads them.  One barrier per stage, ahead of the last of its four steps.
//   * int8 codes become fp16 in eight instructions per fragment (expand_w8).
// us per launch, weights in no cache, before (the register-staged 128 x 256 tile, one wavefront per SIMD) -> now:
//   int8, 2048 rows: 16384 x 4096 282 -> 236 (1.16 PFLOP/s), 12288 x 4096 244 -> 204, 4096 x 16384 297 -> 235, 4096 x 4096 85 -> 71
//   int8, 512 rows: 16384 x 4096 85 -> 70, 12288 x 4096 78 -> 60      fp16, 2048 rows: 16384 x 4096 305 -> 250, 8192 x 2048 95 -> 67
//   fp16, 999 rows: 8192 x 2048 45 -> 38, 6144 x 2048 41 -> 35
#include "gemm_stream.h"

namespace rwkv {

namespace {

constexpr int kTileWaves = 8;
constexpr int kTileK = 64;    // k per stage
constexpr int kTileCols = 256;

template <int FMT, int MT>
struct WideTile {
  static constexpr int BM = 64 * MT;  // wavefronts 2 (rows) x 4 (columns), each 32 MT x 64
  static constexpr int kXBytes = BM * kTileK * 2;
  static constexpr int kPieces = FMT == RWKV_FMT_F16 ? 4 : 2;  // 1 KiB weight pieces of a band and stage
  static constexpr int kStageBytes = kXBytes + 8 * kPieces * 1024;
  static constexpr int kStages = kStageBytes <= 32768 ? 4 : (kStageBytes <= 49152 ? 3 : 2);
  static constexpr int kXLoads = BM / 8 / kTileWaves;   // 1 KiB direct-to-LDS loads per wavefront and stage
  static constexpr int kLoads = kXLoads + kPieces;
  static constexpr int kOutLd = 64 + 4;
  static constexpr int kOutBytes = kTileWaves * 32 * kOutLd * 4;  // the epilogue's 32 rows x 64 columns of every wavefront
  static constexpr int kLdsBytes = kStages * kStageBytes > kOutBytes ? kStages * kStageBytes : kOutBytes;
};

// 64 lanes x 16 bytes from base + off into LDS from `lds` on.  In asm, because the compiler would wait for every such load in flight
// at the next read of LDS.
__device__ __forceinline__ void load_to_lds(uint32_t lds, uint32_t off, const void* base) {
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"{m0}"(lds), "v"(off), "s"(base) : "memory");
}

template <int N>
__device__ __forceinline__ void meet() {  // all but the N youngest loads of this wavefront have landed, its LDS reads are done
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int FMT, int MT>
__device__ __forceinline__ void tile_block(const StreamArgs& g, const StreamProblem& pr, int row_tile, int col_block, int split,
                                           unsigned char* lds) {
  using T = WideTile<FMT, MT>;
  constexpr int S = T::kStages;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int lane = threadIdx.x & 63;
  const int j = lane & 31, h = lane >> 5;
  const int wm = wave & 1, wn = wave >> 1;
  const int m0 = row_tile * T::BM;
  const int kbeg = split * g.k_per_split;
  const int nstages = g.k_per_split / kTileK;

  // this lane's columns of the epilogue and their int8 scales
  const bool partial_out = g.splits > 1;
  const int col = col_block * kTileCols + wn * 64 + (lane & 7) * 8;
  half8_t scale_h;
#pragma unroll
  for (int e = 0; e < 8; ++e) scale_h[e] = static_cast<half_t>(1.0f);
  if (FMT == RWKV_FMT_W8 && !partial_out) scale_h = *reinterpret_cast<const half8_t*>(pr.scale + (col < pr.N ? col : pr.N - 8));

  // Loads of a stage: wavefront w brings rows 8 (8 i + w) .. + 7 of X and band w of the weights.  LDS receives lane after lane; the
  // 16-byte pieces of row r of X lie permuted by r & 7, so the permutation is in the addresses it reads from.
  uint32_t x_off[T::kXLoads];
  const int rows = g.M - m0;
#pragma unroll
  for (int i = 0; i < T::kXLoads; ++i) {
    const int r = (i * kTileWaves + wave) * 8 + (lane >> 3);
    const int row = r < rows ? r : rows - 1;  // rows past M repeat the last one (not stored)
    x_off[i] = static_cast<uint32_t>(row) * static_cast<uint32_t>(g.K) * 2u + (((lane & 7) ^ (r & 7)) << 4);
  }
  const char* x_base = reinterpret_cast<const char*>(pr.x + static_cast<int64_t>(m0) * g.K + kbeg);
  const int band_here = col_block * 8 + wave;
  const int band = band_here * 32 < pr.N ? band_here : pr.N / 32 - 1;  // past the last band: repeat it (columns not stored)
  const char* w_base = reinterpret_cast<const char*>(pr.wp) +
                       (static_cast<int64_t>(band) * (g.K / 32) + kbeg / 32) * (T::kPieces / 2 * 1024);
  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)lds));
  auto request_one = [&](int i, int c, int slot) {
    const uint32_t dst = lds0 + slot * T::kStageBytes;
    if (i < T::kXLoads) {
      load_to_lds(dst + (i * kTileWaves + wave) * 1024, x_off[i < T::kXLoads ? i : 0], x_base + c * (kTileK * 2));
    } else {
      const int q = i - T::kXLoads;
      load_to_lds(dst + T::kXBytes + (wave * T::kPieces + q) * 1024, lane * 16, w_base + (static_cast<int64_t>(c) * T::kPieces + q) * 1024);
    }
  };

  float16_t acc[2][MT];
#pragma unroll
  for (int nb = 0; nb < 2; ++nb)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[nb][mt][v] = 0.0f;

  int x_at[4];  // of the MFMA steps (16 k each)
#pragma unroll
  for (int st = 0; st < 4; ++st) x_at[st] = wm * MT * 4096 + j * 128 + ((((st >> 1) * 4 + h * 2 + (st & 1)) ^ (j & 7)) << 4);
  const int w_at = T::kXBytes + wn * 2 * T::kPieces * 1024 + lane * 16;

  half8_t a[2][MT];
  uint4_t w[2][2];  // fp16: of two steps; int8: of two 32-k groups, each two steps
  auto load_x = [&](const unsigned char* xs, int st, half8_t (&dst)[MT]) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) dst[mt] = *reinterpret_cast<const half8_t*>(xs + x_at[st] + mt * 4096);
  };
  auto load_w = [&](const unsigned char* xs, int piece, uint4_t (&dst)[2]) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) dst[nb] = *reinterpret_cast<const uint4_t*>(xs + w_at + (nb * T::kPieces + piece) * 1024);
  };
  auto multiply = [&](int st) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      half8_t b;
      if constexpr (FMT == RWKV_FMT_F16) {
        b = __builtin_bit_cast(half8_t, w[st & 1][nb]);
      } else {
        const uint4_t& p = w[st >> 1][nb];
        b = st & 1 ? expand_w8(p[2], p[3]) : expand_w8(p[0], p[1]);
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) acc[nb][mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b, a[st & 1][mt], acc[nb][mt], 0, 0, 0);
    }
  };

#pragma unroll
  for (int c = 0; c < S - 1; ++c)
    if (c < nstages) {
#pragma unroll
      for (int i = 0; i < T::kLoads; ++i) request_one(i, c, c);
    }
  if (nstages >= S - 1) meet<T::kLoads * (S - 2)>();
  else meet<0>();
  load_x(lds, 0, a[0]);
  load_w(lds, 0, w[0]);

  int slot = 0, slot_free = S - 1;
  // Stage c; `more`: stage c + S - 1 exists and is requested, into the place of stage c - 1, which everybody has read.  The block meets
  // ahead of the last step, whose fragments are in registers by then: stage c + 1 has landed and its first ones are read under
  // that step's products.
  auto stage = [&](int c, auto more) {
    const unsigned char* xs = lds + slot * T::kStageBytes;
    slot = slot + 1 == S ? 0 : slot + 1;
    const unsigned char* xs_next = lds + slot * T::kStageBytes;
#pragma unroll
    for (int st = 0; st < 4; ++st) {
      if constexpr (decltype(more)::value) {
#pragma unroll
        for (int i = 0; i < T::kLoads; ++i)
          if (i * 3 / T::kLoads == st) request_one(i, c + S - 1, slot_free);
      }
      if (st < 3) {
        load_x(xs, st + 1, a[(st + 1) & 1]);
        if constexpr (FMT == RWKV_FMT_F16) load_w(xs, st + 1, w[(st + 1) & 1]);
        else if (st == 0) load_w(xs, 1, w[1]);
      } else {
        if constexpr (decltype(more)::value) meet<T::kLoads * (S - 2)>();
        else meet<0>();
        load_x(xs_next, 0, a[0]);
        if constexpr (FMT == RWKV_FMT_F16) load_w(xs_next, 0, w[0]);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(st);
      if constexpr (FMT != RWKV_FMT_F16) {
        if (st == 3) load_w(xs_next, 0, w[0]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    slot_free = slot_free + 1 == S ? 0 : slot_free + 1;
  };
  int c = 0;
  for (; c + S - 1 < nstages; ++c) stage(c, std::true_type{});
  for (; c < nstages; ++c) stage(c, std::false_type{});  // (the last one reads on into a stage that is not multiplied)

  // 32 rows x 64 columns of a wavefront at a time through its own part of LDS, written in 16/32-byte pieces along the rows
  meet<0>();
  float* out = reinterpret_cast<float*>(lds) + wave * 32 * T::kOutLd;
  float* part_out = partial_out ? pr.partial + static_cast<int64_t>(split) * g.M * pr.N : nullptr;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<float4_t*>(out + j * T::kOutLd + nb * 32 + 8 * q + 4 * h) =
            float4_t{acc[nb][mt][4 * q], acc[nb][mt][4 * q + 1], acc[nb][mt][4 * q + 2], acc[nb][mt][4 * q + 3]};
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = i * 8 + (lane >> 3);
      const int row = m0 + (wm * MT + mt) * 32 + r;
      const float4_t lo = *reinterpret_cast<const float4_t*>(out + r * T::kOutLd + (lane & 7) * 8);
      const float4_t hi = *reinterpret_cast<const float4_t*>(out + r * T::kOutLd + (lane & 7) * 8 + 4);
      if (row >= g.M || col >= pr.N) continue;
      float val[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if (!partial_out) {
#pragma unroll
        for (int e = 0; e < 8; ++e) val[e] = finish_value(mul_f32(val[e], h2f(scale_h[e])), g.epilogue);
      }
      const int64_t o = static_cast<int64_t>(row) * pr.N + col;
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
    __builtin_amdgcn_wave_barrier();
  }
}

template <int MT>
__global__ __launch_bounds__(64 * kTileWaves, 2) void gemm_tile_kernel(StreamArgs g) {
  constexpr int kA = WideTile<RWKV_FMT_W8, MT>::kLdsBytes, kB = WideTile<RWKV_FMT_F16, MT>::kLdsBytes;
  __shared__ __align__(1024) unsigned char lds[kA > kB ? kA : kB];
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
  const StreamProblem& pr = g.p[pi];
  if (pr.fmt == RWKV_FMT_W8) tile_block<RWKV_FMT_W8, MT>(g, pr, row_tile, col_block, split, lds);
  else tile_block<RWKV_FMT_F16, MT>(g, pr, row_tile, col_block, split, lds);
}

}  // namespace

int gemm_tile_launch(hipStream_t st, int rows, const StreamArgs& g) {
  const dim3 grid(g.row_tiles * ceil_div(g.col_blocks * g.splits, 8) * 8);
  if (rows == 256) hipLaunchKernelGGL(gemm_tile_kernel<4>, grid, dim3(64 * kTileWaves), 0, st, g);
  else hipLaunchKernelGGL(gemm_tile_kernel<2>, grid, dim3(64 * kTileWaves), 0, st, g);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

}  // namespace rwkv
