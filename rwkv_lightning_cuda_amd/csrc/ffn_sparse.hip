// Channel-mix down projection of a few tokens that reads, per token, only the rows of ffn.value whose activation
// is non-zero.
//
// Reference: rwkv7_cmix_sparse_down_relu_one_launch / _rows_launch and cmix_sparse_spmv_relu_one_kernel / _rows_kernel
// (cuda/rwkv7_fast_ops_fp16.cu:966-992,618-737; call site src/rwkv7_fast_v4.cu:1285-1292), per token:
//   vec[f] = f16(relu(preact[f])^2);  out[c] = sum over f with vec[f] != 0 of vec[f] * Wv[f][c]
// over ffn.value stored [F,C], so that a skipped f skips a contiguous row.  The reference accumulates in half2
// with atomicAdd (the result depends on block order); here the products are exact, the accumulation is fp32 and
// the order is fixed, so the result is the dense product of the same codes up to fp32 summation order.
//
// Weights: the [C,F] matrix transposed to [F,C]: fp16 values as they are, or int8 codes stored offset by 128
// (u = q + 128, one byte each) with the same per-output-channel fp16 scale.
//
// Kernel 1: grid = (row blocks, column chunks, tokens), block = 8 wavefronts.  A wavefront owns 32 .. 128 consecutive f and a
// chunk of 256 columns (fp16: 128), one row's piece of it per lane group of 16 lanes: it lists the rows with a non-zero
// activation in LDS, its four lane groups walk the list two rows each at a time (v_dot2_f32_f16: v_perm_b32 pairs the values of
// the two rows; int8: bytes under exponent 0x64, then one packed subtract gives the exact codes), the groups' sums meet by
// lane swaps, the wavefronts' in LDS in wavefront order, and the block writes one fp32 partial row.  Kernel 2 sums the
// partial rows in a fixed order, applies the scale and rounds to fp16.
//
// Narrow chunks make few partial rows: 7.2B int8 has 16 of them (256 blocks; a chunk of a whole wavefront's 1024 columns had
// 64) and 1.5B int8 still a block per CU.  us per layer, one / two tokens, in the decode step: 7.2B int8 54.1 / 62.6 ->
// 52.9 / 60.5, int4 44.9 / 56.7 -> 42.0 / 52.6, fp16 79.1 / 89.8 -> 76.8 / 85.6; 1.5B int8 35.0 / 43.0 -> 32.1 / 37.8, int4 36.2 /
// 45.8 -> 32.6 / 39.4.  Measured and left: the block that draws a chunk's last ticket sums the partial rows instead of the
// second launch (3.4 us of tail against the launch's 4.4 in a trace, but 0.9 us per layer slower in the replayed step).
#include <mutex>

#include "ops.h"

namespace rwkv {

// Partial rows of the entry point that allocates nothing (rwkv_hip_cmix_sparse_down_relu_rows_static): a fixed
// array in the library's device image, one copy per GPU, held until the process ends.  In host code this name
// is only a handle for hipGetSymbolAddress; kernels get the address that call returns.
constexpr size_t kStaticScratchBytes = static_cast<size_t>(16) << 20;
static __device__ __align__(256) float scratch[kStaticScratchBytes / sizeof(float)];

constexpr int kSparseWaves = 8;
constexpr int kSparseRowsPerBlock = 32 * kSparseWaves;  // 256: the fewest rows of a block that the entry points' workspace is sized for

// columns per lane = values in a 16-byte piece
constexpr int sparse_lane_cols(int fmt) { return fmt == RWKV_FMT_F16 ? 8 : 16; }

bool ffn_sparse_supported(int fmt, int C, int F) {
  if (fmt != RWKV_FMT_W8 && fmt != RWKV_FMT_F16 && fmt != RWKV_FMT_W4) return false;
  return C >= 16 && C % 16 == 0 && F >= kSparseRowsPerBlock && F % kSparseRowsPerBlock == 0;
}

// Bytes of the transposed copy.  int4: the [F,C/2] codes, then the scales [F/128,C] (fp16), then the zero points
// [F/128,C] (one byte each) - a wavefront's 32 rows lie in one 128-group, so it needs one scale and one zero point
// per column.
size_t ffn_sparse_packed_bytes(int fmt, int C, int F) {
  const size_t cf = static_cast<size_t>(C) * F;
  if (fmt == RWKV_FMT_F16) return cf * 2;
  if (fmt == RWKV_FMT_W8) return cf;
  return cf / 2 + static_cast<size_t>(F / 128) * C * 3;
}

size_t ffn_sparse_workspace_bytes(int rows, int C, int F) {
  return static_cast<size_t>(rows) * (F / kSparseRowsPerBlock) * C * sizeof(float);
}

// ---- [C,F] -> [F,C] (int8 codes get the offset) ----------------------------------------------------------------------
// grid = (F/64, C/64) tiles through LDS; C and F multiples of 64 are not required (edges are predicated).
template <typename E>
__global__ __launch_bounds__(256) void ffn_sparse_pack_kernel(int C, int F, const E* __restrict__ w, E* __restrict__ wt) {
  __shared__ E tile[64][65];
  const int f0 = blockIdx.x * 64;
  const int c0 = blockIdx.y * 64;
  for (int i = threadIdx.x; i < 64 * 64; i += 256) {
    const int c = i >> 6;
    const int f = i & 63;
    E v = 0;
    if (c0 + c < C && f0 + f < F) v = w[static_cast<int64_t>(c0 + c) * F + f0 + f];
    if constexpr (sizeof(E) == 1) v ^= 0x80u;
    tile[c][f] = v;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 64; i += 256) {
    const int f = i >> 6;
    const int c = i & 63;
    if (c0 + c < C && f0 + f < F) wt[static_cast<int64_t>(f0 + f) * C + c0 + c] = tile[c][f];
  }
}

int ffn_sparse_pack_launch(hipStream_t st, int fmt, int C, int F, const void* w, void* wt) {
  RWKV_REQUIRE(fmt != RWKV_FMT_W4 && ffn_sparse_supported(fmt, C, F),
               "ffn_sparse_pack: unsupported format %d or shape C=%d F=%d (int4 codes: ffn_sparse_pack_w4)", fmt, C, F);
  RWKV_REQUIRE(w && wt && w != wt, "ffn_sparse_pack: bad pointers");
  const dim3 grid(ceil_div(F, 64), ceil_div(C, 64));
  if (fmt == RWKV_FMT_W8) {
    hipLaunchKernelGGL(ffn_sparse_pack_kernel<uint8_t>, grid, dim3(256), 0, st, C, F, static_cast<const uint8_t*>(w),
                       static_cast<uint8_t*>(wt));
  } else {
    hipLaunchKernelGGL(ffn_sparse_pack_kernel<uint16_t>, grid, dim3(256), 0, st, C, F, static_cast<const uint16_t*>(w),
                       static_cast<uint16_t*>(wt));
  }
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

// int4: q [C,F/2] (even f in the low nibble) -> t [F,C/2] (even c in the low nibble); 64 x 64 tiles of nibbles.
__global__ __launch_bounds__(256) void ffn_sparse_pack_w4_kernel(int C, int F, const uint8_t* __restrict__ q,
                                                                 uint8_t* __restrict__ t) {
  __shared__ uint8_t tile[64][65];
  const int f0 = blockIdx.x * 64;
  const int c0 = blockIdx.y * 64;
  for (int i = threadIdx.x; i < 64 * 32; i += 256) {
    const int c = i >> 5;
    const int fb = i & 31;
    uint8_t v = 0;
    if (c0 + c < C && f0 + 2 * fb < F) v = q[static_cast<int64_t>(c0 + c) * (F / 2) + f0 / 2 + fb];
    tile[c][2 * fb] = v & 15;
    tile[c][2 * fb + 1] = v >> 4;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * 32; i += 256) {
    const int f = i >> 5;
    const int cb = i & 31;
    if (c0 + 2 * cb < C && f0 + f < F)
      t[static_cast<int64_t>(f0 + f) * (C / 2) + c0 / 2 + cb] = tile[2 * cb][f] | (tile[2 * cb + 1][f] << 4);
  }
}

// scale / zp [C,F/128] -> [F/128,C]
__global__ __launch_bounds__(256) void ffn_sparse_pack_w4_groups_kernel(int C, int G, const half_t* __restrict__ scale,
                                                                        const uint8_t* __restrict__ zp,
                                                                        half_t* __restrict__ scale_t,
                                                                        uint8_t* __restrict__ zp_t) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (i >= static_cast<int64_t>(C) * G) return;
  const int g = static_cast<int>(i / C);
  const int c = static_cast<int>(i - static_cast<int64_t>(g) * C);
  scale_t[i] = scale[static_cast<int64_t>(c) * G + g];
  zp_t[i] = zp[static_cast<int64_t>(c) * G + g];
}

int ffn_sparse_pack_w4_launch(hipStream_t st, int C, int F, const void* q, const half_t* scale, const uint8_t* zp,
                              void* wt) {
  RWKV_REQUIRE(ffn_sparse_supported(RWKV_FMT_W4, C, F), "ffn_sparse_pack: unsupported shape C=%d F=%d", C, F);
  RWKV_REQUIRE(q && scale && zp && wt && q != wt, "ffn_sparse_pack: bad pointers");
  uint8_t* codes = static_cast<uint8_t*>(wt);
  const int G = F / 128;
  half_t* scale_t = reinterpret_cast<half_t*>(codes + static_cast<size_t>(C) * F / 2);
  uint8_t* zp_t = reinterpret_cast<uint8_t*>(scale_t + static_cast<size_t>(G) * C);
  hipLaunchKernelGGL(ffn_sparse_pack_w4_kernel, dim3(ceil_div(F, 64), ceil_div(C, 64)), dim3(256), 0, st, C, F,
                     static_cast<const uint8_t*>(q), codes);
  RWKV_LAUNCH_CHECK();
  hipLaunchKernelGGL(ffn_sparse_pack_w4_groups_kernel, dim3(static_cast<unsigned>((static_cast<int64_t>(C) * G + 255) / 256)),
                     dim3(256), 0, st, C, G, scale, zp, scale_t, zp_t);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

// ---- kernel 1 ------------------------------------------------------------------------------------------------------------
constexpr int kSparseSteps = 2;  // steps of a batch (4: the same within 1 %; 8, or loads under branches: 2-6 % of the step slower)
constexpr int kSparseGroups = 4;  // lane groups of a wavefront, each with a row's piece of the chunk
constexpr int kSparseListed = 128 + 8;  // entries of a wavefront's list, the pad of the last step among them

template <int FMT>
struct SparsePiece {
  typedef uint4_t type;
};
template <>
struct SparsePiece<RWKV_FMT_W4> {
  typedef uint2_t type;
};

// acc += a_lo * (the piece's columns of row lo) + a_hi * (those of row hi), for every token's pair ap = (a_lo, a_hi)
template <int FMT, int TOK>
__device__ __forceinline__ void sparse_pair(const typename SparsePiece<FMT>::type& qlo, const typename SparsePiece<FMT>::type& qhi,
                                            const half2_t (&ap)[TOK], float (&acc)[TOK][sparse_lane_cols(FMT)]) {
  constexpr int kDwords = sizeof(qlo) / 4;
#pragma unroll
  for (int d = 0; d < kDwords; ++d) {
    const uint32_t lo = qlo[d];
    const uint32_t hi = qhi[d];
    if constexpr (FMT == RWKV_FMT_F16) {
      // a dword holds two columns of a row: pair the low halves and the high halves of the two rows
      const half2_t w0 = as_half2(__builtin_amdgcn_perm(hi, lo, 0x05040100u));
      const half2_t w1 = as_half2(__builtin_amdgcn_perm(hi, lo, 0x07060302u));
#pragma unroll
      for (int t = 0; t < TOK; ++t) {
        acc[t][2 * d + 0] = __builtin_amdgcn_fdot2(ap[t], w0, acc[t][2 * d + 0], false);
        acc[t][2 * d + 1] = __builtin_amdgcn_fdot2(ap[t], w1, acc[t][2 * d + 1], false);
      }
    } else if constexpr (FMT == RWKV_FMT_W8) {
      const half2_t bias = {static_cast<half_t>(1152.0f), static_cast<half_t>(1152.0f)};
      half2_t w[4];
      w[0] = as_half2(__builtin_amdgcn_perm(hi, lo, 0x0c040c00u) | 0x64006400u) - bias;
      w[1] = as_half2(__builtin_amdgcn_perm(hi, lo, 0x0c050c01u) | 0x64006400u) - bias;
      w[2] = as_half2(__builtin_amdgcn_perm(hi, lo, 0x0c060c02u) | 0x64006400u) - bias;
      w[3] = as_half2(__builtin_amdgcn_perm(hi, lo, 0x0c070c03u) | 0x64006400u) - bias;
#pragma unroll
      for (int t = 0; t < TOK; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[t][4 * d + i] = __builtin_amdgcn_fdot2(ap[t], w[i], acc[t][4 * d + i], false);
    } else {
      // nibble n of the dword is column 8 d + n.  The bytes of the two rows are paired once for both of their nibbles; under exponent
      // 0x64 the low one is 1024 + q, the high one in place 1024 + 16 q, exact after the subtract (the 16 comes off after the walk).
      // (Codes as fp16 denormals would save the subtract, but v_dot2_f32_f16 keeps fewer bits of such products: 2.26e-4
      // instead of 2.09e-4 from the 64-bit result at 4096 x 16384.)
      const half2_t bias = {static_cast<half_t>(1024.0f), static_cast<half_t>(1024.0f)};
      half2_t w[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t both = __builtin_amdgcn_perm(hi, lo, 0x0c040c00u + 0x00010001u * i);
        w[2 * i] = as_half2((both & 0x000f000fu) | 0x64006400u) - bias;
        w[2 * i + 1] = as_half2((both & 0x00f000f0u) | 0x64006400u) - bias;
      }
#pragma unroll
      for (int t = 0; t < TOK; ++t)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[t][8 * d + i] = __builtin_amdgcn_fdot2(ap[t], w[i], acc[t][8 * d + i], false);
    }
  }
}

// Sums over the four lane groups of a wavefront, each group keeping a quarter of the columns (v[0 .. N/4) afterwards): after the
// swap of v[i] and v[i + N/2] the lower half of the wavefront holds both halves' v[i], the upper half both halves' v[i + N/2];
// then the same between neighbouring rows of 16 lanes.  (Two idle slots between a register's write and the swap that reads it.)
template <int N>
__device__ __forceinline__ void sum_scatter_groups(float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(v[i]), "+v"(v[i + N / 2]));
    v[i] += v[i + N / 2];
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1" : "+v"(v[i]), "+v"(v[i + N / 4]));
    v[i] += v[i + N / 4];
  }
}

struct SparseArgs {
  int C, F;
  int rpw;        // rows of ffn.value per wavefront: 32, 64 or 128 (int4: within one 128-group)
  int activated;  // `in` already holds f16(relu(preact)^2) (the model's ffn.key launch applies it)
  const half_t* in;
  const uint8_t* wt;
  float* partial;
};

template <int FMT, int TOK>
__global__ __launch_bounds__(64 * kSparseWaves) void ffn_sparse_kernel(SparseArgs a) {
  typedef typename SparsePiece<FMT>::type piece_t;
  constexpr int LC = sparse_lane_cols(FMT);  // columns per lane
  constexpr int G = kSparseGroups;
  constexpr int kLanes = 64 / G;             // lanes of a group: one row's piece of the column chunk
  constexpr int kCols = kLanes * LC;         // columns per block
  constexpr int kKept = LC / G;              // columns a lane keeps (sum_scatter_groups)
  constexpr int kThreads = 64 * kSparseWaves;
  __shared__ __align__(16) float red[kSparseWaves][kCols];
  __shared__ __align__(8) uint16_t row_s[kSparseWaves][kSparseListed];
  __shared__ __align__(8) uint16_t coef_s[TOK][kSparseWaves][kSparseListed];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int group = lane / kLanes;
  const int C = a.C;
  const int f0 = (blockIdx.x * kSparseWaves + wave) * a.rpw;
  const int c0 = blockIdx.y * kCols;
  const int cl = c0 + LC * (lane % kLanes);  // this lane's first column
  const half_t* in = a.in + static_cast<int64_t>(blockIdx.z) * a.F;                   // this token's activations ...
  float* partial = a.partial + static_cast<int64_t>(blockIdx.z) * gridDim.x * C;      // ... and partial rows
  const uint32_t row_bytes = static_cast<uint32_t>(C / LC) * sizeof(piece_t);
  const uint8_t* wlane = a.wt + static_cast<int64_t>(f0) * row_bytes + (cl < C ? cl / LC : 0) * sizeof(piece_t);

  // the columns this lane ends with
  const int cq = LC * (lane % kLanes) + (LC / 2) * (lane >> 5) + (LC / 4) * ((lane >> 4) & 1);
  half4_t w4_scale[kKept / 4 + 1];
  uint32_t w4_zp[kKept / 4 + 1];
  if constexpr (FMT == RWKV_FMT_W4) {
    const int n_groups = a.F / 128;
    const half_t* scale_t = reinterpret_cast<const half_t*>(a.wt + static_cast<size_t>(C) * a.F / 2);
    const uint8_t* zp_t = reinterpret_cast<const uint8_t*>(scale_t + static_cast<size_t>(n_groups) * C);
    const int64_t gat = static_cast<int64_t>(f0 / 128) * C + (c0 + cq < C ? c0 + cq : 0);
#pragma unroll
    for (int i = 0; i < kKept / 4; ++i) {
      w4_scale[i] = *reinterpret_cast<const half4_t*>(scale_t + gat + 4 * i);
      w4_zp[i] = *reinterpret_cast<const uint32_t*>(zp_t + gat + 4 * i);
    }
  }

  // the wavefront's list: rows that are non-zero for any of its tokens, in increasing order, with every token's coefficient
  int n = 0;
  for (int r0 = 0; r0 < a.rpw; r0 += 64) {
    const int r = r0 + lane;
    uint16_t bits[TOK];
    bool any = false;
#pragma unroll
    for (int t = 0; t < TOK; ++t) {
      float x = h2f(in[static_cast<int64_t>(t) * a.F + f0 + (r < a.rpw ? r : 0)]);
      if (!a.activated) {
        x = fmaxf(round_h(x), 0.0f);
        x = round_h(x * x);
      }
      bits[t] = __builtin_bit_cast(uint16_t, f2h(x));
      any |= (bits[t] & 0x7fffu) != 0u;  // +0 and -0 both count as zero
    }
    any &= r < a.rpw;
    const uint64_t mask = __ballot(any);
    if (any) {
      const int at = n + __builtin_popcountll(mask & ((1ull << lane) - 1));
      row_s[wave][at] = static_cast<uint16_t>(r);
#pragma unroll
      for (int t = 0; t < TOK; ++t) coef_s[t][wave][at] = bits[t];
    }
    n += __builtin_popcountll(mask);
  }
  // a step takes two rows per lane group; the last one is filled up with a row that is read anyway, at coefficient zero
  const int steps = (n + 2 * G - 1) / (2 * G);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (n > 0 && n + lane < 2 * G * steps) {
    row_s[wave][n + lane] = row_s[wave][0];
#pragma unroll
    for (int t = 0; t < TOK; ++t) coef_s[t][wave][n + lane] = 0;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");

  float acc[TOK][LC];
  float asum[TOK];
#pragma unroll
  for (int t = 0; t < TOK; ++t) {
    asum[t] = 0.0f;
#pragma unroll
    for (int i = 0; i < LC; ++i) acc[t][i] = 0.0f;
  }
  // Batches of kSparseSteps steps, the next one in flight under the products of this one.  No load sits under a branch (the compiler
  // would wait for all of them at the first use): steps past the last repeat it.
  auto request = [&](int s0, piece_t (&q)[kSparseSteps][2]) {
#pragma unroll
    for (int u = 0; u < kSparseSteps; ++u) {
      const uint32_t rows = *reinterpret_cast<const uint32_t*>(&row_s[wave][2 * (G * min(s0 + u, steps - 1) + group)]);
      q[u][0] = __builtin_nontemporal_load(reinterpret_cast<const piece_t*>(wlane + static_cast<uint64_t>(rows & 0xffffu) * row_bytes));
      q[u][1] = __builtin_nontemporal_load(reinterpret_cast<const piece_t*>(wlane + static_cast<uint64_t>(rows >> 16) * row_bytes));
    }
  };
  auto take = [&](int s, const piece_t (&q)[2]) {
    half2_t ap[TOK];
#pragma unroll
    for (int t = 0; t < TOK; ++t) {
      ap[t] = as_half2(*reinterpret_cast<const uint32_t*>(&coef_s[t][wave][2 * (G * s + group)]));
      if constexpr (FMT == RWKV_FMT_W4) asum[t] += h2f(ap[t][0]) + h2f(ap[t][1]);
    }
    sparse_pair<FMT, TOK>(q[0], q[1], ap, acc);
  };
  if (steps > 0) {
    piece_t q[kSparseSteps][2];
    request(0, q);
    int s0 = 0;
    for (; s0 + kSparseSteps < steps; s0 += kSparseSteps) {
      piece_t next[kSparseSteps][2];
      request(s0 + kSparseSteps, next);
#pragma unroll
      for (int u = 0; u < kSparseSteps; ++u) take(s0 + u, q[u]);
#pragma unroll
      for (int u = 0; u < kSparseSteps; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i) q[u][i] = next[u][i];
    }
#pragma unroll
    for (int u = 0; u < kSparseSteps; ++u)
      if (s0 + u < steps) take(s0 + u, q[u]);
  }

#pragma unroll
  for (int t = 0; t < TOK; ++t) {
    sum_scatter_groups(acc[t]);
    if constexpr (FMT == RWKV_FMT_W4) {
      // sum_f a_f (q_fc - zp_c) = sum_f a_f q_fc - zp_c sum_f a_f, and the scale of the wavefront's 128-group
      asum[t] = add_swapped_rows<false>(add_swapped_rows<true>(asum[t]));
#pragma unroll
      for (int i = 0; i < kKept; ++i) {
        const float zp = static_cast<float>((w4_zp[i >> 2] >> (8 * (i & 3))) & 0xffu);
        acc[t][i] = (acc[t][i] * (i & 1 ? 0.0625f : 1.0f) - zp * asum[t]) * h2f(w4_scale[i >> 2][i & 3]);
      }
    }
    if (t > 0) __syncthreads();  // the sums of the token before have been read
#pragma unroll
    for (int i = 0; i < kKept; ++i) red[wave][cq + i] = acc[t][i];
    __syncthreads();
    // the wavefronts' sums meet in wavefront order
    for (int c = threadIdx.x; c < kCols && c0 + c < C; c += kThreads) {
      float sum = red[0][c];
#pragma unroll
      for (int w = 1; w < kSparseWaves; ++w) sum += red[w][c];
      partial[(static_cast<int64_t>(t) * gridDim.x + blockIdx.x) * C + c0 + c] = sum;
    }
  }
}

// ---- kernel 2: out[c] = f16(scale[c] * sum of the partial rows) -----------------------------------
// grid = (ceil(C/64) and one for the optional row copy, tokens), block = 256 = 16 groups of partial rows x 16 column quads.  Group g sums rows g, g+16, ... (its
// loads are independent, so they are all in flight together), the 16 group sums meet in LDS in group order.
__global__ __launch_bounds__(256) void ffn_sparse_finish_kernel(int C, int n_partial, const float* __restrict__ partial,
                                                                const half_t* __restrict__ scale,
                                                                half_t* __restrict__ out, RowCopy copy) {
  __shared__ __align__(16) float red[16][64];
  if (static_cast<int>(blockIdx.x) * 64 >= C) {  // the block past the columns
    if (blockIdx.y == 0)
      for (int i = threadIdx.x * 8; i < copy.n; i += 256 * 8)
        *reinterpret_cast<uint4_t*>(copy.dst + i) = *reinterpret_cast<const uint4_t*>(copy.src + i);
    return;
  }
  const int g = threadIdx.x >> 4;
  const int cq = (threadIdx.x & 15) * 4;
  const int c = blockIdx.x * 64 + cq;
  partial += static_cast<int64_t>(blockIdx.y) * n_partial * C;  // this token's partial rows ...
  out += static_cast<int64_t>(blockIdx.y) * C;                  // ... and output row
  float4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
  if (c < C) {
#pragma unroll 4
    for (int p = g; p < n_partial; p += 16) sum = sum + *reinterpret_cast<const float4_t*>(partial + static_cast<int64_t>(p) * C + c);
  }
  *reinterpret_cast<float4_t*>(&red[g][cq]) = sum;
  __syncthreads();
  if (threadIdx.x >= 16 || c >= C) return;
  float4_t total = *reinterpret_cast<const float4_t*>(&red[0][cq]);
#pragma unroll
  for (int i = 1; i < 16; ++i) total = total + *reinterpret_cast<const float4_t*>(&red[i][cq]);
  half4_t sv = {static_cast<half_t>(1.0f), static_cast<half_t>(1.0f), static_cast<half_t>(1.0f), static_cast<half_t>(1.0f)};
  if (scale) sv = *reinterpret_cast<const half4_t*>(scale + c);
  half4_t o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = f2h(total[i] * h2f(sv[i]));
  *reinterpret_cast<half4_t*>(out + c) = o;
}

template <int FMT>
static void launch_walk(hipStream_t st, dim3 grid, int tokens, const SparseArgs& a) {
  const dim3 block(64 * kSparseWaves);
  if (tokens == 1) hipLaunchKernelGGL((ffn_sparse_kernel<FMT, 1>), grid, block, 0, st, a);
  else if (tokens == 2) hipLaunchKernelGGL((ffn_sparse_kernel<FMT, 2>), grid, block, 0, st, a);
  else if (tokens == 3) hipLaunchKernelGGL((ffn_sparse_kernel<FMT, 3>), grid, block, 0, st, a);
  else hipLaunchKernelGGL((ffn_sparse_kernel<FMT, 4>), grid, block, 0, st, a);
}

// Bytes of ffn.value from which the walk can beat the dense product; below, the dense product is the faster one however many
// activations are zero, because the walk's second launch and its lists cost more than the whole matrix.  us per layer of a decode
// step, dense / walk with the given share of the rows needed by any token of the step (1 - z^tokens at a share z of zeros; random-init
// weights have z = 0.5, and the dense product costs the same at any z):
//   one token    0.1B fp16 (5 MB) 20.7 / 23.1 at 0.51, 22.2 at 0.04   1.5B int4 (9 MB) 30.5 / 29.9 at 0.49, 29.2 at 0.05
//   two tokens   0.1B fp16 23.9 / 27.0 at 0.75, 25.7 at 0.07          1.5B int4 38.5 / 37.0 at 0.70, 35.8 at 0.07
//   three        1.5B int8 (17 MB) 38.9 / 41.1 at 0.82, 40.4 at 0.49, 38.9 at 0.08    1.5B fp16 (32 MB) 43.9 / 44.7, 43.1, 40.7
//   four         1.5B int8 40.7 / 43.5 at 0.88, 43.0 at 0.54, 41.3 at 0.09            1.5B fp16 45.4 / 46.8, 45.3, 42.8
//   three, four  7.2B int8 (64 MB) 67.0 / 68.3 at 0.82, 65.3 at 0.49, 60.7 at 0.09 and 67.6 / 69.4 at 0.87, 66.4 at 0.52, 61.7 at 0.09;
//                7.2B int4 (34 MB) 60.4 / 61.9, 59.5, 55.9 and 60.5 / 64.2, 61.1, 56.6
// From 32 MB on three and four tokens gain from some 70 to 80 % of zeros per token on and lose 1 to 6 % at one half: the choice counts
// on weights that are trained (the reference walks for up to 12 tokens by default).
bool ffn_sparse_pays(int fmt, int rows, int C, int F) {
  const size_t bytes = ffn_sparse_packed_bytes(fmt, C, F);
  return rows <= 2 ? bytes >= (8u << 20) : rows <= kSparseUnionMaxRows && bytes >= (32u << 20);
}

int ffn_sparse_launch(hipStream_t st, int fmt, int rows, int C, int F, int activated, const half_t* in, const void* wt,
                      const half_t* scale, void* workspace, size_t workspace_bytes, half_t* out, const RowCopy* copy,
                      bool one_walk) {
  RWKV_REQUIRE(ffn_sparse_supported(fmt, C, F), "ffn_sparse: unsupported format %d or shape C=%d F=%d", fmt, C, F);
  RWKV_REQUIRE(rows >= 1 && rows <= kSparseMaxRows, "ffn_sparse: %d rows (1..%d)", rows, kSparseMaxRows);
  RWKV_REQUIRE(in && wt && out && (fmt != RWKV_FMT_W8 || scale), "ffn_sparse: NULL tensor");
  RWKV_REQUIRE(workspace && workspace_bytes >= ffn_sparse_workspace_bytes(rows, C, F),
               "ffn_sparse: workspace of %zu bytes needed, got %zu", ffn_sparse_workspace_bytes(rows, C, F), workspace_bytes);
  RowCopy cp;
  if (copy) {
    RWKV_REQUIRE(copy->n % 8 == 0, "ffn_sparse: row copy length %d must be a multiple of 8", copy->n);
    cp = *copy;
  }
  // 2 .. 4 tokens share one walk over the rows that are non-zero for any of them; otherwise a walk per token
  const int tokens = one_walk && rows >= 2 && rows <= kSparseUnionMaxRows ? rows : 1;
  // Rows per wavefront: as many as leave three blocks to four CUs, or more than three to two CUs where every token has its own walk -
  // what a wavefront does besides its rows, lists and sums, is most of its instructions when few of 32 rows are needed.  us per
  // call with 32 / 64 / 128 rows, half of the activations zero (a tenth not zero): one token, 2048 x 8192 int8 6.6 / 6.9 / 8.4 (5.5 / 5.3 /
  // 6.0), 2560 x 10240 int8 7.9 / 7.5 / 8.4 (6.2 / 5.7 / 6.1), fp16 9.9 / 9.9 / 9.3 (7.1 / 6.1 / 6.2), three that share a walk 13.9 / 13.9 / 13.1; 12 tokens, 2048 x
  // 8192 int8 20.8 / 17.6 / 15.8 (14.6 / 9.9 / 8.5), 2560 x 10240 int4 29.8 / 23.1 / 21.4 (22.3 / 14.3 / 11.5); 3 tokens, 2048 x 8192 fp16 13.3 / 11.8 /
  // 13.1 (8.5 / 6.7 / 6.7).
  const int walks = rows / tokens;
  const int chunks = ceil_div(C, 64 / kSparseGroups * sparse_lane_cols(fmt));
  const int64_t least = walks > 1 ? device_cu_count() * 3 / 2 + 1 : device_cu_count() * 3 / 4;
  int rpw = 128;
  while (rpw > 32 && (F % (kSparseWaves * rpw) != 0 || static_cast<int64_t>(chunks) * (F / (kSparseWaves * rpw)) * walks < least)) rpw /= 2;
  const SparseArgs a = {C, F, rpw, activated, in, static_cast<const uint8_t*>(wt), static_cast<float*>(workspace)};
  const int n_partial = F / (kSparseWaves * rpw);
  const dim3 grid(n_partial, chunks, walks);
  if (fmt == RWKV_FMT_W4) launch_walk<RWKV_FMT_W4>(st, grid, tokens, a);
  else if (fmt == RWKV_FMT_W8) launch_walk<RWKV_FMT_W8>(st, grid, tokens, a);
  else launch_walk<RWKV_FMT_F16>(st, grid, tokens, a);
  RWKV_LAUNCH_CHECK();
  hipLaunchKernelGGL(ffn_sparse_finish_kernel, dim3(ceil_div(C, 64) + (cp.n > 0 ? 1 : 0), rows), dim3(256), 0, st, C, n_partial,
                     static_cast<const float*>(workspace), fmt == RWKV_FMT_W8 ? scale : nullptr, out, cp);
  RWKV_LAUNCH_CHECK();
  return RWKV_OK;
}

}  // namespace rwkv

using namespace rwkv;

extern "C" {

int rwkv_hip_cmix_sparse_pack(rwkv_stream_t s, int fmt, int C, int F, const void* w, void* wt) {
  return ffn_sparse_pack_launch(as_stream(s), fmt, C, F, w, wt);
}

int rwkv_hip_cmix_sparse_pack_w4(rwkv_stream_t s, int C, int F, const void* q, const void* scale, const void* zp,
                                 void* wt) {
  return ffn_sparse_pack_w4_launch(as_stream(s), C, F, q, static_cast<const half_t*>(scale),
                                   static_cast<const uint8_t*>(zp), wt);
}

int rwkv_hip_cmix_sparse_packed_bytes(int fmt, int C, int F, size_t* bytes) {
  RWKV_REQUIRE(bytes, "cmix_sparse_packed_bytes: NULL argument");
  RWKV_REQUIRE(ffn_sparse_supported(fmt, C, F), "cmix_sparse_packed_bytes: unsupported format %d or shape C=%d F=%d", fmt, C,
               F);
  *bytes = ffn_sparse_packed_bytes(fmt, C, F);
  return RWKV_OK;
}

int rwkv_hip_cmix_sparse_workspace(int rows, int C, int F, size_t* bytes) {
  RWKV_REQUIRE(bytes, "cmix_sparse_workspace: NULL argument");
  RWKV_REQUIRE(ffn_sparse_supported(RWKV_FMT_W8, C, F), "cmix_sparse_workspace: unsupported shape C=%d F=%d", C, F);
  RWKV_REQUIRE(rows >= 1 && rows <= kSparseMaxRows, "cmix_sparse_workspace: %d rows (1..%d)", rows, kSparseMaxRows);
  *bytes = ffn_sparse_workspace_bytes(rows, C, F);
  return RWKV_OK;
}

int rwkv_hip_cmix_sparse_down_relu_rows(rwkv_stream_t s, int fmt, int rows, int C, int F, const void* preact,
                                        const void* wt, const void* scale, void* workspace, size_t workspace_bytes,
                                        void* out) {
  return ffn_sparse_launch(as_stream(s), fmt, rows, C, F, 0, static_cast<const half_t*>(preact), wt,
                           static_cast<const half_t*>(scale), workspace, workspace_bytes, static_cast<half_t*>(out), nullptr, false);
}

int rwkv_hip_cmix_sparse_down_relu_rows_shared(rwkv_stream_t s, int fmt, int rows, int C, int F, const void* preact,
                                               const void* wt, const void* scale, void* workspace,
                                               size_t workspace_bytes, void* out) {
  RWKV_REQUIRE(rows >= 2 && rows <= kSparseUnionMaxRows, "cmix_sparse_shared: %d rows (2..%d)", rows, kSparseUnionMaxRows);
  return ffn_sparse_launch(as_stream(s), fmt, rows, C, F, 0, static_cast<const half_t*>(preact), wt,
                           static_cast<const half_t*>(scale), workspace, workspace_bytes, static_cast<half_t*>(out), nullptr, true);
}

// Device address of this GPU's copy of `scratch`, looked up once per device (with that device current).
static int static_scratch_address(float** out) {
  constexpr int kMaxDevices = 64;
  static std::mutex lock;
  static float* address[kMaxDevices] = {nullptr};
  int dev = 0;
  RWKV_HIP_TRY(hipGetDevice(&dev));
  RWKV_REQUIRE(dev >= 0 && dev < kMaxDevices, "cmix_sparse_static: device index %d out of range", dev);
  std::lock_guard<std::mutex> guard(lock);
  if (address[dev] == nullptr) {
    float* p = nullptr;
    RWKV_HIP_TRY(hipGetSymbolAddress(reinterpret_cast<void**>(&p), HIP_SYMBOL(scratch)));
    RWKV_REQUIRE(p != nullptr, "cmix_sparse_static: no device address for the scratch array");
    address[dev] = p;
  }
  *out = address[dev];
  return RWKV_OK;
}

int rwkv_hip_cmix_sparse_down_relu_rows_static(rwkv_stream_t s, int fmt, int rows, int C, int F, const void* preact,
                                               const void* wt, const void* scale, void* out) {
  RWKV_REQUIRE(ffn_sparse_supported(fmt, C, F), "cmix_sparse_static: unsupported format %d or shape C=%d F=%d", fmt, C, F);
  RWKV_REQUIRE(rows >= 1 && rows <= kSparseMaxRows, "cmix_sparse_static: %d rows (1..%d)", rows, kSparseMaxRows);
  const size_t need = ffn_sparse_workspace_bytes(rows, C, F);
  RWKV_REQUIRE(need <= kStaticScratchBytes,
               "cmix_sparse_static: rows=%d C=%d F=%d needs %zu bytes of partial rows, the built-in scratch holds %zu", rows,
               C, F, need, kStaticScratchBytes);
  float* ws = nullptr;
  const int rc = static_scratch_address(&ws);
  if (rc != RWKV_OK) return rc;
  return ffn_sparse_launch(as_stream(s), fmt, rows, C, F, 0, static_cast<const half_t*>(preact), wt,
                           static_cast<const half_t*>(scale), ws, kStaticScratchBytes, static_cast<half_t*>(out), nullptr, false);
}

int rwkv_hip_cmix_sparse_down_relu_one(rwkv_stream_t s, int fmt, int C, int F, const void* preact, const void* wt,
                                       const void* scale, void* workspace, size_t workspace_bytes, void* out) {
  return rwkv_hip_cmix_sparse_down_relu_rows(s, fmt, 1, C, F, preact, wt, scale, workspace, workspace_bytes, out);
}

}  // extern "C"
