// What the two files of the packed-weight GEMM share: the launch arguments and the exact expansion of int8 / int4 codes
// to fp16 (gemm_stream.hip: packing, dispatch, split-K reduce and the 64 x 256 tile; gemm_ring.hip: the LDS-ring tiles; gemm_tile.hip: the
// tiles of many rows).
#pragma once

#include "ops.h"

namespace rwkv {

typedef float float16_t __attribute__((ext_vector_type(16)));

struct StreamProblem {
  const half_t* x;
  const uint4_t* wp;
  const half_t* scale;
  const uint8_t* zp;
  void* y;
  float* partial;  // [splits][M][N] fp32, only with splits > 1
  int N;
  int fmt;
  int group_n, group_k;  // int4: scale and zero point of (column n, 128-group k) at n * group_n + k * group_k
};

// Up to kMaxProblems products that share M, K and the split (each with its own weights, format, x and y) in one
// launch: its column blocks run over all problems, block_end[] are the prefix sums.
struct StreamArgs {
  StreamProblem p[kMaxProblems];
  int block_end[kMaxProblems];
  int n_problems;
  int M, K;
  int splits, k_per_split;
  int row_tiles, col_blocks;
  int epilogue, out_f32;
  RowCopy copy;  // rides on the launch: its first blocks move these rows (they are no operand of the product)
};

// shared out between the first blocks of the launch (those with y == z == 0 among the first `blocks` of x, every one of which
// has to come here: a share nobody takes is never copied), so that no single block carries it on its critical path; called by
// the last `threads` of the block
__device__ __forceinline__ void ride_along_copy(const RowCopy& cp, unsigned blocks, unsigned threads) {
  constexpr unsigned kCopyBlocks = 8;
  const unsigned nb = blocks < kCopyBlocks ? blocks : kCopyBlocks;
  if (blockIdx.x < nb && blockIdx.y == 0 && blockIdx.z == 0 && cp.n > 0) {
    const unsigned t = threadIdx.x - (blockDim.x - threads);
    for (int i = (blockIdx.x * threads + t) * 8; i < cp.n; i += nb * threads * 8)
      *reinterpret_cast<uint4_t*>(cp.dst + i) = *reinterpret_cast<const uint4_t*>(cp.src + i);
  }
}

__device__ __forceinline__ half8_t make_half8(half2_t a, half2_t b, half2_t c, half2_t d) {
  half8_t r;
  r[0] = a[0]; r[1] = a[1]; r[2] = b[0]; r[3] = b[1];
  r[4] = c[0]; r[5] = c[1]; r[6] = d[0]; r[7] = d[1];
  return r;
}

// 8 int8 codes (two dwords) -> 8 fp16, exact: a conversion per code that reads the byte and writes the half in place.  (Bytes under the exponent of
// 1024, less the bias, take ten instructions; many rows of these products are bound by the chip's power: 16384 x 4096, 2048 rows, blocks of 256
// x 256 252 us so, 245 with eight conversions.  It ends in the two wait states that a product which reads the last of them needs: the compiler does
// not see these writes.)
__device__ __forceinline__ half8_t expand_w8(uint32_t d0, uint32_t d1) {
  uint4_t r;
#define RWKV_LOW(R, D, BYTE) "v_cvt_f16_i16_sdwa " R ", sext(" D ") dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:" BYTE "\n\t"
#define RWKV_HIGH(R, D, BYTE) "v_cvt_f16_i16_sdwa " R ", sext(" D ") dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:" BYTE "\n\t"
  asm(RWKV_LOW("%0", "%4", "BYTE_0") RWKV_LOW("%1", "%4", "BYTE_2") RWKV_LOW("%2", "%5", "BYTE_0") RWKV_LOW("%3", "%5", "BYTE_2")
      RWKV_HIGH("%0", "%4", "BYTE_1") RWKV_HIGH("%1", "%4", "BYTE_3") RWKV_HIGH("%2", "%5", "BYTE_1") RWKV_HIGH("%3", "%5", "BYTE_3") "s_nop 1"
      : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3])
      : "v"(d0), "v"(d1));
#undef RWKV_LOW
#undef RWKV_HIGH
  return __builtin_bit_cast(half8_t, r);
}

// 8 int4 codes (one dword, element 2i in the low nibble of byte i) minus the zero point -> 8 fp16, exact.
__device__ __forceinline__ half8_t expand_w4(uint32_t d, half2_t bias) {
  const uint32_t even = d & 0x0f0f0f0fu;
  const uint32_t odd = (d >> 4) & 0x0f0f0f0fu;
  return make_half8(as_half2(__builtin_amdgcn_perm(odd, even, 0x0c040c00u) | 0x64006400u) - bias,
                    as_half2(__builtin_amdgcn_perm(odd, even, 0x0c050c01u) | 0x64006400u) - bias,
                    as_half2(__builtin_amdgcn_perm(odd, even, 0x0c060c02u) | 0x64006400u) - bias,
                    as_half2(__builtin_amdgcn_perm(odd, even, 0x0c070c03u) | 0x64006400u) - bias);
}

__device__ __forceinline__ float finish_value(float v, int epilogue) {
  v = round_h(v);
  if (epilogue == RWKV_EPI_RELU_SQUARE) {
    v = fmaxf(v, 0.0f);
    v = round_h(v * v);
  }
  return v;
}

// gemm_ring.hip: the tile shapes of the LDS-ring kernel: 32 * mt rows, nb * wp bands of 32 columns, kc k per stage.
struct RingShape {
  int mt, nb, wp, kc;
};
constexpr RingShape kRingShapes[] = {{1, 1, 2, 128}, {1, 1, 2, 256}, {2, 1, 2, 256}, {2, 2, 2, 128}, {1, 1, 4, 128}, {2, 1, 4, 128}, {4, 1, 2, 128}, {4, 1, 4, 128}};
// fmt: the format of the launch's problems; mixed: fp16 problems among them, with half as many columns per block
bool gemm_ring_has(const RingShape& shape, int fmt, bool mixed);
int gemm_ring_launch(hipStream_t st, const RingShape& shape, int fmt, bool mixed, const StreamArgs& g);
// gemm_tile.hip: blocks of 128 or 256 rows x 256 columns for many rows; int8 and fp16 problems
int gemm_tile_launch(hipStream_t st, int rows, const StreamArgs& g);

}  // namespace rwkv
