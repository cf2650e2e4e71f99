// What the grouped-GEMM kernels share: a launch's parameters and the weights' conversion to matrix-core operands.
#pragma once

#include <type_traits>
#include <utility>

#include "common.h"

namespace dew {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
typedef __attribute__((ext_vector_type(2))) float f32x2_t;
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;  // a 16-byte register quad (native vector: stays in VGPRs)
typedef __attribute__((ext_vector_type(8))) int i32x8_t;       // an operand of the scaled matrix instruction
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;

struct BankView {
  const uint8_t* codes;
  const void* scales;
  const float* tensor_scale;
};

struct GemmParams {
  const bf16_t* x;
  const int32_t* gather;
  const int32_t* offsets;  // [experts + 1] exclusive prefix of the group sizes, or null where `sizes` is given
  const int32_t* sizes;    // [experts] group sizes as jax.lax.ragged_dot takes them: the prefix is then formed in the tile search
  const int32_t* scatter;
  BankView w0, w1;
  bf16_t* out;
  const uint8_t* a_scale;  // split activations: each source row's e8m0 scale, or its row of block_scale_pitch(depth) of them
  uint8_t* out_scale;      // split output: each written row's block_scale_pitch(width) e8m0 scales, one for 128 columns
  const float* bias;  // [experts, width] fp32, or null
  int round_bias;     // the bias is a parameter of a bf16 product: rounded to bf16 as it is read (a quantized-rows recipe's stays fp32)
  float limit;        // the interleaved gated epilogue's clamp; a paired launch's (0: none)
  int gating;         // a paired launch's gate: DEW_MOE_GATE_SILU (SwiGLU) or DEW_MOE_GATE_GELU_TANH (GeGLU)
  int experts, depth, width, rows, m_tile_bound;
  // A launch normally multiplies every group in tiles of its BM rows, the last of a group partly empty. Where that
  // waste matters two launches share the groups: the taller tiles' launch leaves a last tile that would hold at most
  // skip_tails rows to a launch of tiles that many rows tall, which multiplies (tail_of = the taller tile's rows)
  // only those last rows, the ones past a group's whole tiles of tail_of rows where they are at most its own BM.
  int skip_tails, tail_of;
  // A kernel gradient (kFormatMxFp8Window): every group multiplies the same window_rows rows over its own window of
  // the depth, tokens windows[g] .. windows[g + 1] in whole 128s; `depth` is then all the tokens.
  const int32_t* windows;
  int window_rows;
  float* out_f32;  // the product in fp32 (kPlainF32) instead of `out`
  int group_m;     // m-tiles of a chunk of 8 group_m tiles that one XCD's resident blocks cover together (set by launch_tile)
  const float* factor0;  // a kernel gradient's fp32 sums times *factor0 * *factor1 before the rounding (each may be null):
  const float* factor1;  // the tensor scales of NVFP4 operands
};

// What the epilogue writes: the rounded product (plus bias); SwiGLU of two banks' products; for one bank whose
// columns interleave gate (even) and up (odd), the clamped quick-GELU gating of each column pair; or the SwiGLU of
// two banks' products already split into two e4m3 terms under one scale per row and 128 columns, which is what the
// next product's scaled matrix instructions read (kFormatMxSplitBlocks).
enum Epilogue { kPlain = 0, kSwigluOfTwo = 1, kInterleavedGated = 2, kSwigluOfTwoSplit = 3, kPlainF32 = 4 };

__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  bf16x2_t pair = {static_cast<__bf16>(a), static_cast<__bf16>(b)};
  return __builtin_bit_cast(uint32_t, pair);
}

// Eight e4m3 codes (two dwords) times one fp32 scale -> one bf16x8 fragment: bf16(f32(code) * scale), the
// value the reference's dequantize-then-cast produces (src/dew/interop/codecs.py:670-703; gemm.py:1067-1071).
__device__ __forceinline__ bf16x8_t fragment_fp8(uint32_t w0, uint32_t w1, float scale) {
  const f32x2_t a = __builtin_amdgcn_cvt_pk_f32_fp8(w0, false), b = __builtin_amdgcn_cvt_pk_f32_fp8(w0, true);
  const f32x2_t c = __builtin_amdgcn_cvt_pk_f32_fp8(w1, false), d = __builtin_amdgcn_cvt_pk_f32_fp8(w1, true);
  return __builtin_bit_cast(bf16x8_t, u32x4_t{pack_bf16(a.x * scale, a.y * scale), pack_bf16(b.x * scale, b.y * scale),
                                              pack_bf16(c.x * scale, c.y * scale), pack_bf16(d.x * scale, d.y * scale)});
}

// Eight E2M1 nibbles (one dword) under one e4m3 block scale already over 2^8 -> one bf16x8 fragment; each
// product code * scale / 2^8 is exact in bf16 (src/dew/nn/kernels/formats.py:108-113).
__device__ __forceinline__ bf16x8_t fragment_fp4(uint32_t word, float scale) {
  const f32x2_t a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 0), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 1);
  const f32x2_t c = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 2), d = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 3);
  return __builtin_bit_cast(bf16x8_t, u32x4_t{pack_bf16(a.x * scale, a.y * scale), pack_bf16(b.x * scale, b.y * scale),
                                              pack_bf16(c.x * scale, c.y * scale), pack_bf16(d.x * scale, d.y * scale)});
}

// The same for a bank whose block scales are all powers of two (an MXFP4 checkpoint's): the hardware
// conversion applies the scale's exponent itself, one instruction for two codes, exactly.
__device__ __forceinline__ bf16x8_t fragment_fp4_pow2(uint32_t word, float scale) {
  return __builtin_bit_cast(bf16x8_t, u32x4_t{
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 0)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 1)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 2)),
      __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(word, scale, 3))});
}

// The same eight codes as f16 values times the block scale itself (an e4m3 value is exact in f16, and so is its product
// with an E2M1 code): one packed conversion and one packed multiply for two codes.
__device__ __forceinline__ bf16x8_t fragment_fp4_f16(uint32_t word, _Float16 scale) {
  const f16x2_t both = {scale, scale};
  const f16x2_t a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 0) * both, b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 1) * both;
  const f16x2_t c = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 2) * both, d = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(word, 1.0f, 3) * both;
  return __builtin_bit_cast(bf16x8_t, u32x4_t{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                              __builtin_bit_cast(uint32_t, c), __builtin_bit_cast(uint32_t, d)});
}

// f(integral_constant<0>), ..., f(integral_constant<N - 1>): a loop whose index is a constant expression in its body.
template <class F, int... Is>
__device__ __forceinline__ void static_for_each(std::integer_sequence<int, Is...>, F&& f) {
  (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_each(std::make_integer_sequence<int, N>{}, f);
}

constexpr int BK = 64;
constexpr int kChunksPerRow = BK / 8;  // 16-byte chunks in an LDS row
constexpr int kMaxDepthBlocks = 256;   // FP8 128 x 128 blocks: depth up to 32768

// LDS index of 16-byte chunk `chunk` of row `row` (128-byte rows). The chunk is xor-swizzled by
// f(row) = ((row >> 1) & 7) ^ ((row & 1) << 2), chosen against the measured service order of gfx950's LDS:
// ds_read_b128 serves 16 lanes a pass over 64 banks, the passes being lanes {0-3,12-15,20-23,24-27},
// {4-7,8-11,16-19,28-31} and the same + 32; ds_write_b128 serves 8 consecutive lanes a pass over 128 bytes.
// With lane = row (mod 32) on the read side, f is injective on every read pass's rows of one parity, and a
// store pass writes the 8 chunks of one row, so fragment reads and stores are conflict-free.
__device__ __forceinline__ int swizzled(int row, int chunk) {
  return row * kChunksPerRow + (chunk ^ (((row >> 1) & 7) ^ ((row & 1) << 2)));
}

// f(integral_constant<B>), f(integral_constant<B + 1>), ...: a loop whose index is a constant expression in its body.
template <int B, int... Is, class F>
__device__ __forceinline__ void static_range(std::integer_sequence<int, Is...>, F&& f) {
  (f(std::integral_constant<int, B + Is>{}), ...);
}

// An inclusive sum over the lanes, by lane moves of the vector unit (a sixth of the time of as many trips through the LDS).
__device__ __forceinline__ int lanes_scanned(int value) {
  value += __builtin_amdgcn_update_dpp(0, value, 0x111, 0xF, 0xF, false);  // row_shr:1
  value += __builtin_amdgcn_update_dpp(0, value, 0x112, 0xF, 0xF, false);  // row_shr:2
  value += __builtin_amdgcn_update_dpp(0, value, 0x114, 0xF, 0xF, false);  // row_shr:4
  value += __builtin_amdgcn_update_dpp(0, value, 0x118, 0xF, 0xF, false);  // row_shr:8
  value += __builtin_amdgcn_update_dpp(0, value, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1, 3
  value += __builtin_amdgcn_update_dpp(0, value, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2, 3
  return value;
}

// The launch for few tiles of few rows (decode.hip); `mode`: kPlain, kSwigluOfTwo or kInterleavedGated.
int launch_few_tiles(const char* who, const GemmParams& p, int format, int mode, hipStream_t stream);

constexpr int kMostCombinedSlots = 8;  // wavefronts of a block: more have no registers for eight steps of weights each in flight
// The down product and the combine as one launch (decode.hip); `p.scatter`: the sorted positions' slots, `p.rows` of them.
int launch_few_combined(const char* who, const GemmParams& p, int format, const float* weights, int tokens, int top_k, bool shared, void* out,
                        hipStream_t stream);

// The launch in tiles of up to 256 rows on eight wavefronts (tall.hip); of FP8 block or bf16 banks, one or two (gate and up,
// gated), or of one FP8 channel or NVFP4 bank.
int launch_tall(const char* who, const GemmParams& p, int format, bool paired, hipStream_t stream);

}  // namespace dew
