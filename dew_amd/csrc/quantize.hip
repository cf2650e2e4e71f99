// Activation rows quantized for the blockwise FP8 recipe (DeepSeek-V3's): e4m3 codes a 1 x 128 tile at a time
// along the depth under one power-of-two scale a tile (reference src/dew/nn/kernels/projections.py:176-182 over
// src/dew/nn/fake_quant.py:117-128, 48-76): amax floored at 1e-4, scale = the least power of two >= amax * f32(1 / 448)
// (read off the product's fp32 bits: its exponent, plus one where any fraction bit is set), code = e4m3(x / scale),
// ties to even; the quotient by a power of two is exact and lies within +-448 by the scale's choice.
// The codes are written in the order the scaled matrix instruction reads its 8-bit operand, so that the grouped
// GEMM copies rows into the LDS as they are: of each 128 depths, byte 16 (4 g + 2 t + h) + b holds depth
// 64 t + 32 h + 16 g + b (t the 64-deep half, g the instruction's lane group, h the half of the group's 32 bytes).
// The scales are kept as their e8m0 bytes, block_scale_pitch(depth) a row (one byte per 128 depths, padded to 16).
// HBM-bound: 2 bytes read and 1 written per element.
#include "common.h"
#include "nvfp4.h"

namespace dew {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
typedef __attribute__((ext_vector_type(2))) uint32_t u32x2_t;

constexpr int kQuantizeWaves = 4;  // wavefronts a 256-thread block

// What eight neighbouring lanes hold, taken together by `both` (which lane holds what must not matter).
template <class Both>
__device__ __forceinline__ uint32_t over_eight(uint32_t v, Both both) {
  v = both(v, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, true)));   // quad_perm 1 0 3 2
  v = both(v, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, true)));   // quad_perm 2 3 0 1
  return both(v, static_cast<uint32_t>(__builtin_amdgcn_mov_dpp(v, 0x141, 0xF, 0xF, true)));  // row_half_mirror
}

// MX: the MXFP8 recipe's rows (OCP MX; reference src/dew/nn/kernels/formats.py:186-229): e4m3 codes under one E8M0 scale
// every 32 depths, the scale 2 to the largest magnitude's binary exponent less 8 (its fp32 exponent field less 8 is
// the byte; a block of zeros, or one whose largest magnitude lies under 2^-119, takes byte 0), each value over its
// scale rounded to e4m3, ties to even, saturating at +-448. Codes in the same operand order as above; the scale
// bytes in depth order, depth / 32 a row (a 128-deep step's four bytes are one aligned dword).
//
// Rows are whole 128s, so the operand is one run of 128-deep tiles: eight lanes a tile, 16 depths each, which are 16 bytes of the operand
// order, ITEMS such pieces a lane with all their loads in flight: two where that leaves four blocks a CU, more gave nothing. Bound by memory, 2 bytes read
// and 1 written an element. (A wavefront a row, 8 depths a lane, had one load in flight and stored 8 bytes.) Measured (us, FP8, operands that the last-level
// cache holds and ones it has lost): 4096 x 2048 4.7 and 8.8 -> 4.1 and 5.8, 8192 x 4096 16.5 and 27.6 -> 15.5 and 25.1, 32 768 x 7168 136 and 159 -> 124 and 149 (5.7 TB/s).
template <bool MX, int ITEMS>
__global__ __launch_bounds__(64 * kQuantizeWaves) void quantize_rows_kernel(const bf16_t* __restrict__ x, uint8_t* __restrict__ codes, uint8_t* __restrict__ scales,
                                                                          long long pieces, uint32_t row_tiles, uint32_t pitch) {
  const long long first = static_cast<long long>(blockIdx.x) * (64 * kQuantizeWaves * ITEMS) + threadIdx.x;
  u32x4_t words[ITEMS][2];
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const u32x4_t* source = reinterpret_cast<const u32x4_t*>(x) + 2 * min(first + 64 * kQuantizeWaves * k, pieces - 1);
    words[k][0] = source[0];
    words[k][1] = source[1];
  }
#pragma unroll
  for (int k = 0; k < ITEMS; ++k) {
    const long long piece = first + 64 * kQuantizeWaves * k;
    if (piece >= pieces) return;  // (eight lanes of a tile together)
    float v[16];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[2 * i] = __uint_as_float(words[k][i / 4][i % 4] << 16);
      v[2 * i + 1] = __uint_as_float(words[k][i / 4][i % 4] & 0xFFFF0000u);
    }
    float most = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) most = fmaxf(most, fabsf(v[i]));
    const int within = threadIdx.x % 8;
    const uint32_t tile = static_cast<uint32_t>(piece / 8);
    uint32_t byte;
    if constexpr (MX) {
      most = fmaxf(most, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(most), 0xB1, 0xF, 0xF, true)));
      byte = static_cast<uint32_t>(min(max(static_cast<int>(__float_as_uint(most) >> 23) - 8, 0), 254));  // (0 for a zero or subnormal magnitude; <= 247 for finite rows)
      const uint32_t four = over_eight(byte << (8 * (within / 2)), [](uint32_t a, uint32_t b) { return a | b; });
      if (within == 0) reinterpret_cast<uint32_t*>(scales)[tile] = four;
    } else {
      // (a magnitude's bits order as it does, and none here is a NaN: fmaxf left it out)
      most = __uint_as_float(over_eight(__float_as_uint(most), [](uint32_t a, uint32_t b) { return max(a, b); }));
      const uint32_t bits = __float_as_uint(fmaxf(most, 1e-4f) * 0x1.24924ap-9f);  // f32(1 / 448)
      byte = min(max((bits >> 23) + ((bits & 0x7FFFFFu) != 0u ? 1u : 0u), 1u), 253u);
      if (within == 0) scales[static_cast<size_t>(tile / row_tiles) * pitch + tile % row_tiles] = static_cast<uint8_t>(byte);
    }
    const float inverse = __uint_as_float((254u - byte) << 23);  // 1 / scale, exactly
    u32x4_t packed;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      float q[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[i] = v[4 * w + i] * inverse;
        if (MX) q[i] = fminf(fmaxf(q[i], -448.0f), 448.0f);
      }
      packed[w] = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
      packed[w] = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], packed[w], true);
    }
    const int half = within / 4, low = within % 4 / 2, group = within % 2;
    *reinterpret_cast<u32x4_t*>(codes + static_cast<size_t>(tile) * 128 + 16 * (4 * group + 2 * half + low)) = packed;
  }
}

template <bool MX>
static int quantize_rows(const char* who, const void* x, void* codes, uint8_t* scales, int rows, int depth, void* stream) {
  DEW_REQUIRE(rows >= 0 && depth >= 128 && depth % 128 == 0, "%s: rows %d, depth %d (whole 128s)", who, rows, depth);
  if (rows == 0) return DEW_MOE_OK;
  DEW_REQUIRE(x && codes && scales, "%s: x, codes and scales must not be null", who);
  DEW_REQUIRE(aligned16(x) && aligned16(codes) && aligned16(scales), "%s: x, codes and scales must be 16-byte aligned", who);
  constexpr int kMany = 2, kThreads = 64 * kQuantizeWaves;
  const long long pieces = static_cast<long long>(rows) * depth / 16;
  const bool many = pieces >= 4ll * 256 * kThreads * kMany;
  const long long blocks = (pieces + kThreads * (many ? kMany : 1) - 1) / (kThreads * (many ? kMany : 1));
  DEW_REQUIRE(blocks < (1ll << 31) && pieces / 8 < (1ll << 32), "%s: %d rows of %d", who, rows, depth);
  hipLaunchKernelGGL((many ? quantize_rows_kernel<MX, kMany> : quantize_rows_kernel<MX, 1>), dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), static_cast<const bf16_t*>(x), static_cast<uint8_t*>(codes), scales, pieces,
                     static_cast<uint32_t>(depth / 128), static_cast<uint32_t>((depth / 128 + 15) / 16 * 16));
  return launched("quantize_rows_kernel");
}

// The NVFP4 recipe's rows (reference src/dew/nn/kernels/formats.py:263-274 over src/dew/algebra/bits.py:941-982):
// E2M1 codes under an E4M3 scale every 16 depths and one tensor scale over the whole operand. The scaled matrix
// instruction takes power-of-two scales of 32 depths only, so this operand goes to the bf16 instruction: each value is
// written as what it stands for short of the tensor scale, code x block scale, which bf16 holds exactly (5 significant
// bits), and the product applies the tensor scale to its fp32 sums with the bank's.
// Two passes, because the tensor scale needs the whole operand's largest magnitude first.
__global__ __launch_bounds__(256) void absmax_clear_kernel(uint32_t* __restrict__ largest) { *largest = 0u; }

__global__ __launch_bounds__(256) void absmax_kernel(const bf16_t* __restrict__ x, long long chunks, uint32_t* __restrict__ largest) {
  uint32_t mine = 0;  // magnitudes of bf16 values order as their bit patterns do
  const long long stride = static_cast<long long>(gridDim.x) * blockDim.x;
  long long chunk = static_cast<long long>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; chunk + 7 * stride < chunks; chunk += 8 * stride) {  // eight loads in flight a lane
    u32x4_t words[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) words[k] = reinterpret_cast<const u32x4_t*>(x)[chunk + k * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) mine = max(mine, max(words[k][i] & 0x7FFFu, (words[k][i] >> 16) & 0x7FFFu));
  }
  for (; chunk < chunks; chunk += stride) {
    const u32x4_t words = reinterpret_cast<const u32x4_t*>(x)[chunk];
#pragma unroll
    for (int i = 0; i < 4; ++i) mine = max(mine, max(words[i] & 0x7FFFu, (words[i] >> 16) & 0x7FFFu));
  }
#pragma unroll
  for (int offset = 32; offset >= 1; offset >>= 1) mine = max(mine, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mine), offset, 64)));
  // One atomic a block, and none where the word already holds as much: on one address they are served one after another, some
  // 10 ns each (one a wavefront of 4096 blocks took 190 us whatever the operand's size).
  __shared__ uint32_t waves[4];
  if (threadIdx.x % 64 == 0) waves[threadIdx.x / 64] = mine;
  __syncthreads();
  if (threadIdx.x == 0) {
    mine = max(max(waves[0], waves[1]), max(waves[2], waves[3])) << 16;  // (as fp32 bits)
    if (mine > __hip_atomic_load(largest, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicMax(largest, mine);
  }
}

// `count` partial magnitudes; `bank_scales` (or null): the `experts` tensor scales of the bank these rows will multiply, which leave times
// the rows' own as `products`. The blocks stay for row after row: what each first makes of the partials it makes once.
__global__ __launch_bounds__(64 * kQuantizeWaves) void quantize_rows_nvfp4_kernel(const bf16_t* __restrict__ x, const uint32_t* __restrict__ largest, int count,
                                                                                bf16_t* __restrict__ out, float* __restrict__ tensor_scale,
                                                                                const float* __restrict__ bank_scales, float* __restrict__ products,
                                                                                int experts, int rows, int depth) {
  const float top = nvfp4_top(nvfp4_share(largest, count));
  const float tensor = nvfp4_tensor_scale(top);
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) *tensor_scale = tensor;
    if (bank_scales)
      for (int e = threadIdx.x; e < experts; e += blockDim.x) products[e] = bank_scales[e] * tensor;
  }
  const bool quick = nvfp4_in_range(top, tensor);  // (the same for the whole launch)
  const float inverse_tensor = 1.0f / tensor;
  const int lane = threadIdx.x % 64;
  for (int row = blockIdx.x * kQuantizeWaves + threadIdx.x / 64; row < rows; row += gridDim.x * kQuantizeWaves) {
    const bf16_t* source = x + static_cast<size_t>(row) * depth;
    bf16_t* target = out + static_cast<size_t>(row) * depth;
    for (int chunk = lane; chunk < depth / 8; chunk += 64) {  // 8 depths a lane, 2 lanes a block of 16
      const u32x4_t words = *reinterpret_cast<const u32x4_t*>(source + chunk * 8);
      float v[8];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(words[i] << 16);
        v[2 * i + 1] = __uint_as_float(words[i] & 0xFFFF0000u);
      }
      float block = 0.0f;
#pragma unroll
      for (int i = 0; i < 8; ++i) block = fmaxf(block, fabsf(v[i]));
      block = fmaxf(block, __shfl_xor(block, 1, 64));
      const float each = nvfp4_block_scale(block, tensor);
      u32x4_t packed;
      if (quick) {
        const Nvfp4Scales by{tensor, inverse_tensor, each, nvfp4_inverse(each)};
#pragma unroll
        for (int i = 0; i < 4; ++i) packed[i] = by.values(v[2 * i], v[2 * i + 1]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) packed[i] = nvfp4_values_divided(v[2 * i], v[2 * i + 1], tensor, each);
      }
      *reinterpret_cast<u32x4_t*>(target + chunk * 8) = packed;
    }
  }
}

// The operands of a step's gradients, x [tokens, dim] quantized ALONG THE TOKENS where it lies (the kernel gradient of dense operands
// contracts the tokens of both as they are: no transposed copy), and, ROWS, along its rows too from the same read, which the cotangent's
// other product takes. A thread owns 16 tokens x 4 columns: a block of each column, and a quarter of a block of each row, the others three
// neighbouring lanes' (8 columns a thread took
// 256 registers, one wavefront a SIMD: 34 M elements 139 us, 47 here; tokens alone, 17 M, 29 and 17). The arithmetic of quantize_rows_nvfp4_kernel.
// Bound by memory: 2 bytes read and 2 (ROWS: 4) written an element.
template <bool ROWS>
__global__ __launch_bounds__(256) void quantize_tokens_nvfp4_kernel(const bf16_t* __restrict__ x, const uint32_t* __restrict__ largest,
                                                                    bf16_t* __restrict__ rows_out, bf16_t* __restrict__ tokens_out,
                                                                    float* __restrict__ tensor_scale, const float* __restrict__ bank_scales,
                                                                    float* __restrict__ products, int experts, int tokens, int dim) {
  const uint32_t share = nvfp4_share(largest, kNvfp4Partials);
  const long long item = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x, items = static_cast<long long>(tokens / 16) * (dim / 4);
  const long long mine = item < items ? item : items - 4 + item % 4;  // (past the end: the last four's again, which store the same)
  const int chunks = dim / 4;  // (whole 32s: four lanes are of the same tokens)
  const size_t at = static_cast<size_t>(mine / chunks) * 16 * dim + mine % chunks * 4;
  u32x2_t words[16];
#pragma unroll
  for (int t = 0; t < 16; ++t) words[t] = *reinterpret_cast<const u32x2_t*>(x + at + static_cast<size_t>(t) * dim);
  const float top = nvfp4_top(share);
  const float tensor = nvfp4_tensor_scale(top), inverse_tensor = 1.0f / tensor;
  const bool quick = nvfp4_in_range(top, tensor);  // (the same for the whole launch)
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) *tensor_scale = tensor;
    if (ROWS && bank_scales)
      for (int e = threadIdx.x; e < experts; e += 256) products[e] = bank_scales[e] * tensor;
  }
  auto low = [](uint32_t word) { return __uint_as_float(word << 16); };
  auto high = [](uint32_t word) { return __uint_as_float(word & 0xFFFF0000u); };
  auto scales = [&](float block) {
    const float each = nvfp4_block_scale(block, tensor);
    return Nvfp4Scales{tensor, inverse_tensor, each, nvfp4_inverse(each)};
  };
  if (!quick) {  // an operand with a NaN, an infinity or a scale out of range: read again, value by value
    if constexpr (ROWS) {
#pragma unroll 1
      for (int t = 0; t < 16; ++t) {
        const u32x2_t word = *reinterpret_cast<const u32x2_t*>(x + at + static_cast<size_t>(t) * dim);
        float block = fmaxf(fmaxf(fabsf(low(word[0])), fabsf(high(word[0]))), fmaxf(fabsf(low(word[1])), fabsf(high(word[1]))));
        block = fmaxf(block, __shfl_xor(block, 1, 64));
        block = fmaxf(block, __shfl_xor(block, 2, 64));
        const float each = nvfp4_block_scale(block, tensor);
        *reinterpret_cast<u32x2_t*>(rows_out + at + static_cast<size_t>(t) * dim) =
            u32x2_t{nvfp4_values_divided(low(word[0]), high(word[0]), tensor, each), nvfp4_values_divided(low(word[1]), high(word[1]), tensor, each)};
      }
    }
#pragma unroll 1
    for (int c = 0; c < 4; ++c) {
      float block = 0.0f;
#pragma unroll 1
      for (int t = 0; t < 16; ++t) block = fmaxf(block, fabsf(bf16_to_f32(x[at + static_cast<size_t>(t) * dim + c])));
      const float each = nvfp4_block_scale(block, tensor);
#pragma unroll 1
      for (int t = 0; t < 16; ++t) {
        const size_t place = at + static_cast<size_t>(t) * dim + c;
        tokens_out[place] = static_cast<bf16_t>(nvfp4_values_divided(bf16_to_f32(x[place]), 0.0f, tensor, each));
      }
    }
    return;
  }
  if constexpr (ROWS) {
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float block = fmaxf(fmaxf(fabsf(low(words[t][0])), fabsf(high(words[t][0]))), fmaxf(fabsf(low(words[t][1])), fabsf(high(words[t][1]))));
      block = fmaxf(block, __shfl_xor(block, 1, 64));
      block = fmaxf(block, __shfl_xor(block, 2, 64));
      const Nvfp4Scales by = scales(block);
      const u32x2_t packed = {by.values(low(words[t][0]), high(words[t][0])), by.values(low(words[t][1]), high(words[t][1]))};
      *reinterpret_cast<u32x2_t*>(rows_out + at + static_cast<size_t>(t) * dim) = packed;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {  // two columns
    float first = 0.0f, second = 0.0f;
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      first = fmaxf(first, fabsf(low(words[t][i])));
      second = fmaxf(second, fabsf(high(words[t][i])));
    }
    const Nvfp4Scales by_first = scales(first), by_second = scales(second);
#pragma unroll
    for (int t = 0; t < 16; t += 2) {
      const uint32_t a = by_first.values(low(words[t][i]), low(words[t + 1][i])), b = by_second.values(high(words[t][i]), high(words[t + 1][i]));
      words[t][i] = __builtin_amdgcn_perm(b, a, 0x05040100u);
      words[t + 1][i] = __builtin_amdgcn_perm(b, a, 0x07060302u);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int t = 0; t < 16; ++t) *reinterpret_cast<u32x2_t*>(tokens_out + at + static_cast<size_t>(t) * dim) = words[t];
}

// Operands' partial largest magnitudes, bf16 or fp32, a partial a block: blockIdx.y is the operand. A step quantizes two or three operands, whose
// magnitudes one launch forms side by side: 8192 rows' step on 8 x 2048 x 4096 had five launches of 8 to 26 us, 89 in all, and has two.
constexpr int kMostOperands = 3;
struct LargestOperands {
  const u32x4_t* x[kMostOperands];
  long long chunks[kMostOperands];
  int f32[kMostOperands];
};
template <bool F32>
__device__ __forceinline__ uint32_t largest_of(const u32x4_t* __restrict__ x, long long chunks) {
  uint32_t mine = 0;
  auto take = [&](const u32x4_t& words) {
#pragma unroll
    for (int i = 0; i < 4; ++i) mine = F32 ? max(mine, words[i] & 0x7FFFFFFFu) : max(mine, max((words[i] << 16) & 0x7FFF0000u, words[i] & 0x7FFF0000u));
  };
  const long long stride = static_cast<long long>(gridDim.x) * 256;
  long long chunk = static_cast<long long>(blockIdx.x) * 256 + threadIdx.x;
  for (; chunk + 7 * stride < chunks; chunk += 8 * stride) {  // eight loads in flight a lane
    u32x4_t words[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) words[k] = x[chunk + k * stride];
#pragma unroll
    for (int k = 0; k < 8; ++k) take(words[k]);
  }
  for (; chunk < chunks; chunk += stride) take(x[chunk]);
  return mine;
}
__global__ __launch_bounds__(256) void nvfp4_largest_kernel(LargestOperands of, uint32_t* __restrict__ partials) {
  const int operand = blockIdx.y;
  uint32_t mine = of.f32[operand] ? largest_of<true>(of.x[operand], of.chunks[operand]) : largest_of<false>(of.x[operand], of.chunks[operand]);
#pragma unroll
  for (int offset = 32; offset >= 1; offset >>= 1) mine = max(mine, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mine), offset, 64)));
  __shared__ uint32_t waves[4];
  if (threadIdx.x % 64 == 0) waves[threadIdx.x / 64] = mine;
  __syncthreads();
  if (threadIdx.x == 0) partials[operand * kNvfp4Partials + blockIdx.x] = max(max(waves[0], waves[1]), max(waves[2], waves[3]));
}

// A kernel gradient's operands: x [tokens, dim] quantized ALONG THE TOKENS and written transposed, for the product
// that contracts each group's tokens (reference src/dew/nn/kernels/projections.py:211-224 `rows_quantized(x.T)`, and
// :263-275 `MxFp8.quantized(x.T)`). MX false: the blockwise FP8 recipe's 1 x 128 tiles (128 tokens of one column under
// the scale rule of quantize_rows_kernel, its byte written for each of the tile's four 32-token blocks); MX true: OCP
// MX blocks of 32 tokens (its MX rule).
//
// As the lhs_t operand, rows of tokens: codes [dim, tokens] in the row operand's order within each 128 tokens (see the head of this
// file) and scales [dim, tokens / 32]. A block takes 128 tokens x 64 columns through the LDS: thread (column c, quarter a) owns the
// 32 tokens of block a. HBM-bound: 2 bytes read and 1 written per element.
template <bool MX>
__global__ __launch_bounds__(256) void quantize_columns_kernel(const bf16_t* __restrict__ x, uint8_t* __restrict__ codes,
                                                               uint32_t* __restrict__ scales, int tokens, int dim) {
  __shared__ uint32_t tile[128][33];     // 128 tokens x 64 columns of bf16, a dword of padding a row
  __shared__ float quarter_amax[4][64];
  __shared__ uint32_t scale_word[64];    // a column's four scale bytes
  __shared__ u32x4_t staged[64][8];      // the lhs_t operand's 64 rows of 128 bytes, chunk xor-swizzled by the row
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * 128, d0 = blockIdx.y * 64;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int item = tid + 256 * k, row = item / 8, chunk = item % 8;
    const u32x4_t words = *reinterpret_cast<const u32x4_t*>(x + static_cast<size_t>(t0 + row) * dim + d0 + chunk * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) tile[row][chunk * 4 + i] = words[i];
  }
  if (tid < 64) scale_word[tid] = 0;
  __syncthreads();
  const int c = tid % 64, quarter = tid / 64;
  float v[32];
  float largest = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const uint32_t word = tile[32 * quarter + i][c / 2];
    v[i] = __uint_as_float(c % 2 ? word & 0xFFFF0000u : word << 16);
    largest = fmaxf(largest, fabsf(v[i]));
  }
  uint32_t byte;
  if constexpr (MX) {
    const int field = static_cast<int>(__float_as_uint(largest) >> 23);
    byte = static_cast<uint32_t>(min(max(field - 8, 0), 254));
  } else {
    quarter_amax[quarter][c] = largest;
    __syncthreads();
    const float amax = fmaxf(fmaxf(quarter_amax[0][c], quarter_amax[1][c]), fmaxf(quarter_amax[2][c], quarter_amax[3][c]));
    const uint32_t bits = __float_as_uint(fmaxf(amax, 1e-4f) * 0x1.24924ap-9f);  // f32(1 / 448)
    byte = min(max((bits >> 23) + ((bits & 0x7FFFFFu) != 0u ? 1u : 0u), 1u), 253u);
  }
  const float inverse = __uint_as_float((254u - byte) << 23);
  uint32_t packed[8];
#pragma unroll
  for (int w = 0; w < 8; ++w) {
    float q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = MX ? fminf(fmaxf(v[4 * w + i] * inverse, -448.0f), 448.0f) : v[4 * w + i] * inverse;
    packed[w] = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
    packed[w] = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], packed[w], true);
  }
  atomicOr(&scale_word[c], byte << (8 * quarter));
  const u32x4_t low = {packed[0], packed[1], packed[2], packed[3]}, high = {packed[4], packed[5], packed[6], packed[7]};
  // tokens 32 a + 16 g + b of the 128 sit at byte 16 (4 g + a) + b
  staged[c][quarter ^ (c & 7)] = low;
  staged[c][(4 + quarter) ^ (c & 7)] = high;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int item = tid + 256 * k, row = item / 8, chunk = item % 8;
    *reinterpret_cast<u32x4_t*>(codes + static_cast<size_t>(d0 + row) * tokens + t0 + chunk * 16) = staged[row][chunk ^ (row & 7)];
  }
  if (tid < 64) scales[static_cast<size_t>(d0 + tid) * (tokens / 128) + t0 / 128] = scale_word[tid];
}

// As the rhs_t operand (or either operand of the launch that takes two such), a prepared MXFP8 bank of one expert, depth = tokens, width =
// dim: codes as 32 column x 32 token atoms [dim / 32][tokens / 32][64 lanes][16 bytes] (lane 32 g + c holds tokens 16 g .. 16 g + 15 of
// column c) and scales [dim / 32][tokens / 128][32 columns][4 bytes]; and, ROWS, along its rows too from the same read, which the
// cotangent's other product takes (quantize_rows_kernel's bytes). A block takes 128 tokens x 128
// columns: eight neighbours of a row a thread as they arrive, for the rows; then, through the LDS, 16 tokens of two neighbouring columns,
// whose codes are 32 bytes of an atom. Every XCD's blocks walk along the columns of its own tokens, so that the few bytes of scales that a
// block writes of a row meet in that XCD's L2. HBM-bound: 2 bytes read and 1 (ROWS: 2) written an element, at 4.8 to 5.8 TB/s. Measured (us): a
// cotangent both ways, MXFP8, 32 768 x 14 336 567 by a launch each way, 368 here, FP8, 32 768 x 2048 80 and 46; along the tokens alone (once 128
// tokens x 64 columns a block, a half word of the LDS a read) 32 768 x 4096 96 -> 80, 32 768 x 2048 45 -> 39, 32 768 x 14 336 274 -> 271.
template <bool MX, bool ROWS>
__global__ __launch_bounds__(512) void quantize_bank_kernel(const bf16_t* __restrict__ x, uint8_t* __restrict__ codes, uint32_t* __restrict__ scales,
                                                            uint8_t* __restrict__ row_codes, uint8_t* __restrict__ row_scales, int tokens, int dim,
                                                            int pitch) {
  constexpr int kRow = 68;              // dwords of a row of 128 columns as it is staged
  __shared__ u32x4_t tile[128 * kRow / 4];
  __shared__ float largest[8][128];     // of 16 tokens of a column
  const int tid = threadIdx.x, across = dim / 128, tiles = tokens / 128 * across, run = (tiles + 7) / 8;
  const int at = blockIdx.x % 8 * run + blockIdx.x / 8;  // (workgroup b runs on XCD b mod 8)
  if (at >= tiles) return;
  const int t0 = at / across * 128, d0 = at % across * 128;
  const int chunk = tid % 16;
  // Read once, non-temporal (a blockwise step of 32 768 rows 2156 -> 2137 us, steps of 100 to 400 us 0 to 2 %).
  u32x4_t words[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) words[k] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(x + static_cast<size_t>(t0 + tid / 16 + 32 * k) * dim + d0 + chunk * 8));
  auto low = [](uint32_t word) { return __uint_as_float(word << 16); };
  auto high = [](uint32_t word) { return __uint_as_float(word & 0xFFFF0000u); };
  auto scale_byte = [](float most) -> uint32_t {
    if (MX) return min(max(static_cast<int>(__float_as_uint(most) >> 23) - 8, 0), 254);
    const uint32_t bits = __float_as_uint(fmaxf(most, 1e-4f) * 0x1.24924ap-9f);  // f32(1 / 448)
    return min(max((bits >> 23) + ((bits & 0x7FFFFFu) != 0u ? 1u : 0u), 1u), 253u);
  };
  auto code4 = [](float a, float b, float c, float d, float inverse) {
    float q[4] = {a * inverse, b * inverse, c * inverse, d * inverse};
    if (MX) {
#pragma unroll
      for (int i = 0; i < 4; ++i) q[i] = fminf(fmaxf(q[i], -448.0f), 448.0f);
    }
    const uint32_t half = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
    return static_cast<uint32_t>(__builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], half, true));
  };
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int row = tid / 16 + 32 * k;
    tile[row * (kRow / 4) + chunk] = words[k];
    if constexpr (ROWS) {
      float most = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) most = fmaxf(most, fmaxf(fabsf(low(words[k][i])), fabsf(high(words[k][i]))));
#pragma unroll
      for (int offset = 1; offset < (MX ? 4 : 16); offset <<= 1) most = fmaxf(most, __shfl_xor(most, offset, 64));
      const uint32_t byte = scale_byte(most);
      const float inverse = __uint_as_float((254u - byte) << 23);
      const u32x2_t packed = {code4(low(words[k][0]), high(words[k][0]), low(words[k][1]), high(words[k][1]), inverse),
                              code4(low(words[k][2]), high(words[k][2]), low(words[k][3]), high(words[k][3]), inverse)};
      const int half = chunk / 8, piece = chunk % 8 / 4, group = chunk % 4 / 2;  // (the operand order of the head of this file)
      *reinterpret_cast<u32x2_t*>(row_codes + static_cast<size_t>(t0 + row) * dim + d0 + 16 * (4 * group + 2 * half + piece) + 8 * (chunk % 2)) = packed;
      if constexpr (MX) {
        uint32_t word = byte << (8 * (chunk / 4));
        word |= __shfl_xor(word, 4, 64);
        word |= __shfl_xor(word, 8, 64);
        if (chunk == 0) *reinterpret_cast<uint32_t*>(row_scales + static_cast<size_t>(t0 + row) * (dim / 32) + d0 / 32) = word;
      } else {
        if (chunk == 0) row_scales[static_cast<size_t>(t0 + row) * pitch + d0 / 128] = static_cast<uint8_t>(byte);
      }
    }
  }
  __syncthreads();
  const int pair = tid % 64, sixteen = tid / 64;
  uint32_t column[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) column[i] = reinterpret_cast<const uint32_t*>(tile)[(16 * sixteen + i) * kRow + pair];
  float first = 0.0f, second = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    first = fmaxf(first, fabsf(low(column[i])));
    second = fmaxf(second, fabsf(high(column[i])));
  }
  largest[sixteen][2 * pair] = first;
  largest[sixteen][2 * pair + 1] = second;
  __syncthreads();
  auto most_of = [&](int c, int thirty_two) {  // a column's block of 32 tokens, or its 128
    if (MX) return fmaxf(largest[2 * thirty_two][c], largest[2 * thirty_two + 1][c]);
    float most = largest[0][c];
#pragma unroll
    for (int i = 1; i < 8; ++i) most = fmaxf(most, largest[i][c]);
    return most;
  };
  const float inverse_first = __uint_as_float((254u - scale_byte(most_of(2 * pair, sixteen / 2))) << 23);
  const float inverse_second = __uint_as_float((254u - scale_byte(most_of(2 * pair + 1, sixteen / 2))) << 23);
  u32x4_t of_first, of_second;
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    of_first[w] = code4(low(column[4 * w]), low(column[4 * w + 1]), low(column[4 * w + 2]), low(column[4 * w + 3]), inverse_first);
    of_second[w] = code4(high(column[4 * w]), high(column[4 * w + 1]), high(column[4 * w + 2]), high(column[4 * w + 3]), inverse_second);
  }
  const int c = d0 + 2 * pair;
  uint8_t* atom = codes + ((static_cast<size_t>(c / 32) * (tokens / 32) + t0 / 32 + sixteen / 2) * 64 + 32 * (sixteen % 2) + c % 32) * 16;
  *reinterpret_cast<u32x4_t*>(atom) = of_first;
  *reinterpret_cast<u32x4_t*>(atom + 16) = of_second;
  if (tid < 128) {
    uint32_t word = 0;
#pragma unroll
    for (int quarter = 0; quarter < 4; ++quarter) word |= scale_byte(most_of(tid, quarter)) << (8 * quarter);
    scales[(static_cast<size_t>((d0 + tid) / 32) * (tokens / 128) + t0 / 128) * 32 + tid % 32] = word;
  }
}

// A kernel gradient's bf16 operands: x [tokens, dim] written transposed, as it is (`gemm_t`'s operands, reference
// src/dew/nn/kernels/gemm.py:418-431) or, NVFP4 true, quantized ALONG THE TOKENS to the NVFP4 recipe's values (E2M1
// codes under an E4M3 scale every 16 tokens, the tensor scale left to the product: quantize_rows_nvfp4_kernel's
// arithmetic, reference src/dew/nn/kernels/projections.py:330-335). BANK false: rows [dim, tokens] bf16. BANK true: a
// prepared DEW_MOE_W_BF16 bank of one expert, depth = tokens, width = dim: atoms [dim / 32][tokens / 16][64 lanes][8
// bf16], lane 32 g + c holding tokens 8 g .. 8 g + 7 of column c. The same 128-token x 64-column tile and thread
// ownership as quantize_columns_kernel.
// With `offsets` (groups + 1 of them) the groups are ragged: each is written from a whole 64-token step on, its last
// step filled with zeros, so that the product's windows need no mask; `tokens` is then the padded extent (at least
// the rows plus 64 a group, in whole 128s), the tokens past the last group are zeros, and `padded` receives the
// groups' offsets in the written order. Every block scans the group sizes itself (at most 4096 of them).
constexpr int kMaxPaddedGroups = 4096;

template <bool NVFP4, bool BANK>
__global__ __launch_bounds__(256) void transpose_columns_kernel(const bf16_t* __restrict__ x, const uint32_t* __restrict__ largest,
                                                                uint8_t* __restrict__ out, float* __restrict__ tensor_scale,
                                                                int tokens, int dim, const int32_t* __restrict__ offsets, int groups,
                                                                int32_t* __restrict__ padded, int rows) {
  __shared__ uint32_t tile[128][33];
  __shared__ u32x4_t staged[64][16];  // the rows operand's 64 rows of 256 bytes, chunk xor-swizzled by the row
  __shared__ int source_row[128];     // the row of x each of the block's tokens is, -1 for a token of padding
  __shared__ int starts[kMaxPaddedGroups + 1];
  __shared__ int partial[256];
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * 128, d0 = blockIdx.y * 64;
  if (offsets == nullptr) {
    if (tid < 128) source_row[tid] = t0 + tid;
  } else {
    // padded start of every group: an exclusive scan of the sizes rounded up to whole 64s
    const int each = (groups + 255) / 256;
    int sum = 0;
    for (int g = tid * each; g < min((tid + 1) * each, groups); ++g) sum += (offsets[g + 1] - offsets[g] + 63) / 64 * 64;
    partial[tid] = sum;
    __syncthreads();
    for (int offset = 1; offset < 256; offset <<= 1) {
      const int other = tid >= offset ? partial[tid - offset] : 0;
      __syncthreads();
      partial[tid] += other;
      __syncthreads();
    }
    int running = partial[tid] - sum;
    for (int g = tid * each; g < min((tid + 1) * each, groups); ++g) {
      starts[g] = running;
      running += (offsets[g + 1] - offsets[g] + 63) / 64 * 64;
    }
    if (tid == 255) starts[groups] = partial[255];
    __syncthreads();
    if (blockIdx.x == 0 && blockIdx.y == 0)
      for (int g = tid; g <= groups; g += 256) padded[g] = starts[g];
    if (tid < 128) {
      const int token = t0 + tid;
      int low = 0, high = groups;  // the last group that starts at or before the token
      while (high - low > 1) {
        const int middle = (low + high) / 2;
        if (starts[middle] <= token) low = middle; else high = middle;
      }
      const int within = token - starts[low];
      const int source = offsets[low] + within;  // (offsets that leave x's rows read nothing)
      source_row[tid] = (token < starts[groups] && within < offsets[low + 1] - offsets[low] && source >= 0 && source < rows) ? source : -1;
    }
  }
  __syncthreads();
  float tensor = 1.0f;
  bool quick = false;  // (the same for the whole launch)
  if constexpr (NVFP4) {
    const float top = __uint_as_float(*largest);
    tensor = nvfp4_tensor_scale(top);
    quick = nvfp4_in_range(top, tensor);
    if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) *tensor_scale = tensor;
  }
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int item = tid + 256 * k, row = item / 8, chunk = item % 8;
    const int source = source_row[row];
    u32x4_t words = {0, 0, 0, 0};
    if (source >= 0) words = *reinterpret_cast<const u32x4_t*>(x + static_cast<size_t>(source) * dim + d0 + chunk * 8);
#pragma unroll
    for (int i = 0; i < 4; ++i) tile[row][chunk * 4 + i] = words[i];
  }
  __syncthreads();
  const int c = tid % 64, quarter = tid / 64;
  uint32_t bits[32];  // the thread's 32 tokens of column c as bf16 patterns
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const uint32_t word = tile[32 * quarter + i][c / 2];
    bits[i] = c % 2 ? word >> 16 : word & 0xFFFFu;
  }
  if constexpr (NVFP4) {
#pragma unroll
    for (int block = 0; block < 2; ++block) {
      float largest_of_block = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) largest_of_block = fmaxf(largest_of_block, fabsf(__uint_as_float(bits[16 * block + i] << 16)));
      const float each = nvfp4_block_scale(largest_of_block, tensor);
      if (quick) {
        const Nvfp4Scales by{tensor, 1.0f / tensor, each, nvfp4_inverse(each)};
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
          const uint32_t both = by.values(__uint_as_float(bits[16 * block + i] << 16), __uint_as_float(bits[16 * block + i + 1] << 16));
          bits[16 * block + i] = both & 0xFFFFu;
          bits[16 * block + i + 1] = both >> 16;
        }
        continue;
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float value = __uint_as_float(bits[16 * block + i] << 16);
        const float over_tensor = each > 0.0f ? value / tensor : 0.0f;
        bits[16 * block + i] = __float_as_uint(copysignf(e2m1_scaled(fabsf(over_tensor), each), over_tensor)) >> 16;
      }
    }
  }
  u32x4_t pieces[4];  // 8 tokens each
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) pieces[j][i] = bits[8 * j + 2 * i] | (bits[8 * j + 2 * i + 1] << 16);
  if constexpr (BANK) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // piece j: atom 2 quarter + j / 2 of the tile's eight, lane group j % 2
      const size_t atom = static_cast<size_t>((d0 + c) / 32) * (tokens / 16) + t0 / 16 + 2 * quarter + j / 2;
      *reinterpret_cast<u32x4_t*>(out + (atom * 64 + 32 * (j % 2) + c % 32) * 16) = pieces[j];
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) staged[c][(4 * quarter + j) ^ (c & 15)] = pieces[j];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int item = tid + 256 * k, row = item / 16, chunk = item % 16;
      *reinterpret_cast<u32x4_t*>(out + (static_cast<size_t>(d0 + row) * tokens + t0) * 2 + chunk * 16) = staged[row][chunk ^ (row & 15)];
    }
  }
}

static int rows_nvfp4_blocks(int rows) { return max(1, min((rows + kQuantizeWaves - 1) / kQuantizeWaves, 2048)); }  // (eight blocks a CU)

static int transpose_columns(const char* who, bool nvfp4, const void* x, void* out, float* tensor_scale, uint32_t* workspace, int tokens,
                             int dim, int as_bank, void* stream, int rows = -1, const int32_t* offsets = nullptr, int groups = 0,
                             int32_t* padded = nullptr) {
  if (rows < 0) rows = tokens;  // (ragged groups: `rows` of x are written into `tokens` padded ones)
  DEW_REQUIRE(tokens >= 0 && tokens % 128 == 0, "%s: %d tokens are not whole 128s", who, tokens);
  if (offsets) {
    DEW_REQUIRE(groups >= 1 && groups <= kMaxPaddedGroups && padded, "%s: %d groups (at most %d) and their padded offsets", who, groups, kMaxPaddedGroups);
    DEW_REQUIRE(rows >= 0 && static_cast<long long>(tokens) >= static_cast<long long>(rows) + 64ll * groups,
                "%s: %d padded tokens do not hold %d rows in %d groups of whole 64s", who, tokens, rows, groups);
  }
  DEW_REQUIRE(dim >= 128 && dim % 128 == 0, "%s: %d columns (whole 128s)", who, dim);
  DEW_REQUIRE(!nvfp4 || (tensor_scale && workspace), "%s: tensor_scale and the 4-byte workspace must not be null", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (nvfp4) {
    hipLaunchKernelGGL(absmax_clear_kernel, dim3(1), dim3(1), 0, s, workspace);
    if (int rc = launched("absmax_clear_kernel")) return rc;
  }
  if (tokens == 0) {
    if (nvfp4) {  // an operand of no tokens: the unit scale
      hipLaunchKernelGGL(quantize_rows_nvfp4_kernel, dim3(1), dim3(64 * kQuantizeWaves), 0, s, static_cast<const bf16_t*>(nullptr), workspace, 1,
                         static_cast<bf16_t*>(nullptr), tensor_scale, static_cast<const float*>(nullptr), static_cast<float*>(nullptr), 0, 0, 0);
      return launched("quantize_rows_nvfp4_kernel");
    }
    return DEW_MOE_OK;
  }
  DEW_REQUIRE(tokens / 128 <= 65535 * 32, "%s: %d tokens", who, tokens);
  DEW_REQUIRE(x && out && aligned16(x) && aligned16(out), "%s: x and out must not be null and must be 16-byte aligned", who);
  if (nvfp4) {
    const long long chunks = static_cast<long long>(rows) * dim / 8;
    const int blocks = static_cast<int>(min((chunks + 255) / 256, 256ll * 2));
    hipLaunchKernelGGL(absmax_kernel, dim3(blocks), dim3(256), 0, s, static_cast<const bf16_t*>(x), chunks, workspace);
    if (int rc = launched("absmax_kernel")) return rc;
  }
  const dim3 grid(tokens / 128, dim / 64);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, static_cast<const bf16_t*>(x), workspace, static_cast<uint8_t*>(out), tensor_scale, tokens, dim,
                       offsets, groups, padded, rows);
  };
  if (nvfp4 && as_bank) launch(transpose_columns_kernel<true, true>);
  else if (nvfp4) launch(transpose_columns_kernel<true, false>);
  else if (as_bank) launch(transpose_columns_kernel<false, true>);
  else launch(transpose_columns_kernel<false, false>);
  return launched("transpose_columns_kernel");
}

// x [tokens, dim] along the tokens, as rows of tokens or as a bank, and with `row_codes` (as a bank) along its rows too.
static int quantize_columns(const char* who, bool mx, const void* x, void* codes, void* scales, int tokens, int dim, int as_bank, void* stream,
                            void* row_codes = nullptr, void* row_scales = nullptr) {
  DEW_REQUIRE(tokens >= 0 && tokens % 128 == 0, "%s: %d tokens are not whole 128-token blocks", who, tokens);
  DEW_REQUIRE(dim >= 128 && dim % 128 == 0, "%s: %d columns (whole 128s)", who, dim);
  if (tokens == 0) return DEW_MOE_OK;
  DEW_REQUIRE(tokens / 128 <= 65535 * 32, "%s: %d tokens", who, tokens);
  DEW_REQUIRE(x && codes && scales, "%s: x, codes and scales must not be null", who);
  DEW_REQUIRE(aligned16(x) && aligned16(codes) && aligned16(scales), "%s: x, codes and scales must be 16-byte aligned", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bf16_t* from = static_cast<const bf16_t*>(x);
  uint8_t* to = static_cast<uint8_t*>(codes);
  uint32_t* scales_to = static_cast<uint32_t*>(scales);
  if (as_bank) {
    const long long tiles = static_cast<long long>(tokens / 128) * (dim / 128);
    DEW_REQUIRE(tiles < (1ll << 30), "%s: %d tokens of %d columns", who, tokens, dim);
    auto kernel = row_codes ? (mx ? quantize_bank_kernel<true, true> : quantize_bank_kernel<false, true>)
                            : (mx ? quantize_bank_kernel<true, false> : quantize_bank_kernel<false, false>);
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>((tiles + 7) / 8 * 8)), dim3(512), 0, s, from, to, scales_to, static_cast<uint8_t*>(row_codes),
                       static_cast<uint8_t*>(row_scales), tokens, dim, (dim / 128 + 15) / 16 * 16);
    return launched("quantize_bank_kernel");
  }
  auto kernel = mx ? quantize_columns_kernel<true> : quantize_columns_kernel<false>;
  hipLaunchKernelGGL(kernel, dim3(tokens / 128, dim / 64), dim3(256), 0, s, from, to, scales_to, tokens, dim);
  return launched("quantize_columns_kernel");
}

}  // namespace dew

extern "C" int dew_moe_transpose_columns(const void* x, void* out, int32_t tokens, int32_t dim, int32_t as_bank, void* stream) {
  return dew::transpose_columns("dew_moe_transpose_columns", false, x, out, nullptr, nullptr, tokens, dim, as_bank, stream);
}

extern "C" int dew_moe_transpose_groups(const void* x, const int32_t* offsets, void* out, int32_t* padded_offsets, int32_t rows,
                                        int32_t padded_tokens, int32_t dim, int32_t groups, int32_t as_bank, void* stream) {
  using namespace dew;
  DEW_REQUIRE(offsets, "dew_moe_transpose_groups: offsets must not be null");
  return transpose_columns("dew_moe_transpose_groups", false, x, out, nullptr, nullptr, padded_tokens, dim, as_bank, stream, rows, offsets, groups,
                           padded_offsets);
}

extern "C" int dew_moe_quantize_columns_nvfp4(const void* x, void* values, float* tensor_scale, uint32_t* workspace, int32_t tokens,
                                              int32_t dim, int32_t as_bank, void* stream) {
  return dew::transpose_columns("dew_moe_quantize_columns_nvfp4", true, x, values, tensor_scale, workspace, tokens, dim, as_bank, stream);
}

extern "C" int dew_moe_quantize_columns_fp8(const void* x, void* codes, void* scales, int32_t tokens, int32_t dim, int32_t as_bank,
                                            void* stream) {
  return dew::quantize_columns("dew_moe_quantize_columns_fp8", false, x, codes, scales, tokens, dim, as_bank, stream);
}

extern "C" int dew_moe_quantize_columns_mxfp8(const void* x, void* codes, void* scales, int32_t tokens, int32_t dim, int32_t as_bank,
                                              void* stream) {
  return dew::quantize_columns("dew_moe_quantize_columns_mxfp8", true, x, codes, scales, tokens, dim, as_bank, stream);
}

extern "C" int dew_moe_quantize_rows_and_columns(const void* x, void* row_codes, uint8_t* row_scales, void* codes, void* scales, int32_t tokens, int32_t dim,
                                                 int32_t mx, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_quantize_rows_and_columns";
  DEW_REQUIRE(tokens == 0 || (row_codes && row_scales && aligned16(row_codes) && aligned16(row_scales)),
              "%s: the rows' codes and scales must not be null and must be 16-byte aligned", who);
  return quantize_columns(who, mx != 0, x, codes, scales, tokens, dim, 1, stream, row_codes, row_scales);
}

extern "C" int dew_moe_quantize_rows_nvfp4(const void* x, void* values, float* tensor_scale, uint32_t* workspace, int32_t rows,
                                           int32_t depth, void* stream) {
  using namespace dew;
  DEW_REQUIRE(rows >= 0 && depth >= 16 && depth % 16 == 0, "dew_moe_quantize_rows_nvfp4: rows %d, depth %d (whole 16s)", rows, depth);
  DEW_REQUIRE(tensor_scale && workspace, "dew_moe_quantize_rows_nvfp4: tensor_scale and the 4-byte workspace must not be null");
  DEW_REQUIRE(rows == 0 || (x && values), "dew_moe_quantize_rows_nvfp4: x and values must not be null");
  DEW_REQUIRE(depth % 8 == 0 && aligned16(x) && aligned16(values), "dew_moe_quantize_rows_nvfp4: x and values must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(absmax_clear_kernel, dim3(1), dim3(1), 0, s, workspace);
  if (int rc = launched("absmax_clear_kernel")) return rc;
  const long long chunks = static_cast<long long>(rows) * depth / 8;
  if (chunks > 0) {
    const int blocks = static_cast<int>(min((chunks + 255) / 256, 256ll * 2));
    hipLaunchKernelGGL(absmax_kernel, dim3(blocks), dim3(256), 0, s, static_cast<const bf16_t*>(x), chunks, workspace);
    if (int rc = launched("absmax_kernel")) return rc;
  }
  hipLaunchKernelGGL(quantize_rows_nvfp4_kernel, dim3(dew::rows_nvfp4_blocks(rows)), dim3(64 * kQuantizeWaves), 0, s, static_cast<const bf16_t*>(x), workspace,
                     1, static_cast<bf16_t*>(values), tensor_scale, static_cast<const float*>(nullptr), static_cast<float*>(nullptr), 0, rows, depth);
  return launched("quantize_rows_nvfp4_kernel");
}

extern "C" int dew_moe_nvfp4_partials(void) { return dew::kNvfp4Partials; }

extern "C" int dew_moe_nvfp4_largest_of(const void* const* operands, const int64_t* elements, const int32_t* is_f32, int32_t count, uint32_t* partials,
                                        void* stream) {
  using namespace dew;
  const char* who = "dew_moe_nvfp4_largest";
  DEW_REQUIRE(operands && elements && is_f32 && count >= 1 && count <= kMostOperands, "%s: %d operands (1 to %d)", who, count, kMostOperands);
  DEW_REQUIRE(partials, "%s: the partials must not be null", who);
  LargestOperands of{};
  for (int i = 0; i < count; ++i) {
    DEW_REQUIRE(elements[i] >= 0 && elements[i] % 8 == 0, "%s: an operand of %lld elements (whole 8s)", who, static_cast<long long>(elements[i]));
    DEW_REQUIRE(elements[i] == 0 || (operands[i] && aligned16(operands[i])), "%s: the operand must not be null and must be 16-byte aligned", who);
    of.x[i] = static_cast<const u32x4_t*>(operands[i]);
    of.chunks[i] = elements[i] / (is_f32[i] ? 4 : 8);
    of.f32[i] = is_f32[i];
  }
  hipLaunchKernelGGL(nvfp4_largest_kernel, dim3(kNvfp4Partials, count), dim3(256), 0, static_cast<hipStream_t>(stream), of, partials);
  return launched("nvfp4_largest_kernel");
}

extern "C" int dew_moe_nvfp4_largest(const void* operand, int64_t elements, int32_t is_f32, uint32_t* partials, void* stream) {
  return dew_moe_nvfp4_largest_of(&operand, &elements, &is_f32, 1, partials, stream);
}

extern "C" int dew_moe_quantize_nvfp4(const void* x, const uint32_t* largest, void* row_values, void* token_values, float* tensor_scale,
                                      const float* bank_scales, float* products, int32_t experts, int32_t rows, int32_t depth, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_quantize_nvfp4";
  DEW_REQUIRE(rows >= 0 && depth >= 16 && depth % 16 == 0, "%s: rows %d, depth %d (whole 16s)", who, rows, depth);
  DEW_REQUIRE(!token_values || (rows >= 1 && rows % 128 == 0 && depth % 128 == 0), "%s: %d tokens of %d columns are not whole 128s", who, rows, depth);
  DEW_REQUIRE(largest && tensor_scale && (row_values || token_values), "%s: largest, tensor_scale and the values must not be null", who);
  DEW_REQUIRE(!bank_scales || (products && experts >= 1 && row_values), "%s: %d products of a bank's tensor scales and the rows'", who, experts);
  DEW_REQUIRE(rows == 0 || (x && aligned16(x) && aligned16(row_values) && aligned16(token_values)), "%s: x and the values must be 16-byte aligned", who);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const bf16_t* from = static_cast<const bf16_t*>(x);
  bf16_t *by_row = static_cast<bf16_t*>(row_values), *by_token = static_cast<bf16_t*>(token_values);
  if (!token_values) {
    hipLaunchKernelGGL(quantize_rows_nvfp4_kernel, dim3(rows_nvfp4_blocks(rows)), dim3(64 * kQuantizeWaves), 0, s, from, largest, kNvfp4Partials, by_row,
                       tensor_scale, bank_scales, products, experts, rows, depth);
    return launched("quantize_rows_nvfp4_kernel");
  }
  const long long blocks = (static_cast<long long>(rows / 16) * (depth / 4) + 255) / 256;
  DEW_REQUIRE(blocks < (1ll << 31), "%s: %d tokens of %d columns", who, rows, depth);
  if (row_values)
    hipLaunchKernelGGL(quantize_tokens_nvfp4_kernel<true>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, from, largest, by_row, by_token,
                       tensor_scale, bank_scales, products, experts, rows, depth);
  else
    hipLaunchKernelGGL(quantize_tokens_nvfp4_kernel<false>, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, s, from, largest, by_row, by_token,
                       tensor_scale, bank_scales, products, experts, rows, depth);
  return launched("quantize_tokens_nvfp4_kernel");
}

extern "C" int dew_moe_quantize_rows_mxfp8(const void* x, void* codes, uint8_t* scales, int32_t rows, int32_t depth, void* stream) {
  return dew::quantize_rows<true>("dew_moe_quantize_rows_mxfp8", x, codes, scales, rows, depth, stream);
}

extern "C" int dew_moe_quantize_rows_fp8(const void* x, void* codes, uint8_t* scales, int32_t rows, int32_t depth, void* stream) {
  return dew::quantize_rows<false>("dew_moe_quantize_rows_fp8", x, codes, scales, rows, depth, stream);
}
