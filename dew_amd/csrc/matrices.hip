// A training step's weight matrices, new at every step, quantized for a recipe's product straight into the prepared layout
// its kernel reads: w [E, K, N] bf16 or fp32 in, a prepared bank of FP8 128 x 128 blocks, MXFP8 or NVFP4 out, in one pass
// (NVFP4 reads w once more first, for its tensor scale). With KMAJOR, w is held [E, N, K]: the same memory as the matrices
// of the transposed product, which is how an input gradient reads the forward's weights with no transposed copy.
// The arithmetic is the rows' quantizers' (quantize.hip), along the depth:
//   FP8 blocks  scale = the least power of two >= max(amax, 1e-4) * f32(1 / 448) of a 128 x 128 block, codes e4m3(w / scale)
//   MXFP8       scale = 2^(exponent of the largest of 32 depths - 8), codes saturating at +-448
//   NVFP4       tensor scale amax / 2688 over all matrices; a block of 16 depths the least e4m3 >= blockmax / tensor / 6;
//               codes the nearest E2M1, ties to the even code
// Bound by HBM: 2 (4) bytes read and 1 (NVFP4: 0.56) written an element, so the layout of the work is the loads': a block of
// 512 threads takes 128 depths x 128 columns, every load 16 bytes of a 256- (512-) byte run of a row. Natural w: a thread
// owns 4 (8) consecutive depths of 8 (4) columns, so that the depth's maxima are taken in registers first and four depths of
// a column leave the conversion as one dword; K-major w: 8 (4) consecutive depths of a column. The codes (not the values)
// cross the LDS into columns, and leave as a lane's 16-byte pieces, 512 bytes a wavefront's half.
// Measured on [8, 4096, 14336] bf16 (0.94 GB in, 0.47 out): FP8 blocks and MXFP8 250 to 275 us, 5.1 to 5.6 TB/s, where the same
// rules as whole-tensor operations and a re-layout of their result took 4.5 (FP8) and 8.5 ms (MXFP8); NVFP4 on [8, 2048, 4096]
// bf16 33 us (K-major 36) and 26 us for the largest magnitude, against some 7 ms. (Its E2M1 choice is nine vector instructions an
// element, nvfp4.h; the general form, which fp32 matrices and operands out of range take, is thirty: 67 us here.)
#include "common.h"
#include "nvfp4.h"
#include "sort.h"

namespace dew {

typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;

constexpr int kMatrixThreads = 512;
constexpr int kMatrixTile = 128;

template <typename T>
__device__ __forceinline__ void values_of(const u32x4_t& words, float (&v)[16 / sizeof(T)]) {
  if constexpr (sizeof(T) == 2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(words[i] << 16);
      v[2 * i + 1] = __uint_as_float(words[i] & 0xFFFF0000u);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(words[i]);
  }
}

// The e4m3 scale byte of a 16-deep NVFP4 block whose largest magnitude is `block`, under the tensor scale: the nearest e4m3
// to block / tensor / 6 and the next one where that lies below (quantize_rows_nvfp4_kernel's rule); a NaN stays one.
__device__ __forceinline__ uint32_t nvfp4_block_byte(float block, float tensor) {
  const float ratio = (block / tensor) / 6.0f;
  if (ratio != ratio) return 0x7Fu;
  uint32_t byte = __builtin_amdgcn_cvt_pk_fp8_f32(fminf(ratio, 448.0f), 0.0f, 0, false) & 0xFFu;
  if (__builtin_amdgcn_cvt_f32_fp8(byte, 0) < ratio) byte = min(byte + 1u, 0x7Eu);
  return byte;
}

// The E2M1 code (sign in bit 3) of value / tensor / each, ties to the even code; zero under a zero (or NaN) scale. The
// thresholds are multiplied by `each` instead of the quotient divided: exact, see e2m1_scaled in nvfp4.h.
__device__ __forceinline__ uint32_t e2m1_code(float value, float tensor, float each) {
  if (!(each > 0.0f)) return 0u;
  const float y = value / tensor, m = fabsf(y);
  const uint32_t code = (m > 0.25f * each ? 1u : 0u) + (m >= 0.75f * each ? 1u : 0u) + (m > 1.25f * each ? 1u : 0u) + (m >= 1.75f * each ? 1u : 0u) +
                        (m > 2.5f * each ? 1u : 0u) + (m >= 3.5f * each ? 1u : 0u) + (m > 5.0f * each ? 1u : 0u);
  return code | ((__float_as_uint(y) >> 31) << 3);
}

__device__ __forceinline__ float mx_inverse(uint32_t byte) { return __uint_as_float((254u - byte) << 23); }

__device__ __forceinline__ uint32_t mx_byte(uint32_t largest_bits) {
  return static_cast<uint32_t>(min(max(static_cast<int>(largest_bits >> 23) - 8, 0), 254));
}

// value times the scale's inverse, saturated at e4m3's largest; a NaN stays one
__device__ __forceinline__ float saturated(float value, float inverse) {
  const float q = fminf(fmaxf(value * inverse, -448.0f), 448.0f);
  return value == value ? q : value;
}

// A step's groups, counted in blocks of `unit` rows, and where their offsets go (null: none): the matrices' launch writes them beside its codes, or
// the step would take a launch of 5 us for a few words.
struct StepGroups {
  const int32_t* blocks;
  int32_t* offsets;
  int groups, unit;
};

template <int FORMAT, typename T, bool KMAJOR, bool CACHED>
__global__ __launch_bounds__(kMatrixThreads) void quantize_matrices_kernel(const T* __restrict__ w, uint8_t* __restrict__ codes,
                                                                         uint8_t* __restrict__ scales, const uint32_t* __restrict__ largest,
                                                                         float* __restrict__ tensor_scales, int depth, int width, StepGroups step) {
  constexpr bool kBlocks = FORMAT == DEW_MOE_W_FP8_BLOCK, kNv = FORMAT == DEW_MOE_W_NVFP4;
  constexpr int kVec = 16 / sizeof(T);                   // elements of a load, along the memory's inner axis
  constexpr int kLanes = kMatrixTile / kVec;             // lanes a row of the tile
  constexpr int kGroups = kMatrixThreads / kLanes;       // rows the block loads at once
  constexpr int kLoads = kMatrixTile / kGroups;          // loads (rows) a thread
  constexpr int kBlock = kNv ? 16 : 32, kScales = kMatrixTile / kBlock;  // depths a scale, scales a column of the tile
  static_assert(kLoads % 4 == 0, "whole dwords of four depths a column");
  // natural: [depths / 4][128 columns] of four codes each; K-major: [128 columns] rows of codes, padded to whole 16 bytes
  constexpr int kPitch = kNv ? 80 : 144;
  __shared__ alignas(16) uint8_t staged[KMAJOR ? kMatrixTile * kPitch : kMatrixTile * kMatrixTile / (kNv ? 2 : 1)];
  __shared__ uint32_t maxima[8][kMatrixTile];            // natural: a wavefront's 16 depths' largest magnitude a column
  __shared__ uint8_t scale_bytes[kScales][kMatrixTile];
  __shared__ float each_of[!KMAJOR && !kBlocks ? kScales : 1][kMatrixTile];  // natural: a block's scale (NVFP4) or its inverse (MXFP8)

  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  const int k0 = (KMAJOR ? blockIdx.x : blockIdx.y) * kMatrixTile, n0 = (KMAJOR ? blockIdx.y : blockIdx.x) * kMatrixTile;
  const size_t e = blockIdx.z;
  const int pitch = KMAJOR ? depth : width;
  const int group = tid / kLanes, piece = tid % kLanes;
  // natural: a thread's rows are consecutive depths; K-major: rows are columns, dealt group by group
  auto row_of = [&](int p) { return KMAJOR ? p * kGroups + group : group * kLoads + p; };
  const T* source = w + e * depth * width + static_cast<size_t>(KMAJOR ? n0 : k0) * pitch + (KMAJOR ? k0 : n0) + piece * kVec;
  const uint32_t share = kNv ? nvfp4_share(largest, kNvfp4Partials) : 0u;
  // Bound by memory, and every weight is read once: non-temporal, so that the weights don't push out what the step's products read next. us of
  // twelve drawn steps of the FP8 recipes 1.00 to 1.12 times as fast (252 -> 224, 535 -> 497, 228 -> 209). CACHED: NVFP4's were just read for their largest
  // magnitude, and where the 256 MB of the last-level cache hold them all, such loads only miss it (steps of 512 to 1024 rows, without and with them: 16 x 768 x
  // 6912, 170 MB, 268 and 279 us, 22 x 768 x 4864, 164, 267 and 279; 31 x 5120 x 1024, 325, 531 and 515). Non-temporal stores too, of codes that the product
  // reads at once: no difference in steps of 400 us and more and of 113 and less, 5 to 10 % slower in those of 180 to 300.
  u32x4_t words[kLoads];
#pragma unroll
  for (int p = 0; p < kLoads; ++p) {
    const u32x4_t* from = reinterpret_cast<const u32x4_t*>(source + static_cast<size_t>(row_of(p)) * pitch);
    words[p] = CACHED ? *from : __builtin_nontemporal_load(from);
  }

  float tensor = 1.0f;
  bool quick = false;  // (the same for the whole launch)
  if constexpr (kNv) {
    const float top = nvfp4_top(share);
    tensor = nvfp4_tensor_scale(top);
    quick = sizeof(T) == 2 && nvfp4_in_range(top, tensor);
    if (blockIdx.x == 0 && blockIdx.y == 0 && tid == 0) tensor_scales[e] = tensor;
  }
  float v[kLoads][kVec];
#pragma unroll
  for (int p = 0; p < kLoads; ++p) values_of<T>(words[p], v[p]);
  const float inverse_tensor = kNv ? 1.0f / tensor : 1.0f;
  auto magnitude = [](float value) { return __float_as_uint(value) & 0x7FFFFFFFu; };
  float inverse = 1.0f;  // FP8 blocks: the tile's one
  if constexpr (kBlocks) {
    uint32_t most = 0;
#pragma unroll
    for (int p = 0; p < kLoads; ++p)
#pragma unroll
      for (int i = 0; i < kVec; ++i) most = max(most, magnitude(v[p][i]));
#pragma unroll
    for (int offset = 32; offset >= 1; offset >>= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), offset, 64)));
    if (lane == 0) maxima[0][wave] = most;
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kMatrixThreads / 64; ++i) most = max(most, maxima[0][i]);
    const uint32_t bits = __float_as_uint(fmaxf(__uint_as_float(most), 1e-4f) * 0x1.24924ap-9f);  // f32(1 / 448)
    const uint32_t field = min(max((bits >> 23) + ((bits & 0x7FFFFFu) != 0u ? 1u : 0u), 1u), 253u);
    inverse = __uint_as_float((254u - field) << 23);
    if (tid == 0)  // a block that holds an infinity or NaN has no power of two: the product writes its tile as NaN
      reinterpret_cast<float*>(scales)[(e * (depth / 128) + k0 / 128) * (width / 128) + n0 / 128] =
          most >= 0x7F800000u ? __builtin_inff() : __uint_as_float(field << 23);
  } else if constexpr (!KMAJOR) {
    uint32_t most[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
      most[i] = magnitude(v[0][i]);
#pragma unroll
      for (int p = 1; p < kLoads; ++p) most[i] = max(most[i], magnitude(v[p][i]));
#pragma unroll
      for (int offset = kLanes; offset < 64; offset <<= 1) most[i] = max(most[i], static_cast<uint32_t>(__shfl_xor(static_cast<int>(most[i]), offset, 64)));
    }
    if (lane < kLanes) {
#pragma unroll
      for (int i = 0; i < kVec; ++i) maxima[wave][piece * kVec + i] = most[i];
    }
    __syncthreads();
    for (int item = tid; item < kScales * kMatrixTile; item += kMatrixThreads) {
      const int block = item / kMatrixTile, column = item % kMatrixTile;
      if constexpr (kNv) {
        const uint32_t byte = nvfp4_block_byte(__uint_as_float(maxima[block][column]), tensor);
        scale_bytes[block][column] = static_cast<uint8_t>(byte);
        const float each = __builtin_amdgcn_cvt_f32_fp8(byte, 0);
        each_of[block][column] = quick ? nvfp4_inverse(each) : each;
      } else {
        const uint32_t byte = mx_byte(max(maxima[2 * block][column], maxima[2 * block + 1][column]));
        scale_bytes[block][column] = static_cast<uint8_t>(byte);
        each_of[block][column] = mx_inverse(byte);
      }
    }
    __syncthreads();
  }

  if constexpr (!KMAJOR) {
    const int block = group * kLoads / kBlock;
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
      const int column = piece * kVec + i;
      const float each = kBlocks ? inverse : each_of[block][column];
#pragma unroll
      for (int d = 0; d < kLoads / 4; ++d) {  // four depths of the column
        const int quad = group * (kLoads / 4) + d;
        if constexpr (kNv) {
          uint32_t nibbles = 0;
          if (quick) {
            const Nvfp4Scales by{tensor, inverse_tensor, __builtin_amdgcn_cvt_f32_fp8(scale_bytes[block][column], 0), each};
            nibbles = by.four(v[4 * d][i], v[4 * d + 1][i], v[4 * d + 2][i], v[4 * d + 3][i]);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) nibbles |= e2m1_code(v[4 * d + r][i], tensor, each) << (4 * r);
          }
          reinterpret_cast<uint16_t*>(staged)[quad * kMatrixTile + column] = static_cast<uint16_t>(nibbles);
        } else {
          float q[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) q[r] = kBlocks ? v[4 * d + r][i] * each : saturated(v[4 * d + r][i], each);
          uint32_t packed = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
          packed = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], packed, true);
          reinterpret_cast<uint32_t*>(staged)[quad * kMatrixTile + column] = packed;
        }
      }
    }
  } else {
#pragma unroll
    for (int p = 0; p < kLoads; ++p) {
      const int column = row_of(p), k = piece * kVec;
      float each = inverse;
      if constexpr (!kBlocks) {
        uint32_t most = magnitude(v[p][0]);
#pragma unroll
        for (int i = 1; i < kVec; ++i) most = max(most, magnitude(v[p][i]));
#pragma unroll
        for (int offset = 1; offset < kBlock / kVec; offset <<= 1) most = max(most, static_cast<uint32_t>(__shfl_xor(static_cast<int>(most), offset, 64)));
        const uint32_t byte = kNv ? nvfp4_block_byte(__uint_as_float(most), tensor) : mx_byte(most);
        each = kNv ? __builtin_amdgcn_cvt_f32_fp8(byte, 0) : mx_inverse(byte);
        if (k % kBlock == 0) scale_bytes[k / kBlock][column] = static_cast<uint8_t>(byte);
      }
#pragma unroll
      for (int d = 0; d < kVec / 4; ++d) {
        if constexpr (kNv) {
          uint32_t nibbles = 0;
          if (quick) {
            const Nvfp4Scales by{tensor, inverse_tensor, each, nvfp4_inverse(each)};
            nibbles = by.four(v[p][4 * d], v[p][4 * d + 1], v[p][4 * d + 2], v[p][4 * d + 3]);
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) nibbles |= e2m1_code(v[p][4 * d + r], tensor, each) << (4 * r);
          }
          *reinterpret_cast<uint16_t*>(staged + column * kPitch + k / 2 + 2 * d) = static_cast<uint16_t>(nibbles);
        } else {
          float q[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) q[r] = kBlocks ? v[p][4 * d + r] * each : saturated(v[p][4 * d + r], each);
          uint32_t packed = __builtin_amdgcn_cvt_pk_fp8_f32(q[0], q[1], 0, false);
          packed = __builtin_amdgcn_cvt_pk_fp8_f32(q[2], q[3], packed, true);
          *reinterpret_cast<uint32_t*>(staged + column * kPitch + k + 4 * d) = packed;
        }
      }
    }
  }
  __syncthreads();

  // thread (column c, quarter q): the 32 depths 32 q .. 32 q + 31 of column c
  const int c = tid % kMatrixTile, q = tid / kMatrixTile;
  const size_t strip = e * (width / 32) + (n0 + c) / 32;
  if constexpr (kNv) {  // one lane's piece of an atom of 64 depths: lane 32 (q % 2) + column
    u32x4_t out;
    if constexpr (KMAJOR) {
      out = *reinterpret_cast<const u32x4_t*>(staged + c * kPitch + 16 * q);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t* at = reinterpret_cast<const uint16_t*>(staged) + (8 * q + 2 * i) * kMatrixTile + c;
        out[i] = static_cast<uint32_t>(at[0]) | (static_cast<uint32_t>(at[kMatrixTile]) << 16);
      }
    }
    const size_t at = (strip * (depth / 64) + k0 / 64 + q / 2) * 64 + 32 * (q % 2) + c % 32;
    *reinterpret_cast<u32x4_t*>(codes + at * 16) = out;
    reinterpret_cast<uint16_t*>(scales)[at] = static_cast<uint16_t>(scale_bytes[2 * q][c] | (scale_bytes[2 * q + 1][c] << 8));
  } else {  // an atom of 32 depths: its lanes c and 32 + c
    u32x4_t low, high;
    if constexpr (KMAJOR) {
      const u32x4_t* at = reinterpret_cast<const u32x4_t*>(staged + c * kPitch + 32 * q);
      low = at[0], high = at[1];
    } else {
      const uint32_t* at = reinterpret_cast<const uint32_t*>(staged) + 8 * q * kMatrixTile + c;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        low[i] = at[i * kMatrixTile];
        high[i] = at[(4 + i) * kMatrixTile];
      }
    }
    uint8_t* atom = codes + (strip * (depth / 32) + k0 / 32 + q) * kAtomBytes + (c % 32) * 16;
    *reinterpret_cast<u32x4_t*>(atom) = low;
    *reinterpret_cast<u32x4_t*>(atom + 512) = high;
    if constexpr (!kBlocks) {  // the column's four scale bytes of this 128-deep step
      if (tid < kMatrixTile) {
        uint32_t word = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) word |= static_cast<uint32_t>(scale_bytes[b][c]) << (8 * b);
        reinterpret_cast<uint32_t*>(scales)[(strip * (depth / 128) + k0 / 128) * 32 + c % 32] = word;
      }
    }
  }
  if (step.blocks && tid < 64 && blockIdx.x + blockIdx.y + blockIdx.z == 0) write_group_offsets(step.blocks, step.offsets, step.groups, step.unit);
}

// An NVFP4 bank's buffer: codes, block scales, then the partial largest magnitudes and the tensor scales.
static size_t nvfp4_scales_at(size_t elements) { return elements / 2; }
static size_t nvfp4_largest_at(size_t elements) { return elements / 2 + elements / 16; }

template <int FORMAT, typename T>
static int quantize_matrices(const T* w, bool kmajor, int experts, int depth, int width, const uint32_t* known_largest, const StepGroups& step, uint8_t* prepared,
                             dew_moe_bank* out, hipStream_t s) {
  const size_t elements = static_cast<size_t>(experts) * depth * width;
  uint8_t* scales = prepared + (FORMAT == DEW_MOE_W_NVFP4 ? nvfp4_scales_at(elements) : elements);
  uint32_t* largest = reinterpret_cast<uint32_t*>(prepared + nvfp4_largest_at(elements));
  float* tensor_scales = reinterpret_cast<float*>(largest + kNvfp4Partials);
  *out = dew_moe_bank{FORMAT, DEW_MOE_LAYOUT_PREPARED, experts, depth, width, prepared, scales, FORMAT == DEW_MOE_W_NVFP4 ? tensor_scales : nullptr};
  if (FORMAT == DEW_MOE_W_NVFP4 && !known_largest) {
    if (int rc = dew_moe_nvfp4_largest(w, static_cast<int64_t>(elements), sizeof(T) == 4, largest, s)) return rc;
  }
  const dim3 grid = kmajor ? dim3(depth / 128, width / 128, experts) : dim3(width / 128, depth / 128, experts);
  constexpr bool kNv = FORMAT == DEW_MOE_W_NVFP4;
  const bool cached = kNv && elements * sizeof(T) <= (size_t{256} << 20);
  auto kernel = cached ? (kmajor ? quantize_matrices_kernel<FORMAT, T, true, kNv> : quantize_matrices_kernel<FORMAT, T, false, kNv>)
                       : (kmajor ? quantize_matrices_kernel<FORMAT, T, true, false> : quantize_matrices_kernel<FORMAT, T, false, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(kMatrixThreads), 0, s, w, prepared, scales, known_largest ? known_largest : largest, tensor_scales, depth, width, step);
  return launched("quantize_matrices_kernel");
}

}  // namespace dew

extern "C" size_t dew_moe_quantized_matrices_bytes(int32_t format, int32_t experts, int32_t depth, int32_t width) {
  if (experts <= 0 || depth <= 0 || width <= 0) return 0;
  const size_t elements = static_cast<size_t>(experts) * depth * width;
  if (format == DEW_MOE_W_NVFP4) return dew::nvfp4_largest_at(elements) + 4 * dew::kNvfp4Partials + (static_cast<size_t>(experts) * 4 + 255) / 256 * 256;
  return dew_moe_prepared_bytes(format, experts, depth, width);
}

static int quantize_matrices_of(const char* who, const void* w, int32_t format, int32_t w_is_f32, int32_t kmajor, int32_t experts, int32_t depth, int32_t width,
                                const uint32_t* largest, const int32_t* blocks, int32_t groups, int32_t unit, int32_t* offsets, void* prepared, dew_moe_bank* out,
                                void* stream) {
  using namespace dew;
  DEW_REQUIRE(w && prepared && out, "%s: w, the prepared buffer and out must not be null", who);
  DEW_REQUIRE(format == DEW_MOE_W_FP8_BLOCK || format == DEW_MOE_W_MXFP8 || format == DEW_MOE_W_NVFP4,
              "%s: format %d is none of the recipes' (FP8 blocks, MXFP8, NVFP4)", who, format);
  DEW_REQUIRE(experts >= 1 && experts <= 4096, "%s: %d matrices", who, experts);
  DEW_REQUIRE(depth >= 128 && depth % 128 == 0 && width >= 128 && width % 128 == 0 && depth / 128 <= 65535 && width / 128 <= 65535,
              "%s: matrices of %d x %d (whole 128s)", who, depth, width);
  DEW_REQUIRE(aligned16(w) && (reinterpret_cast<uintptr_t>(prepared) & 255u) == 0, "%s: w must be 16-byte and the prepared buffer 256-byte aligned", who);
  DEW_REQUIRE(!largest || format == DEW_MOE_W_NVFP4, "%s: a bank of format %d has no tensor scale to form from magnitudes", who, format);
  DEW_REQUIRE(!blocks || (offsets && groups >= 1 && unit >= 1), "%s: offsets must not be null, %d groups in units of %d", who, groups, unit);
  const StepGroups step{blocks, offsets, groups, unit};
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint8_t* buffer = static_cast<uint8_t*>(prepared);
  auto of = [&](auto* typed) {
    switch (format) {
      case DEW_MOE_W_FP8_BLOCK: return quantize_matrices<DEW_MOE_W_FP8_BLOCK>(typed, kmajor != 0, experts, depth, width, largest, step, buffer, out, s);
      case DEW_MOE_W_MXFP8: return quantize_matrices<DEW_MOE_W_MXFP8>(typed, kmajor != 0, experts, depth, width, largest, step, buffer, out, s);
      default: return quantize_matrices<DEW_MOE_W_NVFP4>(typed, kmajor != 0, experts, depth, width, largest, step, buffer, out, s);
    }
  };
  return w_is_f32 ? of(static_cast<const float*>(w)) : of(static_cast<const bf16_t*>(w));
}

extern "C" int dew_moe_quantize_matrices(const void* w, int32_t format, int32_t w_is_f32, int32_t kmajor, int32_t experts, int32_t depth,
                                         int32_t width, void* prepared, dew_moe_bank* out, void* stream) {
  return quantize_matrices_of("dew_moe_quantize_matrices", w, format, w_is_f32, kmajor, experts, depth, width, nullptr, nullptr, 0, 0, nullptr, prepared, out, stream);
}

extern "C" int dew_moe_quantize_step_matrices(const void* w, int32_t format, int32_t w_is_f32, int32_t kmajor, int32_t experts, int32_t depth,
                                              int32_t width, const uint32_t* largest, const int32_t* blocks, int32_t groups, int32_t unit,
                                              int32_t* offsets, void* prepared, dew_moe_bank* out, void* stream) {
  return quantize_matrices_of("dew_moe_quantize_step_matrices", w, format, w_is_f32, kmajor, experts, depth, width, largest, blocks, groups, unit, offsets, prepared, out, stream);
}
