// The grouped product for few tiles of few rows: a decode step of one or a few tokens.
//
// The tiled launch gives a tile of an expert's rows and 128 columns to a block of four wavefronts that share the rows in the
// LDS. One token's eight experts of 768 columns are then 48 blocks, and 208 CUs idle. Here a wavefront is a block of its own
// and owns 32 columns (of both matrices of a pair): the same wavefronts, but on as many CUs, each with the memory pipeline to
// itself and, with no barrier and no LDS stage a step, as much of its weights in flight as the registers hold. The rows are
// few, so their fragments come straight from global memory (the lanes past a group's rows read its last row again, the
// same cache lines). The depth is not split between wavefronts: every sum is taken in the tiled launches' order, so a
// product's bits do not depend on which of them ran.
#include "gemm.h"

namespace dew {

template <int FORMAT, int MODE>
__global__ __launch_bounds__(64) void few_tiles_kernel(GemmParams p) {
  constexpr bool kPaired = MODE == kSwigluOfTwo, kGated = MODE == kInterleavedGated;
  constexpr bool kFp4 = FORMAT == DEW_MOE_W_NVFP4 || FORMAT == DEW_MOE_W_MXFP4, kBf16 = FORMAT == DEW_MOE_W_BF16;
  constexpr int kMatrices = kPaired ? 2 : 1;
  constexpr int kAtomK = kFp4 ? 64 : kBf16 ? 16 : 32, kAtoms = 64 / kAtomK;  // 16-byte loads a lane makes per matrix and 64 depths
  constexpr int kAhead = kMatrices * kAtoms >= 8 ? 4 : kMatrices * kAtoms >= 4 ? 6 : 8;  // steps of 64 depths in flight
  constexpr int kRows = 32;
  const int lane = threadIdx.x;
  const int strips = p.width / 32, m_tile = blockIdx.x / strips, strip = blockIdx.x % strips;

  // ---- which expert owns row tile `m_tile`? Every wavefront scans the groups for itself, 64 a round, without a barrier ----
  auto scanned = [lane](int value) {
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
      const int other = __shfl_up(value, offset, 64);
      if (lane >= offset) value += other;
    }
    return value;
  };
  auto size_of = [&p](int e) { return e >= p.experts ? 0 : p.sizes ? max(p.sizes[e], 0) : p.offsets[e + 1] - p.offsets[e]; };
  auto first_row_of = [&p](int e) { return e >= p.experts || p.sizes ? 0 : p.offsets[e]; };
  int expert = -1, row0 = 0, end = 0, carried = 0, carried_rows = 0;
  int next_size = size_of(lane), next_first = first_row_of(lane);
  for (int base = 0; base < p.experts; base += 64) {
    const int size = next_size;
    int start = next_first;
    next_size = size_of(base + 64 + lane);
    next_first = first_row_of(base + 64 + lane);
    if (p.sizes) {
      const int rows = scanned(size);
      start = carried_rows + rows - size;
      carried_rows += __builtin_amdgcn_readlane(rows, 63);
    }
    const int tiles = (size + kRows - 1) / kRows, inclusive = scanned(tiles), first = carried + inclusive - tiles;
    const unsigned long long hit = __ballot(m_tile >= first && m_tile < first + tiles);
    if (hit != 0ull) {
      const int owner = __builtin_ctzll(hit);
      expert = base + owner;
      row0 = __builtin_amdgcn_readlane(start + (m_tile - first) * kRows, owner);
      end = __builtin_amdgcn_readlane(start + size, owner);
      break;
    }
    carried += __builtin_amdgcn_readlane(inclusive, 63);
  }
  const int out_width = kGated ? p.width / 2 : p.width;
  constexpr int kOutColumns = kGated ? 16 : 32;
  if (expert < 0) {  // past the last tile: zero the rows that no expert owns
    const int tail_begin = (p.sizes ? carried_rows : p.offsets[p.experts]) + (m_tile - carried) * kRows;
    const int tail_end = min(tail_begin + kRows, p.rows);
    for (int item = threadIdx.x; item < (tail_end - tail_begin) * (kOutColumns / 8); item += 64) {
      const int sorted = tail_begin + item / (kOutColumns / 8), row = p.scatter ? p.scatter[sorted] : sorted;
      *reinterpret_cast<u32x4_t*>(p.out + static_cast<size_t>(row) * out_width + strip * kOutColumns + item % (kOutColumns / 8) * 8) = u32x4_t{0, 0, 0, 0};
    }
    return;
  }
  const int valid_rows = min(kRows, end - row0);

  const int steps = p.depth / 64;
  const int k_atoms = p.depth / kAtomK;
  const size_t first_atom = (static_cast<size_t>(expert) * strips + strip) * k_atoms;
  const uint8_t* b_src[kMatrices];
  const uint8_t* b_scale_src[kMatrices];
  const float* block_scales[kMatrices];
  float channel_scale[kMatrices];
#pragma unroll
  for (int m = 0; m < kMatrices; ++m) {
    const BankView& bank = m == 0 ? p.w0 : p.w1;
    b_src[m] = bank.codes + first_atom * kAtomBytes + lane * 16;
    b_scale_src[m] = kFp4 ? static_cast<const uint8_t*>(bank.scales) + first_atom * 128 + lane * 2 : nullptr;
    block_scales[m] = FORMAT == DEW_MOE_W_FP8_BLOCK
                          ? static_cast<const float*>(bank.scales) + static_cast<size_t>(expert) * (p.depth / 128) * (p.width / 128) + strip / 4
                          : nullptr;
    channel_scale[m] = FORMAT == DEW_MOE_W_FP8_CHANNEL ? static_cast<const float*>(bank.scales)[static_cast<size_t>(expert) * p.width + strip * 32 + lane % 32] : 1.0f;
  }
  const int sorted_row = row0 + min(lane % 32, valid_rows - 1);
  const bf16_t* a_row = p.x + static_cast<size_t>(p.gather ? p.gather[sorted_row] : sorted_row) * p.depth;
  u32x4_t a[kAhead][4], b[kAhead][kMatrices][kAtoms];
  uint32_t fp4_bytes[kAhead][kMatrices];
  float scale[kAhead][kMatrices];
  auto load = [&](auto set, int step) __attribute__((always_inline)) {
    constexpr int s = decltype(set)::value;
#pragma unroll
    for (int m = 0; m < kMatrices; ++m) {
#pragma unroll
      for (int i = 0; i < kAtoms; ++i)
        b[s][m][i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(b_src[m] + (static_cast<size_t>(step) * kAtoms + i) * kAtomBytes));
      if constexpr (kFp4) fp4_bytes[s][m] = *reinterpret_cast<const uint16_t*>(b_scale_src[m] + static_cast<size_t>(step) * 128);
      if constexpr (FORMAT == DEW_MOE_W_FP8_BLOCK) scale[s][m] = block_scales[m][static_cast<size_t>(step / 2) * (p.width / 128)];
    }
    // slice kk of a step: the 8 depths that the lane's weight bytes of that slice cover
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int chunk = kFp4 ? 4 * (lane / 32) + kk : kBf16 ? 2 * kk + lane / 32 : 4 * (kk / 2) + 2 * (lane / 32) + kk % 2;
      a[s][kk] = *reinterpret_cast<const u32x4_t*>(a_row + step * 64 + chunk * 8);
    }
  };
  f32x16_t acc[kMatrices];
#pragma unroll
  for (int m = 0; m < kMatrices; ++m)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[m][q] = 0.0f;
  auto multiply = [&](auto set) __attribute__((always_inline)) {
    constexpr int s = decltype(set)::value;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
#pragma unroll
      for (int m = 0; m < kMatrices; ++m) {
        bf16x8_t fragment;
        if constexpr (kFp4) {
          const float half = (kk < 2 ? __builtin_amdgcn_cvt_f32_fp8(fp4_bytes[s][m], 0) : __builtin_amdgcn_cvt_f32_fp8(fp4_bytes[s][m], 1)) * 0.00390625f;
          const uint32_t word = b[s][m][0][kk];
          fragment = FORMAT == DEW_MOE_W_MXFP4 ? fragment_fp4_pow2(word, half) : fragment_fp4(word, half);
        } else if constexpr (kBf16) {
          fragment = __builtin_bit_cast(bf16x8_t, b[s][m][kk % kAtoms]);
        } else {
          const u32x4_t& raw = b[s][m][kk / 2 % kAtoms];
          fragment = fragment_fp8(raw[2 * (kk % 2)], raw[2 * (kk % 2) + 1], FORMAT == DEW_MOE_W_FP8_BLOCK ? scale[s][m] : channel_scale[m]);
        }
        acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[s][kk]), fragment, acc[m], 0, 0, 0);
      }
  };
  static_for<kAhead>([&](auto set) { load(set, min(decltype(set)::value, steps - 1)); });
  // where the rows' results go, asked for behind the first loads
  const int out_row = p.scatter ? p.scatter[sorted_row] : sorted_row;
  int step = 0;
  for (; step + 2 * kAhead <= steps; step += kAhead)
    static_for<kAhead>([&](auto set) {
      multiply(set);
      load(set, step + decltype(set)::value + kAhead);
    });
  // (the last one to two rounds; a load past the depth is the last step's again, which multiplies nothing)
  static_for<kAhead>([&](auto set) {
    if (step + decltype(set)::value < steps) multiply(set);
    load(set, min(step + decltype(set)::value + kAhead, steps - 1));
  });
  static_for<kAhead>([&](auto set) {
    if (step + decltype(set)::value + kAhead < steps) multiply(set);
  });

  const float factor0 = kFp4 ? 256.0f * p.w0.tensor_scale[expert] : 1.0f, factor1 = kFp4 && kPaired ? 256.0f * p.w1.tensor_scale[expert] : 1.0f;
  const int column = strip * 32 + lane % 32;
  float bias = (!kPaired && p.bias) ? p.bias[static_cast<size_t>(expert) * p.width + column] : 0.0f;
  if (p.round_bias) bias = bf16_round(bias);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    if (8 * (q / 4) >= valid_rows) continue;  // (the same for every lane)
    const int row = 8 * (q / 4) + 4 * (lane / 32) + q % 4;
    const int to = __shfl(out_row, row, 64);
    bf16_t value;
    if constexpr (kPaired) {
      value = gated_rounded(acc[0][q] * factor0, acc[kMatrices - 1][q] * factor1, p.limit, p.gating);
    } else if constexpr (kGated) {  // an even lane holds a gate column, the odd one beside it its up column
      const float mine = bf16_round(acc[0][q] * factor0 + bias);
      const float other = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, mine), 0xB1, 0xF, 0xF, true));
      value = gated_pair_rounded(mine, other, p.limit);
    } else {
      value = f32_to_bf16(acc[0][q] * factor0 + bias);
    }
    if (row < valid_rows && (!kGated || lane % 2 == 0)) p.out[static_cast<size_t>(to) * out_width + (kGated ? column / 2 : column)] = value;
  }
}

template <int FORMAT, int MODE>
static int launch_few(const char* who, const GemmParams& p, hipStream_t stream) {
  // every expert with rows ends in one partial tile, and the rows no expert owns fill tiles behind them
  const int tiles = min(p.rows, p.rows / 32 + p.experts + 1), blocks = tiles * (p.width / 32);
  hipLaunchKernelGGL((few_tiles_kernel<FORMAT, MODE>), dim3(blocks), dim3(64), 0, stream, p);
  return launched(who);
}

template <int MODE>
static int launch_few_format(const char* who, const GemmParams& p, int format, hipStream_t stream) {
  switch (format) {
    case DEW_MOE_W_FP8_BLOCK: return launch_few<DEW_MOE_W_FP8_BLOCK, MODE>(who, p, stream);
    case DEW_MOE_W_FP8_CHANNEL: return launch_few<DEW_MOE_W_FP8_CHANNEL, MODE>(who, p, stream);
    case DEW_MOE_W_MXFP4: return launch_few<DEW_MOE_W_MXFP4, MODE>(who, p, stream);
    case DEW_MOE_W_BF16: return launch_few<DEW_MOE_W_BF16, MODE>(who, p, stream);
    default: return launch_few<DEW_MOE_W_NVFP4, MODE>(who, p, stream);
  }
}

int launch_few_tiles(const char* who, const GemmParams& p, int format, int mode, hipStream_t stream) {
  switch (mode) {
    case kSwigluOfTwo: return launch_few_format<kSwigluOfTwo>(who, p, format, stream);
    case kInterleavedGated: return launch_few_format<kInterleavedGated>(who, p, format, stream);
    default: return launch_few_format<kPlain>(who, p, format, stream);
  }
}

}  // namespace dew
