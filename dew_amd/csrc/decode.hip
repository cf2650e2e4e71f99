// The grouped product for few tiles of few rows: a decode step of one or a few tokens.
//
// The tiled launch gives a tile of an expert's rows and 128 columns to a block of four wavefronts that share the rows in the
// LDS. One token's eight experts of 768 columns are then 48 blocks, and 208 CUs idle. Two launches of finer tiles stand in for it:
//  * few_tiles_kernel: a wavefront is a block of its own and owns 32 columns (of both matrices of a pair): the same wavefronts, but on as
//    many CUs, each with the memory pipeline to itself and, with no barrier and no LDS stage a step, as much of its weights in flight as the
//    registers hold. The rows are few, so their fragments come straight from global memory (the lanes past a group's rows read its last
//    row again, the same cache lines).
//  * shared_strips_kernel, where even such strips are few: several wavefronts share a strip's depth and keep the rows in the LDS.
// Every sum is taken in the tiled launches' order (a wavefront that shares a strip goes on from the sums of the one before), so a
// product's bits do not depend on which of them ran.
#include <mutex>

#include "gemm.h"
#include "wide.h"

namespace dew {

constexpr int kFewRows = 32;

// Which expert owns row tile `m_tile` (-1: past the last tile)? Every wavefront scans the groups for itself, 64 a round, without a barrier.
struct FewTile {
  int expert, row0, end;      // the tile's first row, its group's end
  int carried, carried_rows;  // past the last tile: the tiles and (of group sizes) the rows of all groups
};
__device__ __forceinline__ FewTile few_tile(const GemmParams& p, int m_tile) {
  const int lane = threadIdx.x % 64;
  auto size_of = [&p](int e) { return e >= p.experts ? 0 : p.sizes ? max(p.sizes[e], 0) : p.offsets[e + 1] - p.offsets[e]; };
  auto first_row_of = [&p](int e) { return e >= p.experts || p.sizes ? 0 : p.offsets[e]; };
  FewTile tile{-1, 0, 0, 0, 0};
  int next_size = size_of(lane), next_first = first_row_of(lane);
  for (int base = 0; base < p.experts; base += 64) {
    const int size = next_size;
    int start = next_first;
    next_size = size_of(base + 64 + lane);
    next_first = first_row_of(base + 64 + lane);
    if (p.sizes) {
      const int rows = lanes_scanned(size);
      start = tile.carried_rows + rows - size;
      tile.carried_rows += __builtin_amdgcn_readlane(rows, 63);
    }
    const int tiles = (size + kFewRows - 1) / kFewRows, inclusive = lanes_scanned(tiles), first = tile.carried + inclusive - tiles;
    const unsigned long long hit = __ballot(m_tile >= first && m_tile < first + tiles);
    if (hit != 0ull) {
      const int owner = __builtin_ctzll(hit);
      tile.expert = base + owner;
      tile.row0 = __builtin_amdgcn_readlane(start + (m_tile - first) * kFewRows, owner);
      tile.end = __builtin_amdgcn_readlane(start + size, owner);
      break;
    }
    tile.carried += __builtin_amdgcn_readlane(inclusive, 63);
  }
  return tile;
}

// Past the last tile: the rows that no expert owns are zero.
template <int kOutColumns>
__device__ __forceinline__ void clear_past_last(const GemmParams& p, int m_tile, const FewTile& tile, int strip, int out_width) {
  const int tail_begin = (p.sizes ? tile.carried_rows : p.offsets[p.experts]) + (m_tile - tile.carried) * kFewRows;
  const int tail_end = min(tail_begin + kFewRows, p.rows);
  for (int item = threadIdx.x; item < (tail_end - tail_begin) * (kOutColumns / 8); item += blockDim.x) {
    const int sorted = tail_begin + item / (kOutColumns / 8), row = p.scatter ? p.scatter[sorted] : sorted;
    *reinterpret_cast<u32x4_t*>(p.out + static_cast<size_t>(row) * out_width + strip * kOutColumns + item % (kOutColumns / 8) * 8) = u32x4_t{0, 0, 0, 0};
  }
}

// The down product of a few tokens and their weighted sums as one launch (COMBINED): a block is a token's 32 output columns, a wavefront one of the
// token's slots, whose row it multiplies as a tile of its own; the slots' rounded outputs meet in the LDS and are summed as the combine's
// own launch sums them (combine.hip), so the bits are the two launches'. What bounds a step on small experts is its launches, one behind the
// other, and the host that issues them: one of 2 to 3 us, and some 3 us of the host's, fall away (`combines_few`).
struct CombineParams {
  const float* weights;  // [tokens, top_k]
  bf16_t* out;           // [tokens, width]
  int tokens, top_k, shared;
};

// (each product and each sum rounded by itself)
__device__ __forceinline__ float weighted_sum(const float* values, int pitch, const float* weights, int top_k) {
#pragma clang fp contract(off)
  float sum = 0.0f;
  for (int j = 0; j < top_k; ++j) {
    const float product = values[j * pitch] * weights[j];
    sum = sum + product;
  }
  return sum;
}

// The tile of a slot's one row: its sorted position, and the group that holds it.
__device__ __forceinline__ FewTile slot_tile(const GemmParams& p, int slot) {
  const int lane = threadIdx.x % 64;
  FewTile tile{0, 0, 0, 0, 0};
  for (int base = 0; base < p.rows; base += 64) {
    const unsigned long long hit = __ballot(base + lane < p.rows && p.scatter[min(base + lane, p.rows - 1)] == slot);
    if (hit != 0ull) tile.row0 = base + __builtin_ctzll(hit);
  }
  for (int base = 0; base < p.experts; base += 64) {
    const int e = min(base + lane, p.experts - 1);
    const int begin = p.offsets[e], end = p.offsets[e + 1];
    const unsigned long long hit = __ballot(base + lane < p.experts && tile.row0 >= begin && tile.row0 < end);
    if (hit != 0ull) tile.expert = base + __builtin_ctzll(hit);
  }
  tile.end = tile.row0 + 1;
  return tile;
}

template <int FORMAT, int MODE, bool COMBINED>
__device__ __forceinline__ void few_tile_product(const GemmParams& p, const CombineParams& c) {
  static_assert(!COMBINED || MODE == kPlain, "the down product");
  constexpr bool kPaired = MODE == kSwigluOfTwo, kGated = MODE == kInterleavedGated;
  constexpr bool kFp4 = FORMAT == DEW_MOE_W_NVFP4 || FORMAT == DEW_MOE_W_MXFP4, kBf16 = FORMAT == DEW_MOE_W_BF16;
  constexpr int kMatrices = kPaired ? 2 : 1;
  constexpr int kAtomK = kFp4 ? 64 : kBf16 ? 16 : 32, kAtoms = 64 / kAtomK;  // 16-byte loads a lane makes per matrix and 64 depths
  constexpr int kAhead = kMatrices * kAtoms >= 8 ? 4 : kMatrices * kAtoms >= 4 ? 6 : 8;  // steps of 64 depths in flight
  const int lane = COMBINED ? threadIdx.x % 64 : threadIdx.x, wave = COMBINED ? __builtin_amdgcn_readfirstlane(threadIdx.x / 64) : 0;
  const int strips = p.width / 32, m_tile = blockIdx.x / strips /* COMBINED: the token */, strip = blockIdx.x % strips;
  // (the shared expert's rows are the last slots)
  const int slot = !COMBINED ? 0 : wave < c.top_k ? m_tile * c.top_k + wave : c.tokens * c.top_k + m_tile;

  FewTile tile;
  if constexpr (COMBINED)
    tile = slot_tile(p, slot);
  else
    tile = few_tile(p, m_tile);
  const int expert = tile.expert, row0 = tile.row0;
  const int out_width = kGated ? p.width / 2 : p.width;
  constexpr int kOutColumns = kGated ? 16 : 32;
  if (!COMBINED && expert < 0) {
    clear_past_last<kOutColumns>(p, m_tile, tile, strip, out_width);
    return;
  }
  const int valid_rows = min(kFewRows, tile.end - row0);

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
  const int out_row = !COMBINED && p.scatter ? p.scatter[sorted_row] : sorted_row;
  const float share = COMBINED && wave < c.top_k ? c.weights[slot] : 0.0f;
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
  if constexpr (COMBINED) {
    __shared__ float outputs[kMostCombinedSlots][32];
    __shared__ float shares[kMostCombinedSlots];
    if (lane < 32) outputs[wave][lane] = bf16_round(acc[0][0] * factor0 + bias);  // (row 0 of the tile, whose rows are all the slot's)
    if (lane == 0) shares[wave] = share;
    __syncthreads();
    if (threadIdx.x < 32) {
      const float sum = weighted_sum(&outputs[0][lane], 32, shares, c.top_k);
      c.out[static_cast<size_t>(m_tile) * p.width + column] = c.shared ? f32_to_bf16(bf16_round(sum) + outputs[c.top_k][lane]) : f32_to_bf16(sum);
    }
    return;
  }
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
__global__ __launch_bounds__(64) void few_tiles_kernel(GemmParams p) {
  few_tile_product<FORMAT, MODE, false>(p, CombineParams{});
}

template <int FORMAT>
__global__ __launch_bounds__(64 * kMostCombinedSlots) void few_combined_kernel(GemmParams p, CombineParams c) {
  few_tile_product<FORMAT, kPlain, true>(p, c);
}

// Where strips are so few that most CUs have none, a block owns the 32 columns: of a pair each matrix has wavefronts of its own, and
// kShares wavefronts share a matrix's depth in chunks of four steps, dealt round. Each has its chunks' weights fetched and brought to bf16
// while the others multiply; what it multiplies it adds to the one before's sums, handed on through the LDS: every sum is still taken in
// the tiled launches' order. The rows, which are few, are in the LDS.
// One wavefront for a strip of both matrices spent 19 000 of its 28 000 cycles (2048 deep, FP8 blocks) on what is here 8 turns of 1000, half
// of them matrix instructions: one token's 8 experts of 2048 x 768 15.0 -> 11.5 us. FP8 and NVFP4 banks (`launch_few`).
constexpr int kShares = 4, kMostShared = 131072;  // bytes of rows that a block may keep
constexpr int shared_pitch(int depth) { return depth * 2 + 16; }  // (a row's LDS bytes: 32 rows' pieces on different banks)

template <int FORMAT, int MODE>
__global__ __launch_bounds__(64 * kShares * (MODE == kSwigluOfTwo ? 2 : 1)) void shared_strips_kernel(GemmParams p) {
  constexpr bool kPaired = MODE == kSwigluOfTwo, kGated = MODE == kInterleavedGated;
  constexpr bool kFp4 = FORMAT == DEW_MOE_W_NVFP4;
  constexpr int kMatrices = kPaired ? 2 : 1;
  constexpr int kAtomK = kFp4 ? 64 : 32, kAtoms = 64 / kAtomK;  // 16-byte loads a lane makes per matrix and 64 depths
  constexpr int kChunk = 4, kSets = kFp4 ? 3 : 2;  // steps of 64 depths a turn; chunks of weights in flight
  constexpr int kWaves = kMatrices * kShares;
  __shared__ f32x4_t handed[kMatrices][4 * 64];  // a matrix's sums on their way from one wavefront to the next, [quad][lane]
  __shared__ int turn[kMatrices];                // the chunk that they are for
  extern __shared__ u32x4_t shared_rows[];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), matrix = wave % kMatrices, share = wave / kMatrices;
  const int strips = p.width / 32, m_tile = blockIdx.x / strips, strip = blockIdx.x % strips;

  const FewTile tile = few_tile(p, m_tile);
  const int expert = tile.expert, row0 = tile.row0;
  const int out_width = kGated ? p.width / 2 : p.width;
  constexpr int kOutColumns = kGated ? 16 : 32;
  if (expert < 0) {
    clear_past_last<kOutColumns>(p, m_tile, tile, strip, out_width);
    return;
  }
  const int valid_rows = min(kFewRows, tile.end - row0);

  const int steps = p.depth / 64, chunks = (steps + kChunk - 1) / kChunk;
  const int k_atoms = p.depth / kAtomK;
  const size_t first_atom = (static_cast<size_t>(expert) * strips + strip) * k_atoms;
  const BankView bank = matrix == 0 ? p.w0 : p.w1;
  const uint8_t* b_src = bank.codes + first_atom * kAtomBytes + lane * 16;
  const uint8_t* b_scale_src = kFp4 ? static_cast<const uint8_t*>(bank.scales) + first_atom * 128 + lane * 2 : nullptr;
  const float* block_scales =
      FORMAT == DEW_MOE_W_FP8_BLOCK ? static_cast<const float*>(bank.scales) + static_cast<size_t>(expert) * (p.depth / 128) * (p.width / 128) + strip / 4 : nullptr;
  const int sorted_row = row0 + min(lane % 32, valid_rows - 1);
  // The tile's rows, 16 bytes a thread at a time: a thread's first piece is asked for behind its weights, the row's index ahead of them
  // (loads return in order).
  const int pieces = p.depth / 8, pitch = shared_pitch(p.depth) / 16, row_pieces = valid_rows * pieces;
  const int first_row = row0 + min(static_cast<int>(threadIdx.x) / pieces, valid_rows - 1), first_source = p.gather ? p.gather[first_row] : first_row;
  u32x4_t b[kSets][kChunk][kAtoms];
  uint32_t fp4_bytes[kSets][kChunk];
  float scale[kSets][kChunk];
  bf16x8_t fragment[kChunk][4];
  auto load_weights = [&](auto set, int chunk) __attribute__((always_inline)) {
    constexpr int s = decltype(set)::value;
    if (chunk >= chunks) return;  // (the same for the wavefront)
#pragma unroll
    for (int c = 0; c < kChunk; ++c) {
      const int step = min(chunk * kChunk + c, steps - 1);  // (past the depth: the last step's again, which multiplies nothing)
#pragma unroll
      for (int i = 0; i < kAtoms; ++i)
        b[s][c][i] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(b_src + (static_cast<size_t>(step) * kAtoms + i) * kAtomBytes));
      if constexpr (kFp4) fp4_bytes[s][c] = *reinterpret_cast<const uint16_t*>(b_scale_src + static_cast<size_t>(step) * 128);
      if constexpr (FORMAT == DEW_MOE_W_FP8_BLOCK) scale[s][c] = block_scales[static_cast<size_t>(step / 2) * (p.width / 128)];
    }
  };
  static_for<kSets>([&](auto set) { load_weights(set, share + decltype(set)::value * kShares); });
  const float channel_scale = FORMAT == DEW_MOE_W_FP8_CHANNEL ? static_cast<const float*>(bank.scales)[static_cast<size_t>(expert) * p.width + strip * 32 + lane % 32] : 1.0f;
  const u32x4_t first_piece = *reinterpret_cast<const u32x4_t*>(p.x + static_cast<size_t>(first_source) * p.depth + threadIdx.x % pieces * 8);
  // where the rows' results go, asked for behind the first loads
  const int out_row = p.scatter ? p.scatter[sorted_row] : sorted_row;
  const float factor0 = kFp4 ? 256.0f * p.w0.tensor_scale[expert] : 1.0f, factor1 = kFp4 && kPaired ? 256.0f * p.w1.tensor_scale[expert] : 1.0f;
  const int column = strip * 32 + lane % 32;
  float bias = (!kPaired && p.bias) ? p.bias[static_cast<size_t>(expert) * p.width + column] : 0.0f;
  if (p.round_bias) bias = bf16_round(bias);
  auto convert = [&](auto set) __attribute__((always_inline)) {
    constexpr int s = decltype(set)::value;
#pragma unroll
    for (int c = 0; c < kChunk; ++c)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) {
        if constexpr (kFp4) {
          const float half = (kk < 2 ? __builtin_amdgcn_cvt_f32_fp8(fp4_bytes[s][c], 0) : __builtin_amdgcn_cvt_f32_fp8(fp4_bytes[s][c], 1)) * 0.00390625f;
          fragment[c][kk] = fragment_fp4(b[s][c][0][kk], half);
        } else {
          const u32x4_t& raw = b[s][c][kk / 2 % kAtoms];
          fragment[c][kk] = fragment_fp8(raw[2 * (kk % 2)], raw[2 * (kk % 2) + 1], FORMAT == DEW_MOE_W_FP8_BLOCK ? scale[s][c] : channel_scale);
        }
        asm volatile("" : "+v"(fragment[c][kk]));  // (here, and not where it is multiplied)
      }
  };
  if (share < chunks) convert(std::integral_constant<int, 0>{});
  if (threadIdx.x < kMatrices) turn[threadIdx.x] = 0;
  if (static_cast<int>(threadIdx.x) < row_pieces) shared_rows[threadIdx.x / pieces * pitch + threadIdx.x % pieces] = first_piece;
  for (int item = threadIdx.x + 64 * kWaves; item < row_pieces; item += 64 * kWaves) {
    const int row = item / pieces, piece = item % pieces, source = p.gather ? p.gather[row0 + row] : row0 + row;
    shared_rows[row * pitch + piece] = *reinterpret_cast<const u32x4_t*>(p.x + static_cast<size_t>(source) * p.depth + piece * 8);
  }
  asm volatile("" ::: "memory");  // (a barrier that leaves the loads in flight)
  __builtin_amdgcn_s_waitcnt(0xF | (3 << 14) | (7 << 4));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // slice kk of a step: the 8 depths that the lane's weight bytes of that slice cover
  const u32x4_t* a_row = shared_rows + min(lane % 32, valid_rows - 1) * pitch;
  u32x4_t a[2][4];
  auto fetch = [&](auto into, int step) __attribute__((always_inline)) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      const int piece = kFp4 ? 4 * (lane / 32) + kk : 4 * (kk / 2) + 2 * (lane / 32) + kk % 2;
      a[decltype(into)::value][kk] = a_row[min(step, steps - 1) * 8 + piece];
    }
  };
  f32x16_t acc;
#pragma unroll
  for (int q = 0; q < 16; ++q) acc[q] = 0.0f;
  // the sums of the chunks before, once they are there (the wavefronts of a block run together: each turn comes)
  auto take = [&](int chunk) __attribute__((always_inline)) {
    if (chunk == 0) return;
    while (__hip_atomic_load(&turn[matrix], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != chunk) {
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (8 * i >= valid_rows) break;  // (the same for the wavefront: sums of no row)
      const f32x4_t quad = handed[matrix][i * 64 + lane];
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[4 * i + q] = quad[q];
    }
  };
  auto hand_on = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (8 * i < valid_rows) handed[matrix][i * 64 + lane] = f32x4_t{acc[4 * i], acc[4 * i + 1], acc[4 * i + 2], acc[4 * i + 3]};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    if (lane == 0) __hip_atomic_store(&turn[matrix], chunk + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto multiply = [&](int chunk) __attribute__((always_inline)) {  // (its first rows are fetched)
    static_for<kChunk>([&](auto of) __attribute__((always_inline)) {
      constexpr int c = decltype(of)::value;
      if (chunk * kChunk + c >= steps) return;
      if constexpr (c + 1 < kChunk) fetch(std::integral_constant<int, (c + 1) % 2>{}, chunk * kChunk + c + 1);
#pragma unroll
      for (int kk = 0; kk < 4; ++kk)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a[c % 2][kk]), fragment[c][kk], acc, 0, 0, 0);
    });
  };
  for (int chunk = share; chunk < chunks;) {
    static_for<kSets>([&](auto set) __attribute__((always_inline)) {
      constexpr int s = decltype(set)::value;
      if (chunk >= chunks) return;
      load_weights(set, chunk + kSets * kShares);  // (the set's weights are fragments now)
      fetch(std::integral_constant<int, 0>{}, chunk * kChunk);
      take(chunk);
      multiply(chunk);
      hand_on(chunk);
      chunk += kShares;
      if (chunk < chunks) convert(std::integral_constant<int, (s + 1) % kSets>{});
    });
  }
  __syncthreads();

  // ---- a wavefront leaves every kWaves'th of the sixteen sums a lane ----
#pragma unroll
  for (int i = 0; i < 16 / kWaves; ++i) {
    const int q = i * kWaves + wave;
    if (8 * (q / 4) >= valid_rows) continue;  // (the same for every lane)
    const int row = 8 * (q / 4) + 4 * (lane / 32) + q % 4;
    const int to = __shfl(out_row, row, 64);
    const float sum = handed[0][q / 4 * 64 + lane][q % 4];
    bf16_t value;
    if constexpr (kPaired) {
      value = gated_rounded(sum * factor0, handed[kMatrices - 1][q / 4 * 64 + lane][q % 4] * factor1, p.limit, p.gating);
    } else if constexpr (kGated) {  // an even lane holds a gate column, the odd one beside it its up column
      const float mine = bf16_round(sum * factor0 + bias);
      const float other = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, mine), 0xB1, 0xF, 0xF, true));
      value = gated_pair_rounded(mine, other, p.limit);
    } else {
      value = f32_to_bf16(sum * factor0 + bias);
    }
    if (row < valid_rows && (!kGated || lane % 2 == 0)) p.out[static_cast<size_t>(to) * out_width + (kGated ? column / 2 : column)] = value;
  }
}

template <int FORMAT, int MODE>
static int launch_few(const char* who, const GemmParams& p, hipStream_t stream) {
  // every expert with rows ends in one partial tile, and the rows no expert owns fill tiles behind them
  const int tiles = min(p.rows, p.rows / 32 + p.experts + 1), blocks = tiles * (p.width / 32);
  // Shared strips: formats whose conversion costs more than the product, deep enough that the hand-overs are few beside it, and at most one
  // block a CU (us, a wavefront a strip and shared). Pairs, whose blocks hold twice the wavefronts, gain from 1024 deep on: FP8 blocks, 1024 x 2048
  // of one row 7.5 and 6.2, of four 8.2 and 7.9, 4096 x 512 of one 21.5 and 12.4 (640 deep a layer's pass 25.6 and 26.9). One matrix, whose every turn
  // waits for the one before: FP8 blocks, 3072 deep 10.2 and 10.2 to 10.9 and 12.0; 4096, 128 strips, 12.9 and 12.5, 256 13.5 and 14.2; 6144, 256, 18.9
  // and 18.4; NVFP4, 4096, 256 strips, 14.3 and 13.9. At 512 strips, two blocks a CU where their rows leave room, else two rounds, FP8 4096 deep 16.4
  // and 19.9, 6144 deep of eight rows 23.1 and 34.6, NVFP4 22.5 and 33.6. (MXFP4, whose conversion is one instruction for two codes, 1408
  // deep 37.7 and 40.5 a layer's pass; bf16, which has none, 1152 deep 23.6 and 25.7.)
  if constexpr (FORMAT == DEW_MOE_W_FP8_BLOCK || FORMAT == DEW_MOE_W_FP8_CHANNEL || FORMAT == DEW_MOE_W_NVFP4) {
    constexpr int kMatrices = MODE == kSwigluOfTwo ? 2 : 1;
    const long long strips = (min(p.rows, p.experts) + p.rows / 32) * static_cast<long long>(p.width / 32);  // of the tiles that have rows, at most
    const int least_depth = kMatrices == 2 ? 1024 : FORMAT == DEW_MOE_W_NVFP4 || strips <= 128 ? 4096 : 6144;
    const size_t rows_bytes = static_cast<size_t>(min(p.rows, 32)) * shared_pitch(p.depth);
    if (p.depth >= least_depth && strips <= 256 && rows_bytes <= kMostShared) {
      auto kernel = shared_strips_kernel<FORMAT, MODE>;
      static std::once_flag configured;  // dynamic LDS above 64 KiB must be opted into once per kernel
      static hipError_t reserved = hipSuccess;
      std::call_once(configured, [&] { reserved = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kMostShared); });
      if (reserved != hipSuccess) return fail(DEW_MOE_ELAUNCH, "%s: cannot reserve %d bytes of LDS", who, kMostShared);
      hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * kMatrices * kShares), rows_bytes, stream, p);
      return launched(who);
    }
  }
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

int launch_few_combined(const char* who, const GemmParams& p, int format, const float* weights, int tokens, int top_k, bool shared, void* out, hipStream_t stream) {
  const CombineParams c{weights, static_cast<bf16_t*>(out), tokens, top_k, shared ? 1 : 0};
  const dim3 grid(tokens * (p.width / 32)), block(64 * (top_k + c.shared));
  switch (format) {
    case DEW_MOE_W_FP8_BLOCK: hipLaunchKernelGGL(few_combined_kernel<DEW_MOE_W_FP8_BLOCK>, grid, block, 0, stream, p, c); break;
    case DEW_MOE_W_FP8_CHANNEL: hipLaunchKernelGGL(few_combined_kernel<DEW_MOE_W_FP8_CHANNEL>, grid, block, 0, stream, p, c); break;
    case DEW_MOE_W_MXFP4: hipLaunchKernelGGL(few_combined_kernel<DEW_MOE_W_MXFP4>, grid, block, 0, stream, p, c); break;
    case DEW_MOE_W_BF16: hipLaunchKernelGGL(few_combined_kernel<DEW_MOE_W_BF16>, grid, block, 0, stream, p, c); break;
    default: hipLaunchKernelGGL(few_combined_kernel<DEW_MOE_W_NVFP4>, grid, block, 0, stream, p, c);
  }
  return launched(who);
}

}  // namespace dew
