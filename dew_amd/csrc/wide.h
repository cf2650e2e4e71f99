// What the launches of 256 x 256 tiles on blocks that stay share (wide.hip: plain bf16 operands; wide_fp8.hip: the recipes' e4m3 ones):
// a block's tiles, one after another, and a finished tile's way out.
#pragma once

#include <math.h>

#include "common.h"
#include "gemm.h"

namespace dew {

constexpr int kWideThreads = 256, kWideTile = 256;
constexpr int kWideGroups = 256;  // groups that such a launch keeps the tiles of in registers

// The 256 x 256 tiles of a launch, of which a CU takes one a round. A kernel's gradient knows its tiles; a product's are a guess, since its
// groups end where they end: about kGuessed of them may not be there, or more.
constexpr int kGuessed = 8;
inline double product_tiles(int rows, int groups, int width) { return (rows / 256.0 + groups / 2.0) * ((width + 255) / 256); }

inline double gradient_tiles(int groups, int depth, int width) { return static_cast<double>(groups) * ((depth + 255) / 256) * ((width + 255) / 256); }

inline double gradient_quarters(int groups, int depth, int width) { return static_cast<double>(groups) * ((depth + 127) / 128) * ((width + 127) / 128); }

inline bool wide_extents(int groups, int a, int b) { return groups <= kWideGroups && a <= (1 << 20) && b <= (1 << 20); }  // (offsets within a tile are 32-bit)

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Whether a kernel's gradient leaves its last tiles in quarters; its launch carries their code only then (the registers that it keeps for it
// cost every other tile's start: e4m3, eight tiles of a few steps a block, 3 to 5 %). A product's tiles are known on the device alone.
inline bool ends_in_quarters(int groups, int depth, int width, int quarter_turns) {
  const int tiles = static_cast<int>(gradient_tiles(groups, depth, width));
  return (tiles % 256 != 0 && tiles % 256 <= 64 * quarter_turns) || (tiles < 256 && gradient_quarters(groups, depth, width) <= 256);
}

struct WidePlace {
  int group, start, size;  // the tile's group: its first row and its rows
  int within, strip;       // row tile of the group, column strip
};

// The groups' tiles and rows, a lane a group, 64 groups a register. kGradient: every group has the same row tiles, of `outer_m` rows.
template <bool kGradient>
struct WideTiles {
  static constexpr int kRounds = kWideGroups / 64;
  int first_tile[kRounds], first_row[kRounds], group_size[kRounds];
  int gradient_tiles, strips, total, held;  // `held`: rows in all groups
  int whole;                                // tiles that leave as such; those behind them in quarters
  bool fine;                                // the tiles are quarters themselves

  // The groups' first tiles of `of` rows each; how many row tiles there are.
  __device__ __forceinline__ int tabulate(int groups, int outer_m, int of) {
    const int lane = threadIdx.x % 64;
    gradient_tiles = (outer_m + of - 1) / of;
    int m_tiles = 0;
#pragma unroll
    for (int round = 0; round < kRounds; ++round) {
      const int g = 64 * round + lane;
      first_tile[round] = 0x7FFFFFFF;
      if (64 * round < groups) {
        const int tiles = g >= groups ? 0 : kGradient ? gradient_tiles : (group_size[round] + of - 1) / of, inclusive = lanes_scanned(tiles);
        if (g < groups) first_tile[round] = m_tiles + inclusive - tiles;
        m_tiles += __builtin_amdgcn_readlane(inclusive, 63);
      }
    }
    return m_tiles;
  }

  __device__ __forceinline__ void find(const int32_t* offsets, const int32_t* sizes, int groups, int outer_m, int outer_n, int quarter_turns) {
    const int lane = threadIdx.x % 64;
    held = 0;
#pragma unroll
    for (int round = 0; round < kRounds; ++round) {
      const int g = 64 * round + lane;
      first_row[round] = group_size[round] = 0;
      if (64 * round < groups) {
        const int size = g >= groups ? 0 : sizes ? max(sizes[g], 0) : max(offsets[g + 1] - offsets[g], 0);
        const int rows = lanes_scanned(size);
        if (g < groups) {
          first_row[round] = sizes ? held + rows - size : offsets[g];
          group_size[round] = size;
        }
        held += __builtin_amdgcn_readlane(rows, 63);
      }
    }
    if (!sizes) held = offsets[groups];
    strips = (outer_n + kWideTile - 1) / kWideTile;
    total = __builtin_amdgcn_readfirstlane(tabulate(groups, outer_m, kWideTile) * strips);
    const int blocks = gridDim.x, behind = total % blocks;
    whole = behind <= blocks * quarter_turns / 4 ? total - behind : total;
    fine = false;
    // A launch of one quarter a block, though its tiles have more: those past a group's rows and the columns are left out, or blocks would wait
    // a turn for them (us: 1348 rows' gradient of 2624 x 1496, 252 quarters of 66 tiles, 26.1 -> 16.4, a blockwise product of 768 rows of 2 x 5376 x 4352, 204
    // of 68, 39.4 -> 23.1).
    if (quarter_turns > 0 && total < blocks && 4 * total > blocks) {
      int row_quarters = kGradient ? groups * ((outer_m + kWideTile / 2 - 1) / (kWideTile / 2)) : 0;
#pragma unroll
      for (int round = 0; round < kRounds; ++round)
        if (!kGradient && 64 * round < groups) row_quarters += __builtin_amdgcn_readlane(lanes_scanned((group_size[round] + kWideTile / 2 - 1) / (kWideTile / 2)), 63);
      const int strip_quarters = (outer_n + kWideTile / 2 - 1) / (kWideTile / 2);
      if (row_quarters * strip_quarters <= blocks) {
        tabulate(groups, outer_m, kWideTile / 2);
        strips = strip_quarters;
        total = __builtin_amdgcn_readfirstlane(row_quarters * strip_quarters);
        whole = 0;
        fine = true;
      }
    }
  }

  // The block's quarter tile number `turn`, false past its last: its tile, and the quarter's first row in the group and column. Neighbours
  // are an XCD's, and share their operands in its L2. (Of a tile's four, some may lie past the group's rows or the columns; `fine` ones are all
  // real.)
  __device__ __forceinline__ bool quarter_at(int turn, int group_m, WidePlace& out, int& row_at, int& column) const {
    const int xcds = 8, slots = gridDim.x / xcds, count = (fine ? 1 : 4) * (total - whole), run = (count + xcds - 1) / xcds;
    const int slot = blockIdx.x / xcds + turn * slots, order = __builtin_amdgcn_readfirstlane(slot < run ? blockIdx.x % xcds * run + slot : count);
    if (order >= count) return false;
    const int quarter = fine ? 0 : order % 4, shift = fine ? 7 : 8;
    place(fine ? order : whole + order / 4, fine ? 2 * group_m : group_m, shift, out);
    row_at = (out.within << shift) + quarter / 2 * (kWideTile / 2);
    column = (out.strip << shift) + quarter % 2 * (kWideTile / 2);
    return true;
  }

  // The block's tile number `turn`, false past its last. A round of one tile a block is chunks of group_m row tiles x 8 strips, one an XCD;
  // the last round's tiles, however few, are dealt to all XCDs in equal runs. (As whole chunks they filled some XCDs and left others idle,
  // us of an MXFP8 kernel gradient's 168 tiles, 13 952 tokens of 6 x 1024 x 1664: 53 -> 49.5; of 156, 4224 of 3 x 3200 x 1024, 33.9 -> 31.5;
  // of a product's 222, [11 264, 12 800] x 1280, 159 -> 152.)
  __device__ __forceinline__ bool at(int turn, int group_m, WidePlace& out) const {
    const int xcds = 8, slots = gridDim.x / xcds, begun = turn * slots * xcds;
    const int run = min((whole - begun + xcds - 1) / xcds, slots), slot = blockIdx.x / xcds;
    const int order = __builtin_amdgcn_readfirstlane(slot < run ? begun + blockIdx.x % xcds * run + slot : whole);
    if (order >= whole) return false;
    place(order, group_m, 8, out);
    return true;
  }

  __device__ __forceinline__ void place(int order, int group_m, int shift, WidePlace& out) const {
    const int across = order / strips;  // (the tiles of a group are in a row: this many before it at most)
    int group = -1;
#pragma unroll
    for (int round = 0; round < kRounds; ++round) group += __builtin_popcountll(__ballot(first_tile[round] <= across));
    int before = 0, start = 0, size = 0;
#pragma unroll
    for (int round = 0; round < kRounds; ++round)
      if (group / 64 == round) {
        before = __builtin_amdgcn_readlane(first_tile[round], group % 64);
        start = __builtin_amdgcn_readlane(first_row[round], group % 64);
        size = __builtin_amdgcn_readlane(group_size[round], group % 64);
      }
    const int tiles = kGradient ? gradient_tiles : (size + (1 << shift) - 1) >> shift;
    const int place_in_group = order - before * strips;
    const int band = place_in_group / (group_m * strips), band_tiles = min(group_m, tiles - band * group_m), within = place_in_group % (group_m * strips);
    out = WidePlace{group, start, size, band * group_m + within % band_tiles, within / band_tiles};
  }
};

// The rows of no group are zero: rows held .. rows of `out`, `width` wide (a multiple of 8), by all of the launch's threads.
__device__ __forceinline__ void clear_unowned(bf16_t* out, int held, int rows, int width) {
  const int pieces = width / 8;
  const long long items = static_cast<long long>(max(rows - held, 0)) * pieces;
  for (long long item = static_cast<long long>(blockIdx.x) * kWideThreads + threadIdx.x; item < items; item += static_cast<long long>(gridDim.x) * kWideThreads) {
    const int row = held + static_cast<int>(item / pieces);
    *reinterpret_cast<u32x4_t*>(out + static_cast<size_t>(row) * width + item % pieces * 8) = u32x4_t{0, 0, 0, 0};
  }
}

// The sums are zero: sixteen products of zeros, in half the time of as many moves (each of its own, or the compiler makes one and copies it).
template <int kTiles>
__device__ __forceinline__ void clear_sums(f32x16_t (&acc)[kTiles][kTiles]) {
  bf16x8_t zero = __builtin_bit_cast(bf16x8_t, u32x4_t{0, 0, 0, 0});
  f32x16_t none;
#pragma unroll
  for (int q = 0; q < 16; ++q) none[q] = 0.0f;
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      asm volatile("" : "+v"(zero));
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(zero, zero, none, 0, 0, 0);
    }
}

// v[g] of lane 4 m + l becomes v[l] of lane 4 m + g.
__device__ __forceinline__ void across_quads(uint32_t (&v)[4]) {
  const int lane = threadIdx.x;
#pragma unroll
  for (int g = 0; g < 4; g += 2) {
    const uint32_t a = v[g], b = v[g + 1];
    const uint32_t a_beside = __builtin_amdgcn_mov_dpp(a, 0xB1, 0xF, 0xF, true), b_beside = __builtin_amdgcn_mov_dpp(b, 0xB1, 0xF, 0xF, true);  // quad_perm 1 0 3 2
    v[g] = lane & 1 ? b_beside : a;
    v[g + 1] = lane & 1 ? b : a_beside;
  }
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const uint32_t a = v[g], b = v[g + 2];
    const uint32_t a_beside = __builtin_amdgcn_mov_dpp(a, 0x4E, 0xF, 0xF, true), b_beside = __builtin_amdgcn_mov_dpp(b, 0x4E, 0xF, 0xF, true);  // quad_perm 2 3 0 1
    v[g] = lane & 2 ? b_beside : a;
    v[g + 2] = lane & 2 ? b : a_beside;
  }
}

// A wavefront's 128 x 128 sums leave from registers, without the LDS and without a barrier. The operands entered the instruction the
// other way round: acc[i][j][q] is row lane % 32, column 8 (q / 4) + 4 (lane / 32) + q % 4 of its 32 x 32 tile. One exchange between the
// halves of the wavefront makes a lane's sums whole pieces of 16 bytes of its row, in the left or the right of two tiles, and another within
// four lanes puts four such pieces of a row into neighbours: a store is sixteen runs of 64 bytes, both halves of eight 128-byte lines (f32:
// halves of sixteen). Stores of a row a lane, 16 bytes 64 apart, cost the L2 more than these exchanges do: us of a kernel gradient, eight
// steps and a store a tile, FP8, 32 768 tokens of 32 x 7168 x 2048, 561 -> 526 (396 without any store), of 8 x 4096 x 14 336 1510 -> 1487;
// of products, deeper, 1 to 2 % less. `out_row0`, `valid_rows`: the block's tile (what lies past the buffer's end, the rows
// past its last, and the columns sent there are not stored); `tile_row`, `column0`: the wavefront's place in it and in the row.
template <bool kOutF32, int kTiles>
__device__ __forceinline__ void leave(f32x16_t (&acc)[kTiles][kTiles], void* to_rows, size_t out_row0, int valid_rows, int width, int tile_row, int column0, float factor) {
  int lane = threadIdx.x % 64;
  asm volatile("" : "+v"(lane));
  constexpr int kOutBytes = kOutF32 ? 4 : 2;
  const __amdgpu_buffer_rsrc_t out =
      __builtin_amdgcn_make_buffer_rsrc(static_cast<uint8_t*>(to_rows) + out_row0 * width * kOutBytes, 0, valid_rows * width * kOutBytes, 0x00027000);
  constexpr uint32_t kNowhere = 0xFFFFFFF0u;
  // (row tile i's sums are in accumulation registers up to here: moved at the loop's end, all 256 at once took every other register)
  auto stay = [&](int i) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int j = 0; j < kTiles; ++j) asm volatile("" : "+a"(acc[i][j]));
#endif
  };
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    stay(i);
    const uint32_t row = tile_row + 32 * i + lane % 32 / 4 * 4;
#pragma unroll
    for (int pair = 0; pair < kTiles / 2; ++pair) {
      // the lane's row of tile 2 pair + lane / 32, in pieces of 16 bytes
      constexpr int kPieces = kOutF32 ? 8 : 4;
      uint32_t pieces[kPieces][4];
#pragma unroll
      for (int q = 0; q < 16; q += kOutF32 ? 1 : 2) {
        uint32_t words[2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const f32x16_t& sums = acc[i][2 * pair + t];
          words[t] = kOutF32 ? __float_as_uint(sums[q] * factor) : pack_bf16(sums[q] * factor, sums[q + (kOutF32 ? 0 : 1)] * factor);
        }
        const auto swapped = __builtin_amdgcn_permlane32_swap(words[0], words[1], false, false);
        const int piece = kOutF32 ? q / 4 * 2 : q / 4, word = kOutF32 ? q % 4 : q % 4 / 2;
        pieces[piece][word] = swapped[0];
        pieces[piece + (kOutF32 ? 1 : 0)][word + (kOutF32 ? 0 : 2)] = swapped[1];
      }
#pragma unroll
      for (int four = 0; four < kPieces; four += 4) {
#pragma unroll
        for (int word = 0; word < 4; ++word) {
          uint32_t v[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) v[g] = pieces[four + g][word];
          across_quads(v);
#pragma unroll
          for (int g = 0; g < 4; ++g) pieces[four + g][word] = v[g];
        }
        const int column = column0 + 64 * pair + 32 * (lane / 32) + (16 / kOutBytes) * (four + lane % 4);
        const uint32_t to = column < width ? (row * width + column) * kOutBytes : kNowhere, next_row = column < width ? width * kOutBytes : 0;
#pragma unroll
        for (int g = 0; g < 4; ++g)
          __builtin_amdgcn_raw_buffer_store_b128(u32x4_t{pieces[four + g][0], pieces[four + g][1], pieces[four + g][2], pieces[four + g][3]}, out, to + g * next_row, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
}

}  // namespace dew
