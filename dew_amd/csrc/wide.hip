// Grouped products of plain bf16 operands in 256 x 256 tiles: the operands and results of bf16.hip, in rows as they lie, with the same
// bits (the sums run along the contraction in the same order).
//
// A 128 x 256 tile of 32-deep steps asks its CU for 48 bytes a clock at the matrix pipe's rate and the L1 gives 64 at best: those launches
// ran the pipe 38 to 43 % busy. Here a step is 64 KB for 2048 cycles of the pipe, 32 a clock, and whole cache lines either way round.
//  * 256 blocks of 4 wavefronts, one a CU, that stay and take tile after tile: the loads run on into the next tile while one leaves.
//    2 x 2 wavefronts of 128 x 128, their 256 sums a lane in the accumulation registers: 8 fragments read from the LDS for 16 matrix
//    instructions (8 wavefronts of 128 x 64 read half as much again, and were 5 to 10 % slower).
//  * All 160 KB of the LDS: a ring of three stages of the first operand and two of the second, so that of a step's sixteen loads a
//    wavefront one goes out every fourth matrix instruction. In bursts they filled the L1's queue, and the wavefront behind them
//    stopped: 16 384 x 4096 x 4096 515 us against 409.
//  * Loads through a buffer descriptor a step, whose end is the tile's last row (a gradient's: the group's): what lies past it arrives as
//    zeros, without a compare a lane.
//  * Everything between two matrix instructions is placed by hand (`phase`): one wavefront a SIMD issues an instruction every four
//    cycles, eight a matrix instruction, and what stood between the phases was time the pipe lost.
//  * The tiles behind the last whole round are cut in quarters (`quarter_tiles`) where these go round, so that a launch of 1.1 rounds takes
//    1.2 and not 2, and launches of a few tiles are worth their start.
//  * The operands enter the instruction the other way round, so that a lane holds four neighbouring columns of a row; two exchanges
//    between lanes make them runs of 64 bytes, and the tile leaves from registers, without the LDS and without a barrier (wide.h).
//
// us, in 128 x 256 tiles and here: 16 384 x 4096 x 4096 forward 517 and 445 (on another box 468 and 409, 1.34 PFLOP/s; the pipe 75 % busy
// at 1.55 to 1.8 GHz, profiles/wide_tiles_mfma_utilisation.txt), input's gradient 543 and 404, kernel's gradient 498 and 403; 10 007 rows of 16 x
// 2048 x 4096 187 and 165, 235 and 183 (1.5 rounds of tiles), 215 and 178 (268 MB written).
#include <mutex>

#include "dense.h"
#include "gemm.h"
#include "wide.h"

namespace dew {

constexpr int kWideStep = 64;
constexpr int kWideLoads = 8;                                      // 1 KiB loads of each operand that a wavefront makes a step
constexpr int kOperandBytes = kWideTile * kWideStep * 2;           // 32 KB: one operand's stage
constexpr int kFirstStages = 3, kSecondStages = 2;                 // of the first operand's ring and the second's
constexpr int kWideShared = (kFirstStages + kSecondStages) * kOperandBytes;  // all of the LDS

typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

// One operand as it is staged. kAcross false: kExtent rows of 64 depths (128 bytes, chunk index xor-swizzled as in the tiled launch);
// kAcross true: 64 rows of kExtent columns in units of 32 columns (64 bytes) whose index is xor-ed with the row mod 4.
template <bool kAcross, int kExtent>
struct WideOperand {
  static constexpr int kRowLanes = kAcross ? kExtent / 8 : 8, kRowBytes = kRowLanes * 16;
  static __device__ __forceinline__ int row(int load, int lane) { return load * (64 / kRowLanes) + lane / kRowLanes; }
  static __device__ __forceinline__ int chunk(int row, int lane) {  // the 16 bytes of the row that the lane fetches
    if (kAcross) return ((lane % kRowLanes / 4) ^ (row & 3)) * 4 + lane % 4;
    return (lane % 8) ^ (((row >> 1) & 7) ^ ((row & 1) << 2));
  }
  // Address `which` of a lane: of slice `which` (rows along the contraction; the tiles are then constants apart), or of tile
  // `which` (across; the slices are).
  static __device__ __forceinline__ uint32_t address(uint32_t base, int first_tile, int which, int lane) {
    if (kAcross) {
      const int piece = lane % 16;
      return base + (8 * (lane / 32) + piece / 4) * kRowBytes + (((first_tile + which) ^ (piece / 4)) * 64) + (lane / 16 % 2) * 32 + (piece % 4) * 8;
    }
    const int row = 32 * first_tile + lane % 32;
    return base + row * 128 + (((2 * which + lane / 32) ^ (((row >> 1) & 7) ^ ((row & 1) << 2))) * 16);
  }
};

// (Written out: the compiler takes any LDS-DMA load in flight for a write these reads may depend on, and would drain the
// memory pipeline in front of them. What they return is used behind an explicit wait: `arrived`.)
template <bool kAcross, int kExtent, int kSlice, int kTile>
__device__ __forceinline__ bf16x8_t wide_fragment(const uint32_t (&at)[4]) {
  if constexpr (kAcross) {
    u32x2_t low, high;
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(low) : "v"(at[kTile]), "n"(kSlice * 16 * kExtent * 2));
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(high) : "v"(at[kTile]), "n"((kSlice * 16 + 4) * kExtent * 2));
    return __builtin_bit_cast(bf16x8_t, u32x4_t{low[0], low[1], high[0], high[1]});
  } else {
    u32x4_t words;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(words) : "v"(at[kSlice]), "n"(kTile * 32 * 128));
    return __builtin_bit_cast(bf16x8_t, words);
  }
}

// The whole tiles, one after another.
template <bool kAAcross, bool kBAcross, bool kOutF32>
__device__ __forceinline__ void whole_tiles(const DenseParams& p, const WideTiles<kAAcross>& tiles, uint8_t* lds) {
  using A = WideOperand<kAAcross, kWideTile>;
  using B = WideOperand<kBAcross, kWideTile>;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wave_row = wave / 2, wave_column = wave % 2;  // 2 x 2 wavefronts of 128 x 128
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)lds));

  struct Tile {
    int group, row0, valid_rows, n0, m0, depth, steps;
  };
  auto tile_at = [&](int turn, Tile& tile) {
    WidePlace place;
    if (!tiles.at(turn, p.group_m, place)) return false;
    tile.group = place.group;
    tile.n0 = place.strip * kWideTile;
    if constexpr (kAAcross) {
      tile.m0 = place.within * kWideTile;
      tile.row0 = min(max(place.start, 0), p.rows);
      tile.depth = min(max(place.start + place.size, tile.row0), p.rows) - tile.row0;
      tile.valid_rows = min(kWideTile, p.outer_m - tile.m0);
      tile.steps = max((tile.depth + kWideStep - 1) / kWideStep, 1);
    } else {
      tile.m0 = 0;
      tile.row0 = place.start + place.within * kWideTile;
      tile.valid_rows = min(kWideTile, place.size - place.within * kWideTile);
      tile.depth = p.inner;
      tile.steps = p.inner / kWideStep;
    }
    return true;
  };

  // ---- what fetches: the first operand two steps ahead of what multiplies, the second one. A step's bytes are a buffer: what lies
  // past its end (the rows past a tile's last, those past a group's last) reads as zero ----
  Tile fetched;
  if (!tile_at(0, fetched)) return;  // (the same for the whole block)
  Tile tile = fetched;
  int fetched_turn = 0, fetched_step = 0, first_slot = 0, second_slot = 0;
  bool moved = false;
  const uint8_t *a_next = nullptr, *b_next = nullptr;  // the next step's bytes
  int a_bytes = 0, b_bytes = 0, a_rows = 0, b_rows = 0;
  uint32_t a_offset[kWideLoads], b_offset[kWideLoads];  // of the lane's 16 bytes of each load
  const uint32_t a_pitch = (kAAcross ? p.outer_m : p.inner) * 2, b_pitch = (kBAcross ? p.outer_n : p.inner) * 2;
  size_t a_stride = kAAcross ? static_cast<size_t>(kWideStep) * a_pitch : kWideStep * 2;
  size_t b_stride = kBAcross ? static_cast<size_t>(kWideStep) * b_pitch : kWideStep * 2;
#pragma unroll
  for (int i = 0; i < kWideLoads; ++i) {
    const int a_row = A::row(kWideLoads * wave + i, lane), b_row = B::row(kWideLoads * wave + i, lane);
    a_offset[i] = a_row * a_pitch + 16 * A::chunk(a_row, lane);
    b_offset[i] = b_row * b_pitch + 16 * B::chunk(b_row, lane);
  }
  __amdgpu_buffer_rsrc_t a_buffer, b_buffer;
  auto buffer = [](const uint8_t* at, int bytes) __attribute__((always_inline)) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(at), 0, bytes, 0x00027000); };
  auto aim_first = [&]() __attribute__((always_inline)) {
    if constexpr (kAAcross) {
      a_next = reinterpret_cast<const uint8_t*>(p.a) + static_cast<size_t>(fetched.row0) * a_pitch + fetched.m0 * 2;
      a_rows = fetched.depth;
    } else {
      a_next = reinterpret_cast<const uint8_t*>(p.a) + static_cast<size_t>(fetched.row0) * a_pitch;
      a_bytes = fetched.valid_rows * a_pitch;
    }
  };
  auto aim_second = [&]() __attribute__((always_inline)) {
    if constexpr (kAAcross) {
      b_next = reinterpret_cast<const uint8_t*>(p.b) + static_cast<size_t>(fetched.row0) * b_pitch + fetched.n0 * 2;
      b_rows = fetched.depth;
    } else {
      const uint8_t* matrix = reinterpret_cast<const uint8_t*>(p.b + static_cast<size_t>(fetched.group) * p.inner * p.outer_n);
      b_next = kBAcross ? matrix + fetched.n0 * 2 : matrix + static_cast<size_t>(fetched.n0) * b_pitch;
      b_bytes = kBAcross ? kWideStep * b_pitch - fetched.n0 * 2 : min(kWideTile, p.outer_n - fetched.n0) * b_pitch;
    }
  };
  auto next_first = [&]() __attribute__((always_inline)) {  // ahead of a step's loads of the first operand
    if (fetched_step == fetched.steps) {
      if (!tile_at(++fetched_turn, fetched)) a_stride = b_stride = 0;  // (none left: the last one's first step, again and again)
      fetched_step = 0;
      moved = true;
      aim_first();
    }
    ++fetched_step;
  };
  auto next_second = [&]() __attribute__((always_inline)) {  // of the second, which follows the first
    if (moved) {
      moved = false;
      aim_second();
    }
  };
  auto begin_first = [&]() __attribute__((always_inline)) {
    if constexpr (kAAcross) {
      a_bytes = max(min(a_rows, kWideStep) * static_cast<int>(a_pitch) - fetched.m0 * 2, 0);
      a_rows -= kWideStep;
    }
    a_buffer = buffer(a_next, a_bytes);
    a_next += a_stride;
    first_slot = first_slot == kFirstStages - 1 ? 0 : first_slot + 1;
  };
  auto begin_second = [&]() __attribute__((always_inline)) {
    if constexpr (kAAcross) {
      b_bytes = max(min(b_rows, kWideStep) * static_cast<int>(b_pitch) - fetched.n0 * 2, 0);
      b_rows -= kWideStep;
    }
    b_buffer = buffer(b_next, b_bytes);
    b_next += b_stride;
    second_slot ^= 1;
  };
  auto load_first = [&](auto piece) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void* lds_t;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(a_buffer, (lds_t)(lds + first_slot * kOperandBytes + (wave * kWideLoads + piece.value) * 1024), 16, a_offset[piece.value], 0, 0, 0);
#endif
  };
  auto load_second = [&](auto piece) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void* lds_t;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(b_buffer, (lds_t)(lds + (kFirstStages + second_slot) * kOperandBytes + (wave * kWideLoads + piece.value) * 1024), 16,
                                             b_offset[piece.value], 0, 0, 0);
#endif
  };

  // ---- what multiplies ----
  uint32_t a_at[4], b_at[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    a_at[i] = A::address(lds_base, 4 * wave_row, i, lane);
    b_at[i] = B::address(lds_base + kFirstStages * kOperandBytes, 4 * wave_column, i, lane);
  }
  f32x16_t acc[4][4];
  bf16x8_t a_frag[2][4], b_frag[2][4];
  auto clear = [&]() __attribute__((always_inline)) { clear_sums(acc); };
  auto read_piece = [&](auto slice, auto set, auto piece) __attribute__((always_inline)) {
    constexpr int s = decltype(slice)::value, i = decltype(piece)::value;
    if constexpr (i < 4) b_frag[set.value][i] = wide_fragment<kBAcross, kWideTile, s, i>(b_at);
    else if constexpr (i < 4 + 4) a_frag[set.value][i - 4] = wide_fragment<kAAcross, kWideTile, s, i - 4>(a_at);
  };
  // one phase: a slice multiplied, and in the shadows of its matrix instructions the next one's fragments read and `beside` done
  auto phase = [&](auto from, auto slice, auto into, auto&& beside) __attribute__((always_inline)) {
    static_for<16>([&](auto m) __attribute__((always_inline)) {
      constexpr int t = decltype(m)::value;
      read_piece(slice, into, m);
      acc[t / 4][t % 4] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b_frag[from.value][t % 4], a_frag[from.value][t / 4], acc[t / 4][t % 4], 0, 0, 0);
      beside(m);
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto arrived = [&](auto set) __attribute__((always_inline)) {  // this wavefront's reads are back
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xF | (7 << 4) | (3 << 14));  // lgkmcnt(0)
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(a_frag[set.value][i]));
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(b_frag[set.value][j]));
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 2> c2{};
  constexpr std::integral_constant<int, 3> c3{};
  // every wavefront's loads but its `younger` last memory operations are done, and so are its reads of the other stage
  auto landed = [&](auto younger) __attribute__((always_inline)) {
    constexpr int n = decltype(younger)::value;
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4));  // vmcnt(n) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // the loads go out one every four matrix instructions (the L1 takes them at half its rate; in bursts they held up the wavefront
  // that issued them, and its matrix instructions behind them)
  auto second_half = [&](auto m) __attribute__((always_inline)) {
    if constexpr (decltype(m)::value % 4 == 3) load_second(std::integral_constant<int, 4 + decltype(m)::value / 4>{});
  };
  clear();
  aim_first();
  aim_second();
  first_slot = kFirstStages - 1, second_slot = 1;  // (they turn ahead of each step)
  next_first();
  begin_first();
  static_for<8>(load_first);
  begin_second();
  static_for<8>(load_second);
  next_first();
  begin_first();
  static_for<8>(load_first);
  next_second();
  begin_second();
  static_for<4>(load_second);
  landed(c0);
  static_for<8>([&](auto piece) __attribute__((always_inline)) { read_piece(c0, c0, piece); });
  arrived(c0);
  int read_slot = 0, turn = 0;
  uint32_t a_move = 0, b_move = 0;
  constexpr std::integral_constant<int, 8> younger{};  // the first operand's loads of the step after the next
  for (;;) {
    for (int step = 0; step < tile.steps; ++step) {
      phase(c0, c1, c1, second_half);
      next_first();
      arrived(c1);
      phase(c1, c2, c0, [&](auto m) __attribute__((always_inline)) {
        if constexpr (decltype(m)::value == 1) begin_first();
        if constexpr (decltype(m)::value % 4 == 3) load_first(std::integral_constant<int, decltype(m)::value / 4>{});
      });
      arrived(c0);
      phase(c0, c3, c1, [&](auto m) __attribute__((always_inline)) {
        constexpr int t = decltype(m)::value;
        if constexpr (t == 1) {
          a_move = read_slot % kFirstStages == kFirstStages - 1 ? -(kFirstStages - 1) * kOperandBytes : kOperandBytes;
          b_move = read_slot % 2 == 1 ? -kOperandBytes : kOperandBytes;
          read_slot = read_slot == 5 ? 0 : read_slot + 1;
        }
        if constexpr (t % 4 == 3) load_first(std::integral_constant<int, 4 + t / 4>{});
        if constexpr (t >= 8 && t < 12) a_at[t % 4] += a_move;  // (behind the last reads of this step)
        if constexpr (t >= 12) b_at[t % 4] += b_move;
      });
      landed(younger);
      arrived(c1);
      next_second();
      phase(c1, c0, c0, [&](auto m) __attribute__((always_inline)) {  // (reads the next step's first slice; nothing's behind the last)
        if constexpr (decltype(m)::value == 1) begin_second();
        if constexpr (decltype(m)::value % 4 == 3) load_second(std::integral_constant<int, decltype(m)::value / 4>{});
      });
      arrived(c0);
    }

    float factor = 1.0f;
    if constexpr (kAAcross) factor = (p.factor0 ? *p.factor0 : 1.0f) * (p.factor1 ? *p.factor1 : 1.0f);
    const size_t out_row0 = kAAcross ? static_cast<size_t>(tile.group) * p.outer_m + tile.m0 : tile.row0;
    leave<kOutF32>(acc, p.out, out_row0, tile.valid_rows, p.outer_n, 128 * wave_row, tile.n0 + 128 * wave_column, factor);
    if (!tile_at(++turn, tile)) return;
    clear();
  }
}

// The tiles behind the last whole round, where these would leave most CUs without one: a quarter each, 2 x 2 wavefronts of 64 x 64. A
// step's sixteen matrix instructions are one phase, in which the next step's fragments are read and the loads go out five steps ahead,
// into the stage that was read the phase before. Bound by the loads: 32 KB for 512 cycles of the pipe are what the L1 gives at best. A quarter takes
// a fifth of a whole tile's time on a quarter of the CUs, 0.28 on all of them.
template <bool kAAcross, bool kBAcross, bool kOutF32>
__device__ __forceinline__ void quarter_tiles(const DenseParams& p, const WideTiles<kAAcross>& tiles, uint8_t* lds) {
  using A = WideOperand<kAAcross, kWideTile / 2>;
  using B = WideOperand<kBAcross, kWideTile / 2>;
  constexpr int kHalf = kWideTile / 2, kQuarterBytes = kOperandBytes / 2, kStages = 5, kLoads = 4;  // of each operand, a wavefront a step
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wave_row = wave / 2, wave_column = wave % 2;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)lds));
  const uint32_t a_pitch = (kAAcross ? p.outer_m : p.inner) * 2, b_pitch = (kBAcross ? p.outer_n : p.inner) * 2;
  const size_t a_stride = kAAcross ? static_cast<size_t>(kWideStep) * a_pitch : kWideStep * 2;
  const size_t b_stride = kBAcross ? static_cast<size_t>(kWideStep) * b_pitch : kWideStep * 2;
  uint32_t a_offset[kLoads], b_offset[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int a_row = A::row(kLoads * wave + i, lane), b_row = B::row(kLoads * wave + i, lane);
    a_offset[i] = a_row * a_pitch + 16 * A::chunk(a_row, lane);
    b_offset[i] = b_row * b_pitch + 16 * B::chunk(b_row, lane);
  }
  float factor = 1.0f;
  if constexpr (kAAcross) factor = (p.factor0 ? *p.factor0 : 1.0f) * (p.factor1 ? *p.factor1 : 1.0f);

  WidePlace place;
  for (int turn = 0, row_at = 0, n0 = 0; tiles.quarter_at(turn, p.group_m, place, row_at, n0); ++turn) {
    const int valid_rows = __builtin_amdgcn_readfirstlane(min(kHalf, (kAAcross ? p.outer_m : place.size) - row_at));
    if (valid_rows <= 0 || n0 >= p.outer_n) continue;  // (the same for the whole block)
    const uint8_t *a_next = reinterpret_cast<const uint8_t*>(p.a), *b_next = reinterpret_cast<const uint8_t*>(p.b);
    int a_bytes = 0, b_bytes = 0, left = 0, steps = p.inner / kWideStep;
    if constexpr (kAAcross) {
      const int row0 = min(max(place.start, 0), p.rows);
      left = min(max(place.start + place.size, row0), p.rows) - row0;
      steps = max((left + kWideStep - 1) / kWideStep, 1);
      a_next += static_cast<size_t>(row0) * a_pitch + row_at * 2;
      b_next += static_cast<size_t>(row0) * b_pitch + n0 * 2;
    } else {
      a_next += static_cast<size_t>(place.start + row_at) * a_pitch;
      a_bytes = valid_rows * a_pitch;
      b_next += static_cast<size_t>(place.group) * p.inner * p.outer_n * 2 + (kBAcross ? n0 * 2 : static_cast<size_t>(n0) * b_pitch);
      b_bytes = kBAcross ? kWideStep * b_pitch - n0 * 2 : min(kHalf, p.outer_n - n0) * b_pitch;
    }
    int fetched = 0, slot = 0;  // steps asked for, and where the next one goes
    __amdgpu_buffer_rsrc_t a_buffer, b_buffer;
    auto begin = [&]() __attribute__((always_inline)) {  // (steps behind the last read as zeros)
      if constexpr (kAAcross) {
        a_bytes = max(min(left, kWideStep) * static_cast<int>(a_pitch) - row_at * 2, 0);
        b_bytes = max(min(left, kWideStep) * static_cast<int>(b_pitch) - n0 * 2, 0);
        left -= kWideStep;
      }
      const bool any = fetched < steps;
      a_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a_next), 0, any ? a_bytes : 0, 0x00027000);
      b_buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(b_next), 0, any ? b_bytes : 0, 0x00027000);
      a_next += a_stride;
      b_next += b_stride;
      ++fetched;
    };
    auto load = [&](auto piece) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
      typedef __attribute__((address_space(3))) void* lds_t;
      constexpr int i = decltype(piece)::value % kLoads;
      uint8_t* to = lds + slot * 2 * kQuarterBytes + (wave * kLoads + i) * 1024;
      if constexpr (decltype(piece)::value < kLoads)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_buffer, (lds_t)to, 16, a_offset[i], 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(b_buffer, (lds_t)(to + kQuarterBytes), 16, b_offset[i], 0, 0, 0);
#endif
    };
    auto turned = [&]() __attribute__((always_inline)) { slot = slot == kStages - 1 ? 0 : slot + 1; };

    uint32_t a_at[4], b_at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      a_at[i] = A::address(lds_base, 2 * wave_row, i, lane);
      b_at[i] = B::address(lds_base + kQuarterBytes, 2 * wave_column, i, lane);
    }
    f32x16_t acc[2][2];
    bf16x8_t a_frag[2][4][2], b_frag[2][4][2];
    auto read = [&](auto set, auto piece) __attribute__((always_inline)) {
      constexpr int s = decltype(piece)::value / 4, i = decltype(piece)::value % 4;
      if constexpr (i < 2) b_frag[set.value][s][i] = wide_fragment<kBAcross, kHalf, s, i>(b_at);
      else a_frag[set.value][s][i - 2] = wide_fragment<kAAcross, kHalf, s, i - 2>(a_at);
    };
    int read_slot = 0;
    auto moves = [&]() __attribute__((always_inline)) {
      const uint32_t move = read_slot == kStages - 1 ? -(kStages - 1) * 2 * kQuarterBytes : 2 * kQuarterBytes;
      read_slot = read_slot == kStages - 1 ? 0 : read_slot + 1;
#pragma unroll
      for (int i = 0; i < 4; ++i) a_at[i] += move, b_at[i] += move;
    };
    auto landed = [&](auto younger, auto set) __attribute__((always_inline)) {
      constexpr int n = decltype(younger)::value;
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4));  // vmcnt(n) lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(a_frag[set.value][s][i]), "+v"(b_frag[set.value][s][i]));
      __builtin_amdgcn_sched_barrier(0);
    };
    auto phase = [&](auto from, auto into) __attribute__((always_inline)) {
      begin();
      static_for<16>([&](auto m) __attribute__((always_inline)) {
        constexpr int t = decltype(m)::value, s = t / 4, i = t % 4 / 2, j = t % 2;
        read(into, m);
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b_frag[from.value][s][j], a_frag[from.value][s][i], acc[i][j], 0, 0, 0);
        if constexpr (t % 2 == 1) load(std::integral_constant<int, t / 2>{});
        __builtin_amdgcn_sched_barrier(0);
      });
      turned();
      moves();
      // (in flight: the loads of the three steps behind the one that is read next)
      landed(std::integral_constant<int, 3 * 2 * kLoads>{}, into);
    };
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 1> c1{};
    // (the LDS is free of the last tile's reads and loads)
    __builtin_amdgcn_s_waitcnt(7 << 4);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
#pragma unroll
    for (int ahead = 0; ahead < kStages; ++ahead) {
      begin();
      static_for<2 * kLoads>(load);
      turned();
    }
    clear_sums(acc);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    constexpr int kFirst = (kStages - 1) * 2 * kLoads;
    __builtin_amdgcn_s_waitcnt((kFirst & 15) | ((kFirst >> 4) << 14) | (7 << 4));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    static_for<16>([&](auto piece) __attribute__((always_inline)) { read(c0, piece); });
    moves();
    landed(std::integral_constant<int, 3 * 2 * kLoads>{}, c0);
    for (int step = 0; step < steps; step += 2) {  // (an odd last step's second phase multiplies zeros)
      phase(c0, c1);
      phase(c1, c0);
    }
    const size_t out_row0 = kAAcross ? static_cast<size_t>(place.group) * p.outer_m + row_at : place.start + row_at;
    leave<kOutF32>(acc, p.out, out_row0, valid_rows, p.outer_n, 64 * wave_row, n0 + 64 * wave_column, factor);
  }
  __builtin_amdgcn_s_waitcnt(7 << 4);  // (no load into the LDS outlives the block)
}

template <bool kAAcross, bool kBAcross, bool kOutF32, bool kQuarters>
__global__ __launch_bounds__(kWideThreads, 1) void wide_kernel(DenseParams p) {
  extern __shared__ uint8_t lds[];
  WideTiles<kAAcross> tiles;
  tiles.find(p.offsets, p.sizes, p.groups, p.outer_m, p.outer_n, kQuarters ? p.quarter_turns : 0);
  if constexpr (!kAAcross) clear_unowned(static_cast<bf16_t*>(p.out), tiles.held, p.rows, p.outer_n);
  whole_tiles<kAAcross, kBAcross, kOutF32>(p, tiles, lds);
  if (kQuarters && tiles.whole < tiles.total) quarter_tiles<kAAcross, kBAcross, kOutF32>(p, tiles, lds);
}

template <bool kAAcross, bool kBAcross, bool kOutF32, bool kQuarters>
static int launch_wide_kernel(const char* who, const DenseParams& p, hipStream_t stream) {
  auto kernel = wide_kernel<kAAcross, kBAcross, kOutF32, kQuarters>;
  static std::once_flag configured;  // dynamic LDS above 64 KiB must be opted into once per kernel
  static hipError_t reserved = hipSuccess;
  std::call_once(configured, [&] {
    reserved = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kWideShared);
  });
  if (reserved != hipSuccess) return fail(DEW_MOE_ELAUNCH, "%s: cannot reserve %d bytes of LDS", who, kWideShared);
  hipLaunchKernelGGL(kernel, dim3(256), dim3(kWideThreads), kWideShared, stream, p);  // one block a CU
  return launched(who);
}

int launch_wide(const char* who, const DenseParams& params, bool across, bool kmajor, bool out_f32, hipStream_t stream) {
  DenseParams p = params;
  // A last round of at most a quarter of the CUs, or of half of them where a tile's walk is long enough to hide two starts: us, 4096 columns, the
  // contraction 4096 and 1024 deep, of 1.06 rounds 168 and 53 -> 125 and 42, 1.25 169 and 53 -> 135 and 48, 1.5 178 and 56 -> 165 and 57;
  // a kernel gradient of 2048 rows 1.12 93 -> 71, 1.5 100 -> 93, of 512 rows 1.25 33.6 -> 30.7, 1.5 35.6 and 36.8. Three quarters a block take as
  // long as the whole tile or longer (2.7 rounds 110 -> 120, 0.66 228 -> 282).
  p.quarter_turns = (across ? p.rows / p.groups : p.inner) >= 1024 ? 2 : 1;
  p.group_m = 4;  // (4 row tiles x 8 strips are what an XCD's 32 CUs hold at once; 6 or 8 were 0 to 3 % slower)
  if (!across) return kmajor ? launch_wide_kernel<false, false, false, true>(who, p, stream) : launch_wide_kernel<false, true, false, true>(who, p, stream);
  if (ends_in_quarters(p.groups, p.outer_m, p.outer_n, p.quarter_turns))
    return out_f32 ? launch_wide_kernel<true, true, true, true>(who, p, stream) : launch_wide_kernel<true, true, false, true>(who, p, stream);
  return out_f32 ? launch_wide_kernel<true, true, true, false>(who, p, stream) : launch_wide_kernel<true, true, false, false>(who, p, stream);
}

}  // namespace dew
