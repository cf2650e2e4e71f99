// The recipes' products of e4m3 operands in 256 x 256 tiles on blocks that stay: rows and banks as the quantizers leave them, on
// v_mfma_scale_f32_32x32x64_f8f6f4 under both operands' scales, with the tiled launch's bits (the sums run along the depth in the same order).
//
// One tile a block left a CU idle through each tile's start and end: of a blockwise kernel gradient's tile, eight steps of 128 tokens,
// these were more than half. Here 256 blocks of 4 wavefronts, one a CU, go from tile to tile, and the loads run on into the next tile while
// one leaves (wide.h).
//  * A step is 128 depths, two phases of 64. 2 x 2 wavefronts of 128 x 128: a phase is 16 matrix instructions of 64 cycles, 16 reads of
//    16 bytes from the LDS for the next phase's fragments, and 8 loads of the 32 KB that a phase fetches, one every other instruction.
//  * 160 KB of LDS: three stages of 256 rows x 128 bytes (whole cache lines; chunk index xor-swizzled as in the tiled launch), three of
//    the bank's atoms of 64 depths, which lie in the instruction's order and are read as they were fetched, and two of scales.
//  * A row's scale bytes are 16 at a time, those of 4 steps (a byte every 32 depths) or of 16 (one every 128): a dword a row a step
//    filled the L1 with as many lines as the rows themselves.
//  * The pipe is 67 to 69 % busy at 1.9 GHz over 32 and more steps a tile of MXFP8 (2.6 to 2.7 PFLOP/s), 55 to 59 % at 2.0 to 2.3 over 16 and 56 of the blockwise
//    recipe, 39 to 43 % over 8 at 2.1 to 2.4 (profiles/wide_tiles_mfma_utilisation.txt).
//  * The tiles behind the last whole round are cut in quarters (`quarter_fp8_tiles`) where these go round.
//  * Before a phase a wavefront waits for the loads of the phase before the last, and all of them meet: every load has one to two phases.
#include <mutex>

#include "wide_fp8.h"

namespace dew {

constexpr int kFp8Step = 128, kFp8RowStages = 3, kFp8BankStages = 3;
constexpr int kFp8RowBytes = kWideTile * kFp8Step;        // 32 KB: a step's rows
constexpr int kFp8BankBytes = kWideTile * kFp8Step / 2;   // 16 KB: half a step's atoms
constexpr int kFp8BankAt = kFp8RowStages * kFp8RowBytes;
constexpr int kFp8ScalesAt = kFp8BankAt + kFp8BankStages * kFp8BankBytes;
constexpr int kFp8ScaleBytes = 8192;                      // the rows' 4 KB, then the bank's
constexpr int kFp8Shared = kFp8ScalesAt + 2 * kFp8ScaleBytes;  // all of the LDS

template <int kOffset>
__device__ __forceinline__ u32x4_t read_quad(uint32_t at) {  // (written out, as in wide.hip; waited for in `arrived`)
  u32x4_t words;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(words) : "v"(at), "n"(kOffset));
  return words;
}

template <int kOffset, bool kByte>
__device__ __forceinline__ uint32_t read_scale(uint32_t at) {
  uint32_t word;
  if constexpr (kByte)
    asm volatile("ds_read_u8 %0, %1 offset:%2" : "=v"(word) : "v"(at), "n"(kOffset));
  else
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(word) : "v"(at), "n"(kOffset));
  return word;
}

// kMx: a scale byte every 32 depths of a row and of a column; else every 128 of a row, and an fp32 power of two every 128 x 128 of the
// bank. kGradient (kMx): every group contracts its own window of the depth of the same two matrices, both of them banks, whose
// atoms a load takes 4 KB of at a time where a row of the tokens would give it a line (32 x 1024 tokens x 7168 x 2048: 604 -> 583 us).
template <bool kMx, bool kGradient, bool kOutF32>
__device__ __forceinline__ void whole_fp8_tiles(const WideFp8Params& p, const WideTiles<kGradient>& tiles, uint8_t* lds) {
  constexpr int kScaleSteps = kMx ? 4 : 16;  // steps that a row's 16 bytes of scales are for
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wave_row = wave / 2, wave_column = wave % 2;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)lds));

  struct Tile {
    int group, row0, valid_rows, n0, first_step, steps, empty;
  };
  auto tile_at = [&](int turn, Tile& tile) {
    WidePlace place;
    if (!tiles.at(turn, 4, place)) return false;  // (4 row tiles x 8 strips are what an XCD's 32 CUs hold at once)
    tile.group = place.group;
    tile.n0 = place.strip * kWideTile;
    if constexpr (kGradient) {  // (an empty window: one step of zeros, the first: where it stands may be behind the last, whose scales are the last read)
      tile.row0 = place.within * kWideTile;
      tile.valid_rows = min(kWideTile, p.rows - tile.row0);
      const int first_step = min(max(place.start, 0), p.depth) / kFp8Step;
      // (said to be the same in every lane: as conditions of each lane they made a loop over the lanes of every load)
      const int steps = __builtin_amdgcn_readfirstlane(min(max(place.start + place.size, 0), p.depth) / kFp8Step - first_step);
      tile.empty = __builtin_amdgcn_readfirstlane(steps <= 0);
      tile.first_step = tile.empty ? 0 : first_step;
      tile.steps = max(steps, 1);
    } else {
      tile.row0 = place.start + place.within * kWideTile;
      tile.valid_rows = min(kWideTile, place.size - place.within * kWideTile);
      tile.first_step = tile.empty = 0;
      tile.steps = p.depth / kFp8Step;
    }
    return true;
  };

  // ---- what fetches: the rows three steps ahead of what is read, the bank three phases and the scales with it. A load's bytes are a
  // buffer: what lies past its end (the rows past a tile's last, the columns past the width) reads as zero ----
  Tile fetched;
  if (!tile_at(0, fetched)) return;  // (the same for the whole block)
  Tile tile = fetched;
  const int depth_steps = p.depth / kFp8Step, strips32 = p.width / 32;
  const size_t strip_bytes = static_cast<size_t>(p.depth) * 32;  // a 32-column tile's atoms, the whole depth
  int fetched_turn = 0, fetched_step = 0, row_slot = kFp8RowStages - 1, bank_slot = kFp8BankStages - 1;
  int scale_step = 0, scale_slot = 1;  // of the bank's stream: its step in the tile, the scales' buffer
  int scale_shift[2] = {0, 0};         // where a buffer's first step stands in it
  bool moved = false;
  const uint8_t *a_next = nullptr, *b_next = nullptr, *a_scales = nullptr, *b_scales = nullptr;
  int a_bytes = 0, b_bytes = 0, a_scale_bytes = 0, b_scale_bytes = 0, b_first = 0;
  uint32_t a_offset[8], b_offset[4];  // of the lane's 16 bytes of each load
  int a_stride = kGradient ? 4 * kAtomBytes : kFp8Step, b_stride = 2 * kAtomBytes;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int row = 8 * (8 * wave + i) + lane / 8;
    a_offset[i] = kGradient ? (2 * wave + i / 4) * static_cast<uint32_t>(strip_bytes) + (i % 4) * kAtomBytes + lane * 16
                            : row * static_cast<uint32_t>(p.depth) + 16 * ((lane % 8) ^ (((row >> 1) & 7) ^ ((row & 1) << 2)));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) b_offset[i] = (2 * wave + i / 2) * static_cast<uint32_t>(strip_bytes) + (i % 2) * kAtomBytes + lane * 16;
  const uint32_t strip_scale_offset = (2 * wave + lane / 32) * static_cast<uint32_t>(depth_steps) * 128 + (lane % 32) * 16;
  const uint32_t a_scale_offset = kGradient ? strip_scale_offset : (64 * wave + lane) * static_cast<uint32_t>(p.a_scale_pitch);
  const uint32_t b_scale_offset = kMx ? strip_scale_offset : (lane / 2 * (p.width / 128) + lane % 2) * 4;
  __amdgpu_buffer_rsrc_t a_buffer, b_buffer;
  auto buffer = [](const uint8_t* at, int bytes) __attribute__((always_inline)) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(at), 0, bytes, 0x00027000); };
  auto aim_first = [&]() __attribute__((always_inline)) {
    a_next = p.a + static_cast<size_t>(fetched.row0) * p.depth + fetched.first_step * (kGradient ? 4 * kAtomBytes : kFp8Step);
    a_bytes = __builtin_amdgcn_readfirstlane(fetched.empty ? 0 : fetched.valid_rows * p.depth);  // (a gradient's rows are whole 32s)
  };
  auto aim_second = [&]() __attribute__((always_inline)) {
    const size_t strip = static_cast<size_t>(kGradient ? 0 : fetched.group) * strips32 + fetched.n0 / 32;
    const int strips = __builtin_amdgcn_readfirstlane(fetched.empty ? 0 : min(kWideTile / 32, strips32 - fetched.n0 / 32));
    b_next = p.b + strip * strip_bytes + static_cast<size_t>(fetched.first_step) * 4 * kAtomBytes;
    b_bytes = strips * static_cast<int>(strip_bytes);
    a_scales = p.a_scale + static_cast<size_t>(fetched.row0) * p.a_scale_pitch;  // (a bank's, too: as many bytes a row)
    a_scale_bytes = __builtin_amdgcn_readfirstlane(fetched.empty ? 0 : fetched.valid_rows * p.a_scale_pitch);
    if constexpr (kMx) {
      b_scales = static_cast<const uint8_t*>(p.b_scale) + strip * depth_steps * 128;
      b_scale_bytes = strips * depth_steps * 128;
    } else {
      const int blocks = p.width / 128;
      b_scales = static_cast<const uint8_t*>(p.b_scale) + (static_cast<size_t>(fetched.group) * depth_steps * blocks + fetched.n0 / 128) * 4;
      b_scale_bytes = (depth_steps * blocks - fetched.n0 / 128) * 4;
    }
    b_first = fetched.first_step;
  };
  auto next_first = [&]() __attribute__((always_inline)) {  // ahead of a step's loads of rows
    if (fetched_step == fetched.steps) {
      if (!tile_at(++fetched_turn, fetched)) a_stride = 0;  // (none left: the last one's first step, again and again)
      fetched_step = 0;
      moved = true;
      aim_first();
    }
    ++fetched_step;
  };
  auto next_second = [&]() __attribute__((always_inline)) {  // ahead of a step's loads of the bank, before the rows' stream goes on
    if (moved) {
      moved = false;
      scale_step = 0;
      if (a_stride == 0) b_stride = 0;
      aim_second();
    }
  };
  auto begin_first = [&]() __attribute__((always_inline)) {
    a_buffer = buffer(a_next, a_bytes);
    a_next += a_stride;
    row_slot = row_slot == kFp8RowStages - 1 ? 0 : row_slot + 1;
  };
  auto begin_second = [&]() __attribute__((always_inline)) {
    b_buffer = buffer(b_next, b_bytes);
    b_next += b_stride;
    bank_slot = bank_slot == kFp8BankStages - 1 ? 0 : bank_slot + 1;
  };
  auto load_first = [&](auto piece) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void* lds_t;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(a_buffer, (lds_t)(lds + row_slot * kFp8RowBytes + (wave * 8 + piece.value) * 1024), 16, a_offset[piece.value], 0, 0, 0);
#endif
  };
  auto load_second = [&](auto piece) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void* lds_t;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(b_buffer, (lds_t)(lds + kFp8BankAt + bank_slot * kFp8BankBytes + (wave * 4 + piece.value) * 1024), 16,
                                             b_offset[piece.value], 0, 0, 0);
#endif
  };
  // the scales of a group of steps, with its first
  auto load_scales = [&]() __attribute__((always_inline)) {
    if (scale_step % kScaleSteps == 0) {
      scale_slot ^= 1;
      const int first = b_first + scale_step;
      // (a row's last 16 bytes end with it)
      const int from = kMx ? min(first, depth_steps - 4) : first;
      if (scale_slot)
        scale_shift[1] = first - from;
      else
        scale_shift[0] = first - from;
#if defined(__HIP_DEVICE_COMPILE__)
      typedef __attribute__((address_space(3))) void* lds_t;
      uint8_t* to = lds + kFp8ScalesAt + scale_slot * kFp8ScaleBytes;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(a_scales + from * (kGradient ? 128 : kMx ? 4 : 1), a_scale_bytes), (lds_t)(to + wave * 1024), 16, a_scale_offset, 0, 0, 0);
      if constexpr (kMx)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(b_scales + from * 128, b_scale_bytes), (lds_t)(to + 4096 + wave * 1024), 16, b_scale_offset, 0, 0, 0);
      else  // (32 lanes: two column blocks' of 16 steps, each wavefront its own copy)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(b_scales + static_cast<size_t>(from) * (p.width / 128) * 4, b_scale_bytes - from * (p.width / 128) * 4),
                                                 (lds_t)(to + 4096 + wave * 1024), 4, b_scale_offset, 0, 0, 0);
#endif
    }
    ++scale_step;
  };

  // ---- what multiplies ----
  uint32_t a_at[4];  // of the row tiles' 16 bytes 2 * half + piece
  uint32_t b_at = lds_base + kFp8BankAt + wave_column * 4 * 2 * kAtomBytes + lane * 16;
  {
    const int row = 128 * wave_row + lane % 32;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      a_at[i] = kGradient ? lds_base + wave_row * 16 * kAtomBytes + i * kAtomBytes + lane * 16
                          : lds_base + row * 128 + (((4 * (lane / 32) + i) ^ (((row >> 1) & 7) ^ ((row & 1) << 2))) * 16);
  }
  constexpr int kRowTileScales = kGradient ? 512 : 32 * 16;  // from a row tile's scales to the next one's
  const uint32_t a_scale_at = lds_base + kFp8ScalesAt + (kGradient ? wave_row * 4 * 512 + (lane % 32) * 4 : (128 * wave_row + lane % 32) * 16);
  const uint32_t b_scale_at = lds_base + kFp8ScalesAt + 4096 + (kMx ? wave_column * 4 * 512 + (lane % 32) * 4 : wave * 1024 + wave_column * 4);
  constexpr int kBankWords = kMx ? 4 : 1;
  f32x16_t acc[4][4];
  i32x8_t a_frag[2][4], b_frag[2][4];
  uint32_t a_read[4], b_read[kBankWords];  // the next step's scales as they lie
  int a_word[4], b_word[kBankWords];       // this step's: byte 2 * half is the lane's half's (kMx), or byte 0
  int unscalable = 0;                      // mantissa bits met in a weight block scale (the instruction takes powers of two only)
  auto clear = [&]() __attribute__((always_inline)) { clear_sums(acc); };
  auto read_piece = [&](auto half, auto set, auto piece) __attribute__((always_inline)) {
    constexpr int h = decltype(half)::value, i = decltype(piece)::value % 4;
    if constexpr (decltype(piece)::value < 4) {
      const u32x4_t low = read_quad<i * 2 * kAtomBytes>(b_at), high = read_quad<(2 * i + 1) * kAtomBytes>(b_at);
      b_frag[set.value][i] = i32x8_t{static_cast<int>(low[0]), static_cast<int>(low[1]), static_cast<int>(low[2]), static_cast<int>(low[3]),
                                     static_cast<int>(high[0]), static_cast<int>(high[1]), static_cast<int>(high[2]), static_cast<int>(high[3])};
    } else {
      const u32x4_t low = read_quad<i * 32 * kFp8Step>(a_at[2 * h]), high = read_quad<i * 32 * kFp8Step>(a_at[2 * h + 1]);
      a_frag[set.value][i] = i32x8_t{static_cast<int>(low[0]), static_cast<int>(low[1]), static_cast<int>(low[2]), static_cast<int>(low[3]),
                                     static_cast<int>(high[0]), static_cast<int>(high[1]), static_cast<int>(high[2]), static_cast<int>(high[3])};
    }
  };
  int taken_step = 0, taken_slot = 1;  // of the scales read: the step of its group, the buffer
  auto read_scales = [&](bool begins) __attribute__((always_inline)) {
    taken_step = begins || taken_step == kScaleSteps - 1 ? 0 : taken_step + 1;
    if (taken_step == 0) taken_slot ^= 1;
    const uint32_t from = taken_step + (taken_slot ? scale_shift[1] : scale_shift[0]), buffer_at = taken_slot * kFp8ScaleBytes;
    const uint32_t a_from = a_scale_at + (buffer_at + from * (kGradient ? 128 : kMx ? 4 : 1)), b_from = b_scale_at + (buffer_at + from * (kMx ? 128 : 8));
    static_for<4>([&](auto i) __attribute__((always_inline)) { a_read[i.value] = read_scale<i.value * kRowTileScales, !kMx>(a_from); });
    static_for<kBankWords>([&](auto j) __attribute__((always_inline)) { b_read[j.value] = read_scale<j.value * 512, false>(b_from); });
  };
  auto take_scales = [&]() __attribute__((always_inline)) {  // (behind `arrived`)
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(a_read[i]));
#pragma unroll
    for (int j = 0; j < kBankWords; ++j) asm volatile("" : "+v"(b_read[j]));
#pragma unroll
    for (int i = 0; i < 4; ++i) a_word[i] = static_cast<int>(kMx ? a_read[i] >> (8 * (lane / 32)) : a_read[i]);
    if constexpr (kMx) {
#pragma unroll
      for (int j = 0; j < kBankWords; ++j) b_word[j] = static_cast<int>(b_read[j] >> (8 * (lane / 32)));
    } else {
      b_word[0] = static_cast<int>(b_read[0] >> 23);
    }
  };
  // one phase: half `from` of a step multiplied, and in the shadows of its matrix instructions the next half's fragments read and `beside` done
  auto phase = [&](auto from, auto beside) __attribute__((always_inline)) {
    constexpr int h = decltype(from)::value;
    constexpr std::integral_constant<int, 1 - h> other{};
    static_for<16>([&](auto m) __attribute__((always_inline)) {
      constexpr int t = decltype(m)::value, i = t / 4, j = t % 4, byte = kMx ? 2 * h : 0;
      if constexpr (t < 8) read_piece(other, other, m);
      acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(b_frag[h][j], a_frag[h][i], acc[i][j], 0, 0, byte, b_word[kMx ? j : 0], byte, a_word[i]);
      beside(m);
      __builtin_amdgcn_sched_barrier(0);
    });
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int i = 0; i < 4; ++i)  // (the products stay here: nothing else keeps them from sinking behind the branches that follow)
#pragma unroll
      for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[i][j]));
#endif
  };
  auto pin = [&](auto set) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(a_frag[set.value][i]));
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(b_frag[set.value][j]));
    __builtin_amdgcn_sched_barrier(0);
  };
  // every wavefront's loads but its `younger` last memory operations are done, and so are its reads
  auto landed = [&](auto younger) __attribute__((always_inline)) {
    constexpr int n = decltype(younger)::value;
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4));  // vmcnt(n) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  constexpr std::integral_constant<int, 8> c8{};

  // Before the first phase: rows of steps 0, 1 and half of step 2, the bank's halves 0 to 2
  clear();
  aim_first();
  aim_second();
  next_first();
  begin_first();
  static_for<8>(load_first);
  load_scales();
  begin_second();
  static_for<4>(load_second);
  begin_second();
  static_for<4>(load_second);
  next_first();
  begin_first();
  static_for<8>(load_first);
  next_second();
  load_scales();
  begin_second();
  static_for<4>(load_second);
  next_first();
  begin_first();
  static_for<4>(load_first);
  landed(c0);
  static_for<8>([&](auto piece) __attribute__((always_inline)) { read_piece(c0, c0, piece); });
  read_scales(true);
  landed(c0);
  pin(c0);
  take_scales();
  b_at += kFp8BankBytes;
  int read_row_slot = 0, read_bank_slot = 1, turn = 0;
  auto bank_moves = [&]() __attribute__((always_inline)) {
    b_at += read_bank_slot == kFp8BankStages - 1 ? -(kFp8BankStages - 1) * kFp8BankBytes : kFp8BankBytes;
    read_bank_slot = read_bank_slot == kFp8BankStages - 1 ? 0 : read_bank_slot + 1;
  };
  for (;;) {
    for (int step = 0; step < tile.steps; ++step) {
      int last = __builtin_amdgcn_readfirstlane(step + 1 == tile.steps);
      asm volatile("" : "+s"(last));  // (known, it made a loop of the last step: its own copy of the code, and all sums moved on the way there)
      phase(c0, [&](auto m) __attribute__((always_inline)) {  // reads the step's second half
        constexpr int t = decltype(m)::value;
        if constexpr (t == 0) begin_second();
        if constexpr (t % 2 == 1 && t < 8) load_first(std::integral_constant<int, 4 + t / 2>{});
        if constexpr (t % 2 == 1 && t >= 8) load_second(std::integral_constant<int, t / 2 - 4>{});
        if constexpr (t == 8) bank_moves();
        if constexpr (t == 10) {
          const uint32_t move = read_row_slot == kFp8RowStages - 1 ? -(kFp8RowStages - 1) * kFp8RowBytes : kFp8RowBytes;
          read_row_slot = read_row_slot == kFp8RowStages - 1 ? 0 : read_row_slot + 1;
          a_at[0] += move, a_at[1] += move, a_at[2] += move, a_at[3] += move;
        }
        if constexpr (!kMx && t == 12) unscalable |= (b_read[0] & 0x807FFFFFu) | ((b_read[0] >> 23) == 0u) | ((b_read[0] >> 23) == 255u);
      });
      landed(c8);
      pin(c1);
      next_second();
      load_scales();
      next_first();
      phase(c1, [&](auto m) __attribute__((always_inline)) {  // reads the next step's first half and scales; nothing's behind the last
        constexpr int t = decltype(m)::value;
        if constexpr (t == 0) begin_second();
        if constexpr (t == 2) begin_first();
        if constexpr (t % 2 == 1 && t < 8) load_second(std::integral_constant<int, t / 2>{});
        if constexpr (t % 2 == 1 && t >= 8) load_first(std::integral_constant<int, t / 2 - 4>{});
        if constexpr (t == 8) read_scales(last != 0);
        if constexpr (t == 9) bank_moves();
      });
      landed(c8);
      pin(c0);
      take_scales();
    }

    float factor = 1.0f;
    if constexpr (!kMx) factor = unscalable != 0 ? __uint_as_float(0x7FC00000u) : 1.0f;  // (NaN rather than the product under another scale)
    const size_t out_row0 = kGradient ? static_cast<size_t>(tile.group) * p.rows + tile.row0 : tile.row0;
    leave<kOutF32>(acc, p.out, out_row0, tile.valid_rows, p.width, 128 * wave_row, tile.n0 + 128 * wave_column, factor);
    if (!tile_at(++turn, tile)) return;
    unscalable = 0;
    clear();
  }
}

// The tiles behind the last whole round, where these would leave most CUs without one: a quarter each, 2 x 2 wavefronts of 64 x 64. A
// step's eight matrix instructions are one phase, in which the next step's fragments and scales are read and the loads go out four
// steps ahead, into the stage that was read the phase before; the first two wavefronts fetch the rows' scales, the others the bank's.
// Bound by the loads, 64 bytes a clock of the pipe's rate.
template <bool kMx, bool kGradient, bool kOutF32>
__device__ __forceinline__ void quarter_fp8_tiles(const WideFp8Params& p, const WideTiles<kGradient>& tiles, uint8_t* lds) {
  constexpr int kScaleSteps = kMx ? 4 : 16;  // steps that a row's 16 bytes of scales are for
  constexpr int kHalf = kWideTile / 2, kOperand = kHalf * kFp8Step, kStages = 4, kStage = 2 * kOperand, kLoads = 4;  // of each operand, a wavefront a step
  constexpr int kScalesAt = kStages * kStage, kBankScales = kHalf * 16, kScales = 2 * kBankScales;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wave_row = wave / 2, wave_column = wave % 2;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)lds));
  const int depth_steps = p.depth / kFp8Step, strips32 = p.width / 32, blocks = p.width / 128;
  const size_t strip_bytes = static_cast<size_t>(p.depth) * 32;
  uint32_t a_offset[kLoads], b_offset[kLoads];
#pragma unroll
  for (int i = 0; i < kLoads; ++i) {
    const int row = 8 * (kLoads * wave + i) + lane / 8;
    b_offset[i] = wave * static_cast<uint32_t>(strip_bytes) + i * kAtomBytes + lane * 16;
    a_offset[i] = kGradient ? b_offset[i] : row * static_cast<uint32_t>(p.depth) + 16 * ((lane % 8) ^ (((row >> 1) & 7) ^ ((row & 1) << 2)));
  }
  const uint32_t strip_scale_offset = (wave % 2 * 2 + lane / 32) * static_cast<uint32_t>(depth_steps) * 128 + (lane % 32) * 16;
  const uint32_t scale_offset = wave < 2 ? (kGradient ? strip_scale_offset : (64 * wave + lane) * static_cast<uint32_t>(p.a_scale_pitch))
                                         : (kMx ? strip_scale_offset : lane * static_cast<uint32_t>(blocks) * 4);
  auto buffer = [](const uint8_t* at, int bytes) __attribute__((always_inline)) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(at), 0, bytes, 0x00027000); };

  WidePlace place;
  for (int turn = 0, row_at = 0, n0 = 0; tiles.quarter_at(turn, 4, place, row_at, n0); ++turn) {
    const int valid_rows = __builtin_amdgcn_readfirstlane(min(kHalf, (kGradient ? p.rows : place.size) - row_at));
    if (valid_rows <= 0 || n0 >= p.width) continue;  // (the same for the whole block)
    int first_step = 0, steps = depth_steps, row0 = row_at;
    bool empty = false;
    if constexpr (kGradient) {  // (an empty window: one step of zeros, as in the whole tiles)
      first_step = min(max(place.start, 0), p.depth) / kFp8Step;
      steps = __builtin_amdgcn_readfirstlane(min(max(place.start + place.size, 0), p.depth) / kFp8Step - first_step);
      empty = steps <= 0;
      if (empty) first_step = 0;
      steps = max(steps, 1);
    } else {
      row0 += place.start;
    }
    const size_t strip = static_cast<size_t>(kGradient ? 0 : place.group) * strips32 + n0 / 32;
    const int strips = empty ? 0 : min(kHalf / 32, strips32 - n0 / 32);
    const uint8_t* a_next = p.a + static_cast<size_t>(row0) * p.depth + first_step * (kGradient ? 4 * kAtomBytes : kFp8Step);
    const uint8_t* b_next = p.b + strip * strip_bytes + static_cast<size_t>(first_step) * 4 * kAtomBytes;
    const int a_bytes = empty ? 0 : valid_rows * p.depth, b_bytes = strips * static_cast<int>(strip_bytes);
    // this wavefront's scales: the rows', or the bank's
    const uint8_t* scales = wave < 2 ? p.a_scale + static_cast<size_t>(row0) * p.a_scale_pitch
                            : kMx    ? static_cast<const uint8_t*>(p.b_scale) + strip * depth_steps * 128
                                     : static_cast<const uint8_t*>(p.b_scale) + (static_cast<size_t>(place.group) * depth_steps * blocks + n0 / 128) * 4;
    const int scale_bytes = empty ? 0 : wave < 2 ? valid_rows * p.a_scale_pitch : kMx ? strips * depth_steps * 128 : (depth_steps * blocks - n0 / 128) * 4;
    const int scale_step = wave < 2 ? (kGradient ? 128 : kMx ? 4 : 1) : (kMx ? 128 : blocks * 4);  // bytes from a step's to the next one's
    int scale_shift[2] = {0, 0};  // where a buffer's first step stands in it
    int fetched = 0, slot = 0;
    __amdgpu_buffer_rsrc_t a_buffer, b_buffer;
    auto begin = [&]() __attribute__((always_inline)) {  // (steps behind the last read as zeros)
      const bool any = fetched < steps;
      a_buffer = buffer(a_next, any ? a_bytes : 0);
      b_buffer = buffer(b_next, any ? b_bytes : 0);
      a_next += kGradient ? 4 * kAtomBytes : kFp8Step;
      b_next += 4 * kAtomBytes;
      if (fetched % kScaleSteps == 0 && any) {
        const int scale_slot = fetched / kScaleSteps % 2, first = first_step + fetched;
        const int from = kMx ? min(first, depth_steps - 4) : first;  // (a row's last 16 bytes end with it)
        if (scale_slot)
          scale_shift[1] = first - from;
        else
          scale_shift[0] = first - from;
#if defined(__HIP_DEVICE_COMPILE__)
        typedef __attribute__((address_space(3))) void* lds_t;
        uint8_t* to = lds + kScalesAt + scale_slot * kScales + wave / 2 * kBankScales;
        const __amdgpu_buffer_rsrc_t from_scales = buffer(scales + static_cast<size_t>(from) * scale_step, !kMx && wave >= 2 ? scale_bytes - from * scale_step : scale_bytes);
        if (kMx || wave < 2)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(from_scales, (lds_t)(to + wave % 2 * 1024), 16, scale_offset, 0, 0, 0);
        else if (wave == 2)  // (16 steps of the one column block; what the other lanes fetch is not read)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(from_scales, (lds_t)to, 4, scale_offset, 0, 0, 0);
#endif
      }
      ++fetched;
    };
    auto load = [&](auto piece) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
      typedef __attribute__((address_space(3))) void* lds_t;
      constexpr int i = decltype(piece)::value % kLoads;
      uint8_t* to = lds + slot * kStage + (wave * kLoads + i) * 1024;
      if constexpr (decltype(piece)::value < kLoads)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(a_buffer, (lds_t)to, 16, a_offset[i], 0, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(b_buffer, (lds_t)(to + kOperand), 16, b_offset[i], 0, 0, 0);
#endif
    };
    auto turned = [&]() __attribute__((always_inline)) { slot = slot == kStages - 1 ? 0 : slot + 1; };

    uint32_t a_at[4];  // of the row tiles' 16 bytes 2 * half + piece
    uint32_t b_at = lds_base + kOperand + wave_column * 2 * 4 * kAtomBytes + lane * 16;
    {
      const int row = 64 * wave_row + lane % 32;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        a_at[i] = kGradient ? lds_base + wave_row * 2 * 4 * kAtomBytes + i * kAtomBytes + lane * 16
                            : lds_base + row * 128 + (((4 * (lane / 32) + i) ^ (((row >> 1) & 7) ^ ((row & 1) << 2))) * 16);
    }
    constexpr int kRowTileScales = kGradient ? 512 : 32 * 16, kBankWords = kMx ? 2 : 1;
    const uint32_t a_scale_at = lds_base + kScalesAt + (kGradient ? wave_row * 2 * 512 + (lane % 32) * 4 : (64 * wave_row + lane % 32) * 16);
    const uint32_t b_scale_at = lds_base + kScalesAt + kBankScales + (kMx ? wave_column * 2 * 512 + (lane % 32) * 4 : 0);
    f32x16_t acc[2][2];
    i32x8_t a_frag[2][2][2], b_frag[2][2][2];
    uint32_t a_read[2], b_read[kBankWords];
    int a_word[2], b_word[kBankWords], unscalable = 0;
    auto read = [&](auto set, auto piece) __attribute__((always_inline)) {
      constexpr int h = decltype(piece)::value / 4, i = decltype(piece)::value % 2;
      auto whole = [](const u32x4_t& low, const u32x4_t& high) __attribute__((always_inline)) {
        return i32x8_t{static_cast<int>(low[0]), static_cast<int>(low[1]), static_cast<int>(low[2]), static_cast<int>(low[3]),
                       static_cast<int>(high[0]), static_cast<int>(high[1]), static_cast<int>(high[2]), static_cast<int>(high[3])};
      };
      if constexpr (decltype(piece)::value % 4 < 2)
        b_frag[set.value][h][i] = whole(read_quad<(4 * i + 2 * h) * kAtomBytes>(b_at), read_quad<(4 * i + 2 * h + 1) * kAtomBytes>(b_at));
      else
        a_frag[set.value][h][i] = whole(read_quad<i * 32 * kFp8Step>(a_at[2 * h]), read_quad<i * 32 * kFp8Step>(a_at[2 * h + 1]));
    };
    int taken = 0, read_slot = 0;
    auto read_scales = [&]() __attribute__((always_inline)) {  // of step `taken`, and on to the next
      const int scale_slot = taken / kScaleSteps % 2;
      const uint32_t from = taken % kScaleSteps + (scale_slot ? scale_shift[1] : scale_shift[0]), buffer_at = scale_slot * kScales;
      const uint32_t a_from = a_scale_at + (buffer_at + from * (kGradient ? 128 : kMx ? 4 : 1)), b_from = b_scale_at + (buffer_at + from * (kMx ? 128 : 4));
      static_for<2>([&](auto i) __attribute__((always_inline)) { a_read[i.value] = read_scale<i.value * kRowTileScales, !kMx>(a_from); });
      static_for<kBankWords>([&](auto j) __attribute__((always_inline)) { b_read[j.value] = read_scale<j.value * 512, false>(b_from); });
      ++taken;
    };
    auto moves = [&]() __attribute__((always_inline)) {
      const uint32_t move = read_slot == kStages - 1 ? -(kStages - 1) * kStage : kStage;
      read_slot = read_slot == kStages - 1 ? 0 : read_slot + 1;
      a_at[0] += move, a_at[1] += move, a_at[2] += move, a_at[3] += move, b_at += move;
    };
    // every wavefront's loads but its `younger` last are done, and so are its reads, which are the next phase's operands
    auto landed = [&](auto younger, auto set) __attribute__((always_inline)) {
      constexpr int n = decltype(younger)::value;
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4));  // vmcnt(n) lgkmcnt(0)
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(a_frag[set.value][h][i]), "+v"(b_frag[set.value][h][i]));
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        asm volatile("" : "+v"(a_read[i]));
        a_word[i] = static_cast<int>(kMx ? a_read[i] >> (8 * (lane / 32)) : a_read[i]);
      }
#pragma unroll
      for (int j = 0; j < kBankWords; ++j) {
        asm volatile("" : "+v"(b_read[j]));
        b_word[j] = static_cast<int>(kMx ? b_read[j] >> (8 * (lane / 32)) : b_read[j] >> 23);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    auto phase = [&](auto from, auto into) __attribute__((always_inline)) {
      if constexpr (!kMx) unscalable |= (b_read[0] & 0x807FFFFFu) | ((b_read[0] >> 23) == 0u) | ((b_read[0] >> 23) == 255u);
      begin();
      read_scales();
      static_for<8>([&](auto m) __attribute__((always_inline)) {
        constexpr int t = decltype(m)::value, h = t / 4, i = t % 4 / 2, j = t % 2, byte = kMx ? 2 * h : 0;
        read(into, m);
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(b_frag[from.value][h][j], a_frag[from.value][h][i], acc[i][j], 0, 0, byte,
                                                                     b_word[kMx ? j : 0], byte, a_word[i]);
        load(m);
        __builtin_amdgcn_sched_barrier(0);
      });
      turned();
      moves();
      // (in flight: the loads of the two steps behind the one that is read next)
      landed(std::integral_constant<int, 2 * 2 * kLoads>{}, into);
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
    read_scales();
    static_for<8>([&](auto piece) __attribute__((always_inline)) { read(c0, piece); });
    moves();
    landed(std::integral_constant<int, 2 * 2 * kLoads>{}, c0);
    int step = 0;
    for (; step + 2 <= steps; step += 2) {
      phase(c0, c1);
      phase(c1, c0);
    }
    if (step < steps) phase(c0, c1);
    float factor = 1.0f;
    if constexpr (!kMx) factor = unscalable != 0 ? __uint_as_float(0x7FC00000u) : 1.0f;  // (NaN rather than the product under another scale)
    const size_t out_row0 = kGradient ? static_cast<size_t>(place.group) * p.rows + row_at : row0;
    leave<kOutF32>(acc, p.out, out_row0, valid_rows, p.width, 64 * wave_row, n0 + 64 * wave_column, factor);
  }
  __builtin_amdgcn_s_waitcnt(7 << 4);  // (no load into the LDS outlives the block)
}

template <bool kMx, bool kGradient, bool kOutF32, bool kQuarters>
__global__ __launch_bounds__(kWideThreads, 1) void wide_fp8_kernel(WideFp8Params p) {
  extern __shared__ uint8_t lds[];
  WideTiles<kGradient> tiles;
  tiles.find(p.offsets, nullptr, p.groups, p.rows, p.width, kQuarters ? p.quarter_turns : 0);
  if constexpr (!kGradient) clear_unowned(static_cast<bf16_t*>(p.out), tiles.held, p.rows, p.width);
  whole_fp8_tiles<kMx, kGradient, kOutF32>(p, tiles, lds);
  if (kQuarters && tiles.whole < tiles.total) quarter_fp8_tiles<kMx, kGradient, kOutF32>(p, tiles, lds);
}

template <bool kMx, bool kGradient, bool kOutF32, bool kQuarters>
static int launch_kernel(const char* who, const WideFp8Params& p, hipStream_t stream) {
  auto kernel = wide_fp8_kernel<kMx, kGradient, kOutF32, kQuarters>;
  static std::once_flag configured;  // dynamic LDS above 64 KiB must be opted into once per kernel
  static hipError_t reserved = hipSuccess;
  std::call_once(configured, [&] {
    reserved = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kFp8Shared);
  });
  if (reserved != hipSuccess) return fail(DEW_MOE_ELAUNCH, "%s: cannot reserve %d bytes of LDS", who, kFp8Shared);
  hipLaunchKernelGGL(kernel, dim3(256), dim3(kWideThreads), kFp8Shared, stream, p);  // one block a CU
  return launched(who);
}

int launch_wide_fp8(const char* who, const WideFp8Params& params, bool mx, bool gradient, bool out_f32, hipStream_t stream) {
  WideFp8Params p = params;
  // A last round of at most a quarter of the CUs, or of half of them where a tile's walk is long enough to hide two starts. Measured (us): [21 888,
  // 4992] x 2304 of 4, 3.02 rounds, 227 -> 202, [9088, 2816] x 1792 of 20, 1.12, 66 -> 51, [2816, 4608] x 7424 of 4, 1.36, 103 -> 95, [12 032, 896] x 1792 of
  // 9, 1.37, 31.3 and 31.4; kernel gradients of 10 496 tokens, 6 x 4096 x 640, 1.12, 57 -> 43, 8320 of 2 x 2560 x 3456, 1.09, 99 -> 68.
  p.quarter_turns = (gradient ? p.depth / p.groups : p.depth) >= 2048 ? 2 : 1;
  if (!gradient) return mx ? launch_kernel<true, false, false, true>(who, p, stream) : launch_kernel<false, false, false, true>(who, p, stream);
  if (ends_in_quarters(p.groups, p.rows, p.width, p.quarter_turns))
    return out_f32 ? launch_kernel<true, true, true, true>(who, p, stream) : launch_kernel<true, true, false, true>(who, p, stream);
  return out_f32 ? launch_kernel<true, true, true, false>(who, p, stream) : launch_kernel<true, true, false, false>(who, p, stream);
}

}  // namespace dew
