// The grouped GEMM of quantized banks in tiles of up to 256 rows on eight wavefronts, one block a CU.
//
// What bounds a prompt's products on FP8 and general NVFP4 banks is the vector unit: a weight costs two vector instructions on
// its way to a matrix operand, and the clock falls with them. A wavefront here owns 32 columns of one matrix and ALL rows of the
// tile, so a fragment brought to bf16 is multiplied by up to eight 32-row tiles before it is dropped, twice as many as on the
// 128-row tiles of gemm.hip. Of a paired launch (gate and up, SwiGLU) wavefronts 0 to 3 hold the gate's 128 columns and 4 to 7
// the up projection's, and they exchange rounded sums through the LDS in the epilogue.
//
// Unquantized banks, whose launches are bound by their weights' bytes, gain otherwise: a group of 130 to 220 rows reads them once, not
// twice, and one of 70 multiplies 96 rows, not 128.
//
// Tiles follow their groups: a group of n rows is ceil(n / 256) tiles (of at most 224 rows on unquantized banks) of equally many 32-row
// tiles (each count its own copy of the main loop), so that a group's last rows need neither a launch of their own nor a tile that is
// mostly empty.
//
// Cycles of a tile of 256 rows, FP8, 2048 deep (one bank): some 7000 until its first step, 74 000 in 32 steps (the matrix pipe 88 % busy),
// 7400 until its last store; paired 96 000, of which 13 000 are both matrices' sums' arithmetic. Tried and not kept, all the same to a
// percent: several strips a block with the next one's loads under the epilogue (the clock gives back what the wait took: the chip's power
// is the bound); blocks of four wavefronts, two a CU (quantized banks 4 % slower, their rows are fetched twice as often).
#include <algorithm>
#include <mutex>

#include "common.h"
#include "gemm.h"

namespace dew {

constexpr int kTallThreads = 512, kTallRows = 256;
constexpr int kScaleRow = kMaxDepthBlocks + 1;  // a column block's scales; the last step reads one past the deepest bank's (and drops it)

// Dynamic LDS: the ring of A rows, or the staged output tile, behind it the sums that the halves of a paired launch exchange, and
// the table of the rows' destinations.
template <bool PAIRED>
struct TallStaging {
  static constexpr int kColumns = PAIRED ? 128 : 256;       // output columns of the tile
  static constexpr int kRowDwords = kColumns / 2 + 4;       // a staged row in bf16 and 16 bytes of padding
  static constexpr int kExchange = kTallRows * kRowDwords;  // dword offset of the exchanged sums: [4 wavefronts][8 row tiles][2][64 lanes][4]
  static constexpr int kRowTable = kExchange + (PAIRED ? 4 * 8 * 2 * 64 * 4 : 0);
  static constexpr size_t kBytes = static_cast<size_t>(kRowTable + kTallRows) * 4;
};

struct TallTile {
  int expert, row0, valid_rows, n0;
};

// Half of a slice's fragment (words 2 part, 2 part + 1: four of the lane's eight weights), with the arithmetic of fragment_fp8 and
// fragment_fp4.
template <int FORMAT, int PART>
__device__ __forceinline__ void dequantize_half(u32x4_t& fragment, uint32_t word, float scale) {
  if constexpr (FORMAT == DEW_MOE_W_NVFP4) {
    const f32x2_t a = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 2 * PART), b = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(word, 1.0f, 2 * PART + 1);
    fragment[2 * PART] = pack_bf16(a.x * scale, a.y * scale);
    fragment[2 * PART + 1] = pack_bf16(b.x * scale, b.y * scale);
  } else {
    const f32x2_t a = __builtin_amdgcn_cvt_pk_f32_fp8(word, false), b = __builtin_amdgcn_cvt_pk_f32_fp8(word, true);
    fragment[2 * PART] = pack_bf16(a.x * scale, a.y * scale);
    fragment[2 * PART + 1] = pack_bf16(b.x * scale, b.y * scale);
  }
}

// Instruction order of a slice: its matrix instructions, behind the first half of them the next slice's operand reads two at a
// time (a wait for one of them is a wait for all: the rows' DMA loads stand between them in the compiler's eyes), and the
// vector work and the loads dealt evenly.
template <int M, int MFMAS, int DSR, int VALU, int VMEM>
__device__ __forceinline__ void schedule_slice() {
  if constexpr (M < MFMAS) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
    if constexpr (DSR > 2 * M) __builtin_amdgcn_sched_group_barrier(0x100, DSR - 2 * M >= 2 ? 2 : 1, 0);
    __builtin_amdgcn_sched_group_barrier(0x002, (VALU + MFMAS - 1) / MFMAS, 0);
    if constexpr (VMEM > 0) __builtin_amdgcn_sched_group_barrier(0x020, (VMEM + MFMAS - 1) / MFMAS, 0);
    schedule_slice<M + 1, MFMAS, DSR, VALU, VMEM>();
  }
}

// How far ahead of their use a tile of TI 32-row tiles asks for its rows (kAhead steps, a ring of one stage more) and its weights (kSets register
// sets, kAhead + 1 steps). Quantized banks: two steps of 300 to 2400 cycles, with the vector unit the bound. Unquantized ones are bound by the weights'
// stream, four times the bytes a step, and their steps are the shorter: as many as the registers hold.
template <int FORMAT, int TI>
struct TallDepth {
  static constexpr int kAhead = FORMAT != DEW_MOE_W_BF16 || TI > 6 ? 2 : TI > 4 ? 3 : 4, kStages = kAhead + 1, kSets = kAhead + 2;
  static constexpr int kRowLoads = (TI + 1) / 2;                     // A rows' loads a lane issues a step (of an odd TI the last wavefronts' fetch rows again)
  static constexpr int kStageChunks = 64 * kRowLoads * kChunksPerRow;
};
// 32-row tiles of a tile at most: of unquantized banks the registers that a step's weights take leave seven.
template <int FORMAT>
constexpr int kMostTiles = FORMAT == DEW_MOE_W_BF16 ? 7 : 8;

template <int FORMAT, bool PAIRED, int TI>
__device__ __forceinline__ void tall_tile(const GemmParams& p, const TallTile tile, u32x4_t* lds, float* depth_scales) {
  constexpr bool kFp4 = FORMAT == DEW_MOE_W_NVFP4, kBf16 = FORMAT == DEW_MOE_W_BF16;
  constexpr bool kBlockBank = FORMAT == DEW_MOE_W_FP8_BLOCK;
  constexpr int kAtomK = kFp4 ? 64 : kBf16 ? 16 : 32, kAtoms = BK / kAtomK;
  using Depth = TallDepth<FORMAT, TI>;
  constexpr int kAhead = Depth::kAhead, kStages = Depth::kStages, kSets = Depth::kSets, kRowLoads = Depth::kRowLoads, kStageChunks = Depth::kStageChunks;
  constexpr int kLoadsB = kAtoms + (kFp4 ? 1 : 0);

  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int side = wave / 4;  // paired: the matrix; else the 128-column half of the tile
  const int row0 = tile.row0, valid_rows = tile.valid_rows, expert = tile.expert, n0 = tile.n0;
  const int steps = p.depth / BK;

  // ---- weights: the wavefront's strip of 32 columns, its whole depth one stream ----
  // (past a ragged width the wavefront reads the bank's last 32 columns again; what it sums is not stored)
  const int column0 = PAIRED ? n0 + 32 * (wave % 4) : n0 + 32 * wave;
  const int column = min(column0, p.width - 32);
  const BankView& bank = PAIRED && side == 1 ? p.w1 : p.w0;
  const int k_atoms = p.depth / kAtomK;
  const size_t first_atom = (static_cast<size_t>(expert) * (p.width / 32) + column / 32) * k_atoms;
  const uint8_t* b_src = bank.codes + first_atom * kAtomBytes;  // (the same for the wavefront)
  const uint8_t* b_scale_src = kFp4 ? static_cast<const uint8_t*>(bank.scales) + first_atom * 128 : nullptr;
  float channel_scale = 1.0f;
  if constexpr (FORMAT == DEW_MOE_W_FP8_CHANNEL) channel_scale = static_cast<const float*>(bank.scales)[static_cast<size_t>(expert) * p.width + column + lane % 32];
  float tensor_scale = 1.0f;
  if constexpr (kFp4) tensor_scale = bank.tensor_scale[expert];

  u32x4_t b_regs[kSets][kAtoms];
  uint32_t s_regs[kSets];  // FP4: two e4m3 scale bytes in the low half
  auto load_b = [&](auto set, int step) __attribute__((always_inline)) {
    const uint8_t* from = b_src + static_cast<size_t>(step) * (kAtoms * kAtomBytes);
#pragma unroll
    for (int a = 0; a < kAtoms; ++a) {
      const u32x4_t* at = reinterpret_cast<const u32x4_t*>(from + a * kAtomBytes + lane * 16);
      b_regs[set.value][a] = kBf16 ? __builtin_nontemporal_load(at) : *at;  // (unquantized: taken where most groups are one tile, which reads them once)
    }
    if constexpr (kFp4) s_regs[set.value] = *reinterpret_cast<const uint16_t*>(b_scale_src + static_cast<size_t>(step) * 128 + lane * 2);
  };

  // ---- A rows: gathered, then the first weights behind the indices, as in gemm.hip ----
  int a_source[kRowLoads];
#pragma unroll
  for (int i = 0; i < kRowLoads; ++i) {
    const int sorted = row0 + min((wave * kRowLoads + i) * 8 + lane / 8, valid_rows - 1);
    a_source[i] = p.gather ? p.gather[sorted] : sorted;
  }
  // FP8 blocks: the scales of the tile's two column blocks down the depth, one a thread (512 at most), kept in the LDS once the
  // loads behind them are out
  float early_scale = 0.0f;
  const int depth_blocks = p.depth / 128;
  if constexpr (kBlockBank) {
    const int width_blocks = p.width / 128;
    if (tid < 2 * depth_blocks) {
      const int which = tid / depth_blocks, block = tid % depth_blocks;
      const float* scales = static_cast<const float*>(PAIRED && which == 1 ? p.w1.scales : p.w0.scales);
      const int column_block = PAIRED ? n0 / 128 : min(n0 / 128 + which, width_blocks - 1);
      early_scale = scales[(static_cast<size_t>(expert) * depth_blocks + block) * width_blocks + column_block];
    }
  }
  constexpr std::integral_constant<int, 0> c0{};
  constexpr std::integral_constant<int, 1> c1{};
  static_for<kSets - 1>([&](auto set) __attribute__((always_inline)) { load_b(set, min(decltype(set)::value, steps - 1)); });
  const bf16_t* a_src[kRowLoads];
#pragma unroll
  for (int i = 0; i < kRowLoads; ++i) {
    const int row = (wave * kRowLoads + i) * 8 + lane / 8;
    const int chunk = (lane % 8) ^ (((row >> 1) & 7) ^ ((row & 1) << 2));
    a_src[i] = p.x + static_cast<size_t>(a_source[i]) * p.depth + chunk * 8 - i * 512;  // less the load's immediate offset
    asm volatile("" : "+v"(a_src[i]));
  }
  auto load_a = [&](u32x4_t* stage, int step, auto begin, auto end) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    static_range<decltype(begin)::value>(std::make_integer_sequence<int, decltype(end)::value - decltype(begin)::value>{}, [&](auto index) {
      constexpr int i = decltype(index)::value;
      __builtin_amdgcn_global_load_lds(a_src[i] + static_cast<size_t>(step) * BK,
                                       (__attribute__((address_space(3))) void*)(stage + wave * kRowLoads * 64), 16, i * 1024, 0);
    });
#endif
  };
  bf16x8_t a_frag[2][TI];
  u32x4_t b_frag[2];
  float fp4_scale = 1.0f;
  // the lane's chunk of its first row tile in each slice, as a byte offset into a stage; a row tile further is 4 KiB further
  uint32_t slice_at[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk)
    slice_at[kk] = 16 * swizzled(lane % 32, kFp4 ? 4 * (lane / 32) + kk : kBf16 ? 2 * kk + lane / 32 : 4 * (kk / 2) + 2 * (lane / 32) + kk % 2);
  auto fetch = [&](uint32_t stage, auto kk) __attribute__((always_inline)) {  // (`stage` in bytes)
    const uint8_t* from = reinterpret_cast<const uint8_t*>(lds) + (slice_at[kk.value] + stage);
#pragma unroll
    for (int i = 0; i < TI; ++i) a_frag[kk.value % 2][i] = *reinterpret_cast<const bf16x8_t*>(from + 4096 * i);
  };
  float next_scale = 1.0f;
  float block_scale = 1.0f;  // FP8 blocks: the scale of the step whose slices are brought to bf16
  auto dequantize = [&](auto set, auto kk, auto part) __attribute__((always_inline)) {
    u32x4_t& fragment = b_frag[kk.value % 2];
    if constexpr (kBf16) {  // (the atoms are the fragments)
    } else if constexpr (kFp4) {
      if constexpr (kk.value % 2 == 0 && part.value == 0) {  // slices 0, 1 lie in the lane's first 16-deep block, 2, 3 in its second
        const float scale = kk.value == 0 ? __builtin_amdgcn_cvt_f32_fp8(s_regs[set.value], 0) : __builtin_amdgcn_cvt_f32_fp8(s_regs[set.value], 1);
        fp4_scale = scale * 0.00390625f;
      }
      dequantize_half<FORMAT, part.value>(fragment, b_regs[set.value][0][kk.value], fp4_scale);
    } else {
      const float scale = kBlockBank ? block_scale : channel_scale;
      dequantize_half<FORMAT, part.value>(fragment, b_regs[set.value][kk.value / 2 % kAtoms][2 * (kk.value % 2) + part.value], scale);
    }
  };

  f32x16_t acc[TI];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[i][q] = 0.0f;
  auto multiply = [&](auto set, auto kk) __attribute__((always_inline)) {
    const bf16x8_t b = __builtin_bit_cast(bf16x8_t, kBf16 ? b_regs[set.value][kk.value % kAtoms] : b_frag[kk.value % 2]);
#pragma unroll
    for (int i = 0; i < TI; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_frag[kk.value % 2][i], b, acc[i], 0, 0, 0);
  };

  // ---- pipeline: the ring and the waits of gemm.hip. A step's loads go out as A rows (of step s + kAhead) and then weights (of step
  // s + kAhead + 1), all before the barrier in front of the step's last slice, which waits for the A rows of step s + 1, asked for in step
  // s + 1 - kAhead: younger are that step's weights and all loads since. So the weights of step s + 1, asked for one step before those
  // rows, have landed there too, and the last slice brings their first one to bf16. ----
  constexpr int kYounger = (kAhead - 1) * (kRowLoads + kLoadsB) + kLoadsB;
  static_assert(kYounger < 64, "vmcnt is a 6-bit counter");
  constexpr int kWaitLanded = (kYounger & 0xF) | (7 << 4) | (0 << 8) | ((kYounger >> 4) << 14);
  constexpr int kWaitAll = (0 & 0xF) | (7 << 4) | (0 << 8) | (0 << 14);
  int stage_index = 0;
  auto iterate = [&](auto set, int step, auto last_steps) __attribute__((always_inline)) {
    constexpr std::integral_constant<int, (set.value + 1) % kSets> following{};
    constexpr std::integral_constant<int, (set.value + kSets - 1) % kSets> filling{};
    const int next_index = stage_index == kStages - 1 ? 0 : stage_index + 1;
    const int fill_index = stage_index == 0 ? kStages - 1 : stage_index - 1;
    uint32_t current = stage_index * (kStageChunks * 16), next = next_index * (kStageChunks * 16);
    asm volatile("" : "+s"(current), "+s"(next));  // (formed here: hoisted out of the loop, every stage's and slice's addresses fill registers)
    u32x4_t* fill = lds + fill_index * kStageChunks;
    const int ahead_a = min(step + kAhead, steps - 1), ahead_b = min(step + kSets - 1, steps - 1);
    static_range<0>(std::make_integer_sequence<int, 4>{}, [&](auto kk) __attribute__((always_inline)) {
      constexpr int slice = decltype(kk)::value;
      constexpr bool kLast = slice == 3;
      constexpr std::integral_constant<int, (slice + 1) % 4> next_kk{};
      constexpr std::integral_constant<int, kLast ? following.value : set.value> deq_set{};
      if constexpr (kLast) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(last_steps.value ? kWaitAll : kWaitLanded);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
      }
      fetch(kLast ? next : current, next_kk);
      if constexpr (kBlockBank && kLast) block_scale = next_scale;
      dequantize(deq_set, next_kk, c0);
      dequantize(deq_set, next_kk, c1);
      multiply(set, kk);
      if constexpr (kBlockBank && slice == 2) next_scale = depth_scales[side * kScaleRow + (step + 1) / (128 / BK)];
      constexpr int a_each = (kRowLoads + 1) / 2;
      constexpr int a_begin = slice * a_each < kRowLoads ? slice * a_each : kRowLoads;
      constexpr int a_end = a_begin + a_each < kRowLoads ? a_begin + a_each : kRowLoads;
      constexpr bool kWeights = slice == 2;
      load_a(fill, ahead_a, std::integral_constant<int, a_begin>{}, std::integral_constant<int, a_end>{});
      if constexpr (kWeights) load_b(filling, ahead_b);
      constexpr int kLoads = a_end - a_begin + (kWeights ? kLoadsB : 0);
      schedule_slice<0, TI, TI + (kBlockBank && slice == 2 ? 1 : 0), (kBf16 ? 0 : 17) + 2 * kLoads, kLoads>();
      __builtin_amdgcn_sched_barrier(0);
    });
    stage_index = next_index;
  };
  constexpr std::integral_constant<int, kRowLoads> every_row{};
  static_for<kAhead>([&](auto stage) __attribute__((always_inline)) {
    load_a(lds + decltype(stage)::value * kStageChunks, min(decltype(stage)::value, steps - 1), c0, every_row);
  });
  if constexpr (kBlockBank) {
    static_assert(2 * kMaxDepthBlocks <= kTallThreads, "one scale a thread");
    if (tid < 2 * depth_blocks) depth_scales[tid / depth_blocks * kScaleRow + tid % depth_blocks] = early_scale;
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(kWaitAll);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  if constexpr (kFp4) tensor_scale = __builtin_bit_cast(float, __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, tensor_scale)));
  if constexpr (kBlockBank) block_scale = depth_scales[side * kScaleRow];
  fetch(0, c0);
  dequantize(c0, c0, c0);
  dequantize(c0, c0, c1);
  int step = 0;
  for (; step + kSets <= steps; step += kSets)
    static_range<0>(std::make_integer_sequence<int, kSets>{}, [&](auto at) __attribute__((always_inline)) { iterate(at, step + decltype(at)::value, std::false_type{}); });
  static_range<0>(std::make_integer_sequence<int, kSets - 1>{}, [&](auto at) __attribute__((always_inline)) {
    if (step < steps) iterate(at, step++, std::true_type{});
  });
  __builtin_amdgcn_s_waitcnt(kWaitAll);  // the clamped loads of the last steps still target the LDS

  // ---- epilogue: the arithmetic, the staging and the stores of gemm.hip's, in one pass ----
  using Staging = TallStaging<PAIRED>;
  uint32_t* staged = reinterpret_cast<uint32_t*>(lds);
  int* out_row_of = reinterpret_cast<int*>(staged + Staging::kRowTable);
  const bool odd_lane = lane & 1;
  const uint32_t swap_select = odd_lane ? 0x03020706u : 0x05040100u;
  const float factor = kFp4 ? 256.0f * tensor_scale : 1.0f;
  float bias = 0.0f;
  if constexpr (!PAIRED) {
    if (p.bias) bias = p.bias[static_cast<size_t>(expert) * p.width + column + lane % 32];
    if (p.round_bias) bias = bf16_round(bias);
  }
  int out_row = 0;
  if (tid < kTallRows) {
    const int sorted = row0 + min(tid, valid_rows - 1);
    out_row = p.scatter ? p.scatter[sorted] : sorted;
  }
  __builtin_amdgcn_s_barrier();  // every wavefront has read its last A fragments and its loads have landed: the ring is free
  asm volatile("" ::: "memory");
  // the lane's rows q (low half) and q + 1 (high half) of its column, rounded
  auto rounded_pair = [&](auto i, auto q) __attribute__((always_inline)) {
    constexpr int at = decltype(i)::value, pair = decltype(q)::value;
    if constexpr (PAIRED) {
      return pack_bf16(acc[at][pair] * factor, acc[at][pair + 1] * factor);
    } else if constexpr (kFp4) {
      return pack_bf16(acc[at][pair] * factor + bias, acc[at][pair + 1] * factor + bias);
    } else {
      return pack_bf16(acc[at][pair] + bias, acc[at][pair + 1] + bias);
    }
  };
  // the even lane keeps row q of both columns and the odd lane row q + 1
  auto stage_pair = [&](auto i, auto q, uint32_t mine, int tile_column) __attribute__((always_inline)) {
    constexpr int at = decltype(i)::value, pair = decltype(q)::value;
    const int row = 32 * at + 8 * (pair / 4) + 4 * (lane / 32) + pair % 4 + (odd_lane ? 1 : 0);
    const uint32_t other = __builtin_amdgcn_mov_dpp(mine, 0xB1, 0xF, 0xF, true);
    staged[row * Staging::kRowDwords + (tile_column + (lane % 32 & ~1)) / 2] = __builtin_amdgcn_perm(other, mine, swap_select);
  };
  if constexpr (PAIRED) {
    constexpr int kKept = (TI + 1) / 2;  // the gate's wavefronts finish the first row tiles, the up projection's the rest
    u32x4_t* exchange = reinterpret_cast<u32x4_t*>(staged + Staging::kExchange) + (wave % 4) * (8 * 2 * 64) + lane;
    static_for<TI>([&](auto i) __attribute__((always_inline)) {
      constexpr int at = decltype(i)::value;
      if ((at < kKept) != (side == 0)) {
        u32x4_t words[2];
        static_for<8>([&](auto h) __attribute__((always_inline)) {
          words[decltype(h)::value / 4][decltype(h)::value % 4] = rounded_pair(i, std::integral_constant<int, 2 * decltype(h)::value>{});
        });
        exchange[(at * 2) * 64] = words[0];
        exchange[(at * 2 + 1) * 64] = words[1];
      }
    });
    if (tid < kTallRows) out_row_of[tid] = out_row;
    __syncthreads();
    const bool plain_swiglu = p.limit <= 0.0f && p.gating == DEW_MOE_GATE_SILU;
    auto finish = [&](auto plain, auto gate_side) __attribute__((always_inline)) {
      static_for<TI>([&](auto i) __attribute__((always_inline)) {
        constexpr int at = decltype(i)::value;
        if constexpr ((at < kKept) == gate_side.value) {
          const u32x4_t words[2] = {exchange[(at * 2) * 64], exchange[(at * 2 + 1) * 64]};
          static_for<8>([&](auto h) __attribute__((always_inline)) {
            constexpr std::integral_constant<int, 2 * decltype(h)::value> q{};
            const uint32_t own = rounded_pair(i, q), got = words[decltype(h)::value / 4][decltype(h)::value % 4];
            const uint32_t gate = gate_side.value ? own : got, up = gate_side.value ? got : own;
            const float gate0 = __uint_as_float(gate << 16), gate1 = __uint_as_float(gate & 0xFFFF0000u);
            const float up0 = __uint_as_float(up << 16), up1 = __uint_as_float(up & 0xFFFF0000u);
            uint32_t mine;
            if constexpr (decltype(plain)::value)
              mine = swiglu_rounded(gate0, up0) | (static_cast<uint32_t>(swiglu_rounded(gate1, up1)) << 16);
            else
              mine = gated_rounded(gate0, up0, p.limit, p.gating) | (static_cast<uint32_t>(gated_rounded(gate1, up1, p.limit, p.gating)) << 16);
            stage_pair(i, q, mine, 32 * (wave % 4));
          });
        }
      });
    };
    if (plain_swiglu) {
      if (side == 0)
        finish(std::true_type{}, std::true_type{});
      else
        finish(std::true_type{}, std::false_type{});
    } else if (side == 0) {
      finish(std::false_type{}, std::true_type{});
    } else {
      finish(std::false_type{}, std::false_type{});
    }
  } else {
    static_for<TI>([&](auto i) __attribute__((always_inline)) {
      static_for<8>([&](auto h) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, 2 * decltype(h)::value> q{};
        stage_pair(i, q, rounded_pair(i, q), 32 * wave);
      });
    });
    if (tid < kTallRows) out_row_of[tid] = out_row;
  }
  __syncthreads();
  constexpr int kRowChunks = Staging::kColumns / 8, kStoreIters = TI * 32 * kRowChunks / kTallThreads;
  static_assert(TI * 32 * kRowChunks % kTallThreads == 0, "whole store rounds");
  u32x4_t words[kStoreIters];
  int out_rows[kStoreIters];
#pragma unroll
  for (int it = 0; it < kStoreIters; ++it) {
    const int item = tid + it * kTallThreads;
    words[it] = *reinterpret_cast<const u32x4_t*>(staged + (item / kRowChunks) * Staging::kRowDwords + (item % kRowChunks) * 4);
    out_rows[it] = out_row_of[item / kRowChunks];
  }
#pragma unroll
  for (int it = 0; it < kStoreIters; ++it) {
    const int item = tid + it * kTallThreads, chunk = item % kRowChunks;
    if (item / kRowChunks < valid_rows && n0 + chunk * 8 < p.width)
      *reinterpret_cast<u32x4_t*>(p.out + static_cast<size_t>(out_rows[it]) * p.width + n0 + chunk * 8) = words[it];
  }
}

// (MODE: kPlain or kSwigluOfTwo; gemm.hip's kernels of the same name are the shorter tiles', of four wavefronts)
template <int FORMAT, int MODE, int WAVES>
__global__ __launch_bounds__(64 * WAVES, 2) void grouped_gemm_kernel(GemmParams p) {
  constexpr bool PAIRED = MODE == kSwigluOfTwo;
  static_assert(64 * WAVES == kTallThreads, "eight wavefronts");
  extern __shared__ u32x4_t lds[];
  __shared__ float depth_scales[FORMAT == DEW_MOE_W_FP8_BLOCK ? 2 * kScaleRow : 1];
  constexpr int kColumns = TallStaging<PAIRED>::kColumns, kMostRows = 32 * kMostTiles<FORMAT>;
  const int tid = threadIdx.x, lane = tid % 64;

  // block -> (m-tile, strip), as in gemm.hip: chunks of group_m m-tiles x 8 strips dealt round-robin to the XCDs
  const int group_rows = p.group_m, chunk = 8 * group_rows;
  const int n_strips = (p.width + kColumns - 1) / kColumns;
  const int total = p.m_tile_bound * n_strips;
  const int local = blockIdx.x / 8;
  const int order = ((local / chunk) * 8 + blockIdx.x % 8) * chunk + local % chunk;
  if (order >= total) return;
  const int group = order / (group_rows * n_strips);
  const int group_m = min(group_rows, p.m_tile_bound - group * group_rows);
  const int within = order % (group_rows * n_strips);
  const int m_tile = group * group_rows + within % group_m;
  const int n0 = (within / group_m) * kColumns;

  // the m-tile's expert: an inclusive scan of the groups' tiles, 64 experts a round, by every wavefront for itself
  auto size_of = [&](int e) { return e >= p.experts ? 0 : p.sizes ? max(p.sizes[e], 0) : p.offsets[e + 1] - p.offsets[e]; };
  auto first_row_of = [&](int e) { return e >= p.experts || p.sizes ? 0 : p.offsets[e]; };
  int expert = -1, row0 = 0, valid_rows = 0, carried = 0, carried_rows = 0;
  int next_size = size_of(lane), next_first_row = first_row_of(lane);
  for (int base = 0; base < p.experts; base += 64) {
    const int size = next_size;
    int start = next_first_row;
    next_size = size_of(base + 64 + lane);
    next_first_row = first_row_of(base + 64 + lane);
    if (p.sizes) {
      const int rows = lanes_scanned(size);
      start = carried_rows + rows - size;
      carried_rows += __builtin_amdgcn_readlane(rows, 63);
    }
    const int tiles = (size + kMostRows - 1) / kMostRows;
    const int inclusive = lanes_scanned(tiles), first = carried + inclusive - tiles;
    const unsigned long long hit = __ballot(m_tile >= first && m_tile < first + tiles);
    if (hit != 0ull) {
      const int owner = __builtin_ctzll(hit);
      expert = base + owner;
      const int group_size = __builtin_amdgcn_readlane(size, owner), group_tiles = (group_size + kMostRows - 1) / kMostRows;
      const int rows_each = ((group_size + 31) / 32 + group_tiles - 1) / group_tiles * 32;  // equally many 32-row tiles each
      const int begin = (m_tile - __builtin_amdgcn_readlane(first, owner)) * rows_each;
      row0 = __builtin_amdgcn_readlane(start, owner) + begin;
      valid_rows = min(rows_each, group_size - begin);
      break;
    }
    carried += __builtin_amdgcn_readlane(inclusive, 63);
  }
  asm volatile("" : "+s"(expert), "+s"(row0), "+s"(valid_rows));  // (the loop ends here: the tile's code is not to be laid inside it)
  if (expert < 0) {  // past the last tile: the rows no expert owns are zero
    const int tail_begin = (p.sizes ? carried_rows : p.offsets[p.experts]) + (m_tile - carried) * kMostRows;
    const int tail_end = min(tail_begin + kMostRows, p.rows);
    for (int item = tid; item < (tail_end - tail_begin) * (kColumns / 8); item += kTallThreads) {
      const int sorted = tail_begin + item / (kColumns / 8), at = n0 + (item % (kColumns / 8)) * 8;
      const int row = p.scatter ? p.scatter[sorted] : sorted;
      if (at < p.width) *reinterpret_cast<u32x4_t*>(p.out + static_cast<size_t>(row) * p.width + at) = u32x4_t{0, 0, 0, 0};
    }
    return;
  }
  if (valid_rows <= 0) return;  // (a group whose equal tiles end before its last one)
  const TallTile tile{expert, row0, valid_rows, n0};
  switch ((valid_rows + 31) / 32) {
    case 8:
      if constexpr (kMostTiles<FORMAT> == 8) return tall_tile<FORMAT, PAIRED, 8>(p, tile, lds, depth_scales);
      return;
    case 7: return tall_tile<FORMAT, PAIRED, 7>(p, tile, lds, depth_scales);
    case 6: return tall_tile<FORMAT, PAIRED, 6>(p, tile, lds, depth_scales);
    case 5: return tall_tile<FORMAT, PAIRED, 5>(p, tile, lds, depth_scales);
    case 4: return tall_tile<FORMAT, PAIRED, 4>(p, tile, lds, depth_scales);
    case 3: return tall_tile<FORMAT, PAIRED, 3>(p, tile, lds, depth_scales);
    default: return tall_tile<FORMAT, PAIRED, 2>(p, tile, lds, depth_scales);
  }
}

template <int FORMAT, int... TILES>
constexpr size_t largest_ring(std::integer_sequence<int, TILES...>) {
  size_t most = 0;
  ((most = std::max(most, static_cast<size_t>(TallDepth<FORMAT, TILES + 1>::kStages) * TallDepth<FORMAT, TILES + 1>::kStageChunks * 16)), ...);
  return most;
}

template <int FORMAT, bool PAIRED>
static int launch_tall_kernel(const char* who, GemmParams p, hipStream_t stream) {
  constexpr size_t kShared = TallStaging<PAIRED>::kBytes;
  static_assert(largest_ring<FORMAT>(std::make_integer_sequence<int, kMostTiles<FORMAT>>{}) <= kShared, "the rings fit what the staged tile takes");
  auto kernel = grouped_gemm_kernel<FORMAT, PAIRED ? kSwigluOfTwo : kPlain, kTallThreads / 64>;
  static std::once_flag configured;
  static hipError_t reserved = hipSuccess;
  std::call_once(configured, [&] { reserved = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kShared)); });
  if (reserved != hipSuccess) return fail(DEW_MOE_ELAUNCH, "%s: cannot reserve %zu bytes of LDS", who, kShared);
  constexpr int kColumns = TallStaging<PAIRED>::kColumns;
  constexpr int kMostRows = 32 * kMostTiles<FORMAT>;
  p.m_tile_bound = (p.rows + kMostRows - 1) / kMostRows + p.experts + 1;
  p.group_m = 2;
  const int total = p.m_tile_bound * ((p.width + kColumns - 1) / kColumns), round = 64 * p.group_m;
  hipLaunchKernelGGL(kernel, dim3((total + round - 1) / round * round), dim3(kTallThreads), kShared, stream, p);
  return launched(who);
}

int launch_tall(const char* who, const GemmParams& p, int format, bool paired, hipStream_t stream) {
  switch (format) {
    case DEW_MOE_W_FP8_BLOCK:
      return paired ? launch_tall_kernel<DEW_MOE_W_FP8_BLOCK, true>(who, p, stream) : launch_tall_kernel<DEW_MOE_W_FP8_BLOCK, false>(who, p, stream);
    case DEW_MOE_W_FP8_CHANNEL:
      return launch_tall_kernel<DEW_MOE_W_FP8_CHANNEL, false>(who, p, stream);
    case DEW_MOE_W_BF16:
      return paired ? launch_tall_kernel<DEW_MOE_W_BF16, true>(who, p, stream) : launch_tall_kernel<DEW_MOE_W_BF16, false>(who, p, stream);
    default:
      return launch_tall_kernel<DEW_MOE_W_NVFP4, false>(who, p, stream);
  }
}

}  // namespace dew
