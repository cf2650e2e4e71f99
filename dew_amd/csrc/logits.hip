// Router gate logits: logits[t, e] = sum_d f32(x[t, d]) * kernel[d, e], products exact in fp32 and summed in fp32
// (reference src/dew/nn/moe.py:526-534: tokens widened to fp32, Precision.HIGHEST), and group offsets.
// Depths in whole 16s run on the matrix unit, the fp32 gate as three bf16 terms (below): a block takes 32 (or 64) tokens and up to
// four 32-expert tiles, its wavefronts a share of the depth each; the partial sums of a tile meet in LDS in wavefront order, so the
// result does not depend on timing. A decode step's few tokens take 16 x 16 tiles of the fp32 instruction (v_mfma_f32_16x16x4_f32),
// four times the blocks: 64 tokens of GPT-OSS's 2880 x 32 gate in about 5 us. Depths in no whole 16s take the plain kernel below (a
// 64-token x 64-expert tile, 16-deep LDS steps, fp32 FMA; 1.3 ms for 8192 tokens of a 7168 x 256 gate, where the terms take 102 us).
#include <mutex>

#include "common.h"
#include "sort.h"

namespace dew {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The exact split of the gate kernel: an fp32 value of 2^-110 and more is the sum of three bf16 values, its upper 16 bits, the upper 16 of what is
// left and the 8 bits that are left then, and a token's bf16 element times any of them is exact in fp32 (a column with a smaller value,
// whose last bits no term holds, is seen and formed on the fp32 instruction). So three bf16 matrix instructions 16 deep (32 cycles each) give the
// fp32 products that eight fp32 ones 2 deep (64 cycles each) do; the sum of 16 products is cut off inside the instruction, where the fp32 ones
// round after each, so that the cuts of a long chain of sums of one sign add up: chains end, in fp32, after at most 1024 depths (launch_logits).
// What bounds it: the splitting's vector work beside the matrix instructions (11 and a half a pair of gate values against 24 x 32
// cycles a 16 deep chunk of 64 x 128) where the experts are many, x from memory where they are few. Measured against the
// fp32 instruction, the tokens from memory (us; error against float64, 2-norm, of normal tokens and gate and of positive ones): 8192 x 7168 x 256 327 -> 105
// (7.5e-7 -> 3.2e-7, 3.0e-7 -> 1.1e-7), 16384 x 4096 x 8 65 -> 30 (6.2e-7 -> 3.7e-7, 2.5e-7 -> 2.1e-7), 4096 x 4096 x 8 36 -> 18 (5.6e-7 -> 1.8e-7, 2.5e-7 -> 7.5e-8),
// 8192 x 4096 x 128 130 -> 45 (5.8e-7 -> 3.4e-7, 2.5e-7 -> 2.1e-7). The mean error, nil there, is -1e-8 to -5e-8 of normal logits' root mean square here.
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t upper_halves(float high, float low) {
  return __builtin_amdgcn_perm(__float_as_uint(high), __float_as_uint(low), 0x07060302u);
}
// The same, and the bits of both seen in `seen` (one block: apart, the compiler keeps the values for the second, and 8192 x 7168 x 256 takes 137 us
// instead of 102).
__device__ __forceinline__ uint32_t upper_halves(float high, float low, uint32_t& seen) {
  uint32_t word;
  asm("v_or3_b32 %0, %0, %2, %3\n\tv_perm_b32 %1, %2, %3, %4" : "+v"(seen), "=&v"(word) : "v"(high), "v"(low), "s"(0x07060302u));
  return word;
}
__device__ __forceinline__ float below_upper(float value) { return value - __uint_as_float(__float_as_uint(value) & 0xFFFF0000u); }

// The sums of depths `from` to `to` (whole 16s) for the tiles that `needed` names of a tile of 32 tokens beside TILES of 32 experts, `row` and
// `column` the lane's own, on the fp32 instruction: what the terms cannot give. Bound by the matrix pipe, 512 cycles a tile and 16 deep
// chunk, where a row of tiles is needed, by its loads, which go out two chunks ahead, where one is. Finite
// operands, a token of NaN, and nothing else, us: 8192 x 7168 x 256 102, 218 and 317, 2048 x 7168 x 256 46, 81 and 119, 4096 x 4096 x 8 16, 38 and 43 (the
// fp32 instruction alone 300, 92 and 34; where every such sum's lane walked the depth for it a token of NaN took 7057, 1696 and 339).
template <int TILES>
__device__ __forceinline__ void plain_sums(const bf16_t* __restrict__ row, const float* __restrict__ column, int experts, int from, int to, uint32_t needed,
                                           f32x16 (&acc)[TILES]) {
  struct __attribute__((packed, aligned(4))) Neighbours {
    float of[TILES];
  };
  constexpr int kAhead = 2;  // chunks of a set
  const int lower = 8 * (threadIdx.x % 64 / 32);
#pragma unroll
  for (int c = 0; c < TILES; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[c][i] = 0.0f;
  u32x4 words[2][kAhead];
  Neighbours g[2][kAhead][8];
  auto load = [&](int set, int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int ahead = 0; ahead < kAhead; ++ahead) {
      const int at = min(chunk + 16 * ahead, to - 16) + lower;  // (past the share: the last chunk again, which multiplies nothing)
      words[set][ahead] = *reinterpret_cast<const u32x4*>(row + at);
#pragma unroll
      for (int j = 0; j < 8; ++j) g[set][ahead][j] = *reinterpret_cast<const Neighbours*>(column + static_cast<size_t>(at + j) * experts);
    }
  };
  auto multiply = [&](int set, int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int ahead = 0; ahead < kAhead; ++ahead) {
      if (chunk + 16 * ahead >= to) continue;
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        if (!(needed >> c & 1)) continue;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const uint32_t word = words[set][ahead][j / 2];
          acc[c] = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(j % 2 ? word & 0xFFFF0000u : word << 16), g[set][ahead][j].of[c], acc[c], 0, 0, 0);
        }
      }
    }
  };
  load(0, from);
  for (int chunk = from; chunk < to; chunk += 32 * kAhead) {
    load(1, chunk + 16 * kAhead);
    multiply(0, chunk);
    load(0, chunk + 32 * kAhead);
    multiply(1, chunk + 16 * kAhead);
  }
}

// The sums of a share of the depth, its steps of 16 x CHUNKS from `first` to `last`, for ROWS tiles of 32 tokens from t0 on and TILES tiles of
// 32 experts. A lane's depths of a step are contiguous in its token's row (64 bytes of four chunks, so that every line of x is asked
// for once); a chunk's instructions take 8 of each half's. Its experts are TILES neighbours, one a tile, from `column` on: one load a depth.
// `end`: the depth that the share goes to, up to three chunks behind its last step; WHOLE: none, as the depth is whole steps. `chain`: the
// steps, whole sets of loads, after which sums go to `aside`, the lane's place in the LDS, and start from zero.
template <int ROWS, int TILES, int AHEAD, int CHUNKS, bool WHOLE>
__device__ __forceinline__ void logit_terms(const bf16_t* __restrict__ x, const float* __restrict__ kernel, int tokens, int depth, int experts,
                                            int t0, int column, int first, int last, int end, int chain, f32x4* aside, f32x16 (&acc)[ROWS][TILES]) {
  struct __attribute__((packed, aligned(4))) Neighbours {
    float of[TILES];
  };
  constexpr int kStep = 16 * CHUNKS;
  const int lane = threadIdx.x % 64, half = kStep / 2 * (lane / 32);
  const bf16_t* a_src[ROWS];
#pragma unroll
  for (int r = 0; r < ROWS; ++r)  // (rows past the tokens repeat the last one; they are not stored)
    a_src[r] = x + static_cast<size_t>(min(t0 + 32 * r + lane % 32, tokens - 1)) * depth;
#pragma unroll
  for (int r = 0; r < ROWS; ++r)
#pragma unroll
    for (int c = 0; c < TILES; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][c][i] = 0.0f;
  if (first >= last) return;
  // Loads return in order, so the gate's, which the L2 holds, wait for the rows', which come from memory, and both are asked for the
  // same time ahead: AHEAD steps. A chunk's gate values are split one chunk ahead, between the matrix instructions of the chunk before.
  constexpr int kSets = 2 * AHEAD;
  u32x4 a_words[kSets][ROWS][CHUNKS];
  Neighbours g[AHEAD][CHUNKS][8];
  bf16x8 terms[2][TILES][3];
  uint32_t dropped[TILES];  // the bits of a lane's gate values that no term holds, in its lower half
#pragma unroll
  for (int c = 0; c < TILES; ++c) dropped[c] = 0;
  auto load_rows = [&](int set, int step) __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < CHUNKS; ++c) a_words[set][r][c] = *reinterpret_cast<const u32x4*>(a_src[r] + (kStep * step + half + 8 * c));
  };
  auto load_gate = [&](int set, int step, int chunk) __attribute__((always_inline)) {
    // (the same for the wavefront: a load's address is a scalar base and the lane's own offset)
    const float* b_src = kernel + static_cast<size_t>(kStep * step + 8 * chunk) * experts;
    const uint32_t lower = half * experts + column;
#pragma unroll
    for (int j = 0; j < 8; ++j, b_src += experts) g[set][chunk][j] = *reinterpret_cast<const Neighbours*>(b_src + lower);
  };
  auto split = [&](int set, int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < TILES; ++c) {
      float most[8], rest[8], least[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) most[j] = g[set][chunk][j].of[c];
#pragma unroll
      for (int j = 0; j < 8; ++j) rest[j] = below_upper(most[j]);
#pragma unroll
      for (int j = 0; j < 8; ++j) least[j] = below_upper(rest[j]);
      auto fragment = [](const float (&v)[8]) __attribute__((always_inline)) {
        return __builtin_bit_cast(bf16x8, u32x4{upper_halves(v[1], v[0]), upper_halves(v[3], v[2]), upper_halves(v[5], v[4]), upper_halves(v[7], v[6])});
      };
      terms[chunk % 2][c][0] = __builtin_bit_cast(bf16x8, u32x4{upper_halves(least[1], least[0], dropped[c]), upper_halves(least[3], least[2], dropped[c]),
                                                                upper_halves(least[5], least[4], dropped[c]), upper_halves(least[7], least[6], dropped[c])});
      terms[chunk % 2][c][1] = fragment(rest);
      terms[chunk % 2][c][2] = fragment(most);
    }
  };
  auto walk = [&](int set, int step, bool more) __attribute__((always_inline)) {
    if (more) load_rows((set + AHEAD) % kSets, min(step + AHEAD, last - 1));  // (behind the last step: that step again, which multiplies nothing)
#pragma unroll
    for (int chunk = 0; chunk < CHUNKS; ++chunk) {
#pragma unroll
      for (int term = 0; term < 3; ++term)
#pragma unroll
        for (int c = 0; c < TILES; ++c)
#pragma unroll
          for (int r = 0; r < ROWS; ++r)
            acc[r][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a_words[set][r][chunk]), terms[chunk % 2][c][term], acc[r][c], 0, 0, 0);
      const int next = chunk < CHUNKS - 1 ? set % AHEAD : (set + 1) % AHEAD;  // the set of the chunk behind this one
      if (more || chunk < CHUNKS - 1) split(next, (chunk + 1) % CHUNKS);
      if (more) load_gate(next, min(step + AHEAD + (chunk == CHUNKS - 1), last - 1), (chunk + 1) % CHUNKS);
    }
  };
  // Chains end between two loops or within one, by which the compiler keeps the loads in registers: 2 x 4 tiles 105 us between, 119 within (8192 x 7168 x
  // 256), 2 x 1 43 and 46 (2112 x 7168 x 160), but 1 x 1 39 and 34 (5000 x 7168 x 32), and eight wavefronts 45 and 40 (2048 x 7168 x 256).
  constexpr bool kBetween = ROWS * TILES * AHEAD >= 4;
  auto put_aside = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
#pragma unroll
        for (int i = 0; i < 16; i += 4) aside[((r * TILES + c) * 4 + i / 4) * 64] = f32x4{acc[r][c][i], acc[r][c][i + 1], acc[r][c][i + 2], acc[r][c][i + 3]};
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][c][i] = 0.0f;
      }
    aside += ROWS * TILES * 256;
  };
  auto take_back = [&]() __attribute__((always_inline)) {
    aside -= ROWS * TILES * 256;
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int c = 0; c < TILES; ++c)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[r][c][i] += aside[((r * TILES + c) * 4 + i / 4) * 64][i % 4];
  };
#pragma unroll
  for (int ahead = 0; ahead < AHEAD; ++ahead) {
    load_rows(ahead, min(first + ahead, last - 1));
#pragma unroll
    for (int chunk = 0; chunk < CHUNKS; ++chunk) load_gate(ahead, min(first + ahead, last - 1), chunk);
  }
  split(0, 0);
  if (CHUNKS < 4 && last - first == 1) {  // (a share of a short depth: nothing behind it is asked for)
    walk(0, first, false);
  } else {
    load_gate(0, min(first + AHEAD, last - 1), 0);
    int step = first;
    int until = first + chain;
    for (;;) {
      const int stop = kBetween ? min(until, last) : last;
      for (; step + kSets <= stop; step += kSets) {  // (no way out in the middle: every load would be waited for there)
#pragma unroll
        for (int set = 0; set < kSets; ++set) walk(set, step + set, true);
        if (kBetween || step + kSets != until || until >= last) continue;
        put_aside();
        until += chain;
      }
      if (!kBetween || until >= last) break;
      put_aside();
      until += chain;
    }
#pragma unroll
    for (int set = 0; set < kSets - 1; ++set)
      if (step + set < last) walk(set, step + set, AHEAD > 1);
#pragma unroll 1
    for (; until > first + chain; until -= chain) take_back();
  }
  // An infinity among the operands meets a term that is zero, a gate value's terms are not those of an infinity or a NaN, and below 2^-110 its
  // last bits lie under the least bf16 value: tiles with a sum that is no finite number, or with a column that dropped bits, are formed again on
  // the fp32 instruction, and those sums taken from there.
  bool inexact[TILES];
#pragma unroll
  for (int c = 0; c < TILES; ++c) inexact[c] = ((dropped[c] | __shfl_xor(dropped[c], 32, 64)) & 0xFFFFu) != 0;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    uint32_t needed = 0;
#pragma unroll
    for (int c = 0; c < TILES; ++c) {
      float zero = 0.0f;  // (a NaN where any sum is no finite number)
#pragma unroll
      for (int i = 0; i < 16; ++i) zero = fmaf(0.0f, acc[r][c][i], zero);
      if (__any(zero != 0.0f || inexact[c])) needed |= 1u << c;
    }
    if (needed == 0) continue;
    f32x16 plain[TILES];
    plain_sums<TILES>(a_src[r], kernel + column, experts, kStep * first, kStep * last, needed, plain);
#pragma unroll
    for (int c = 0; c < TILES; ++c)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[r][c][i] = __builtin_isfinite(acc[r][c][i]) && !inexact[c] ? acc[r][c][i] : plain[c][i];
  }
  if (WHOLE || end == kStep * last) return;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    f32x16 plain[TILES];
    plain_sums<TILES>(a_src[r], kernel + column, experts, kStep * last, end, (1u << TILES) - 1, plain);
#pragma unroll
    for (int c = 0; c < TILES; ++c) acc[r][c] += plain[c];
  }
}

// WAVES wavefronts a block split the depth; their sums meet in LDS in wavefront order, WAVES registers of the tiles at a time.
template <int ROWS, int TILES, int WAVES, int AHEAD, int CHUNKS, bool WHOLE>
__global__ __launch_bounds__(64 * WAVES) void router_logits_mfma_kernel(const bf16_t* __restrict__ x, const float* __restrict__ kernel,
                                                                        const float* __restrict__ bias, float* __restrict__ logits,
                                                                        int tokens, int depth, int experts, int chain, int slots) {
  struct __attribute__((packed, aligned(4))) Neighbours {
    float of[TILES];
  };
  __shared__ float partial[WAVES][WAVES][TILES][64];  // [wavefront][register][tile][lane]
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int t0 = blockIdx.x * 32 * ROWS, e0 = TILES * (32 * blockIdx.y + lane % 32);
  // (lanes past the experts repeat the last ones: what they share with the lane before is the same sum)
  const int column = min(e0, experts - TILES);
  extern __shared__ f32x4 aside[];  // [wavefront][slot][row tile][tile][quad of registers][lane]
  const int steps = depth / (16 * CHUNKS), first = steps * wave / WAVES, last = steps * (wave + 1) / WAVES;
  f32x16 acc[ROWS][TILES];
  logit_terms<ROWS, TILES, AHEAD, CHUNKS, WHOLE>(x, kernel, tokens, depth, experts, t0, column, first, last, wave == WAVES - 1 ? depth : 16 * CHUNKS * last,
                                                 chain, aside + wave * slots * (ROWS * TILES * 256) + lane, acc);
  // register i of lane l is the sum of token 8 (i / 4) + 4 (l / 32) + i % 4 and the lane's expert
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
#pragma unroll
    for (int i0 = 0; i0 < 16; i0 += WAVES) {
      if (r + i0 > 0) __syncthreads();
#pragma unroll
      for (int i = 0; i < WAVES; ++i)
#pragma unroll
        for (int c = 0; c < TILES; ++c) partial[wave][i][c][lane] = acc[r][c][i0 + i];
      __syncthreads();
      const int i = i0 + wave, t = t0 + 32 * r + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
      Neighbours sums;
#pragma unroll
      for (int c = 0; c < TILES; ++c) {
        float sum = partial[0][wave][c][lane];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) sum += partial[w][wave][c][lane];
        sums.of[c] = sum;
      }
      if (t < tokens && e0 < experts) {
#pragma unroll
        for (int c = 0; c < TILES; ++c)
          // a biased router (GPT-OSS's, src/dew/nn/gpt_oss.py:163-165) adds its fp32 bias to the finished sum
          if (bias) sums.of[c] += bias[column + c];
        *reinterpret_cast<Neighbours*>(logits + static_cast<size_t>(t) * experts + column) = sums;
      }
    }
  }
}

// The chains of a wavefront's share: of at most 1024 depths, and of 512 on eight wavefronts, as far as the LDS has room for the sums set aside (2 x 4
// tiles up to 8192 deep, the others up to 12 288 and more). Sixteen wavefronts walk as much only from 16 384 depths on. Error against float64 (2-norm) of
// positive tokens and gate, in one chain, in these, and by the fp32 instruction: 8192 x 7168 x 256 7.2e-7, 1.1e-7 and 3.0e-7, 3000 x 5120 x 128
// 3.5e-7, 9.5e-8 and 2.8e-7, 2048 x 7168 x 256 1.1e-7, 6.6e-8 and 9.6e-8; at 1024 depths 2.1e-7 and 2.5e-7 (3000 x 4096 x 256).
template <int ROWS, int TILES, int WAVES, int AHEAD, int CHUNKS, bool WHOLE>
static int launch_logits(const bf16_t* x, const float* kernel, const float* bias, float* logits, int tokens, int depth, int experts, hipStream_t stream) {
  auto routine = router_logits_mfma_kernel<ROWS, TILES, WAVES, AHEAD, CHUNKS, WHOLE>;
  constexpr int kSlot = WAVES * ROWS * TILES * 64 * 16 * 4, kSlots = WAVES == 16 ? 0 : 131072 / kSlot;
  static std::once_flag configured;  // dynamic LDS above 64 KiB must be opted into once per kernel
  static hipError_t reserved = hipSuccess;
  std::call_once(configured, [&] {
    if (kSlots > 0) reserved = hipFuncSetAttribute(reinterpret_cast<const void*>(routine), hipFuncAttributeMaxDynamicSharedMemorySize, kSlots * kSlot);
  });
  if (reserved != hipSuccess) return fail(DEW_MOE_ELAUNCH, "dew_moe_router_logits: cannot reserve %d bytes of LDS", kSlots * kSlot);
  constexpr int kChain = (WAVES == 8 ? 512 : 1024) / (16 * CHUNKS), kSets = 2 * AHEAD;
  const int share = (depth / (16 * CHUNKS) + WAVES - 1) / WAVES, slots = min((share + kChain - 1) / kChain - 1, kSlots);
  const int chain = slots > 0 ? (share + (slots + 1) * kSets - 1) / ((slots + 1) * kSets) * kSets : 1 << 30;
  hipLaunchKernelGGL(routine, dim3((tokens + 32 * ROWS - 1) / (32 * ROWS), (experts + 32 * TILES - 1) / (32 * TILES)), dim3(64 * WAVES),
                     static_cast<size_t>(max(slots, 0)) * kSlot, stream, x, kernel, bias, logits, tokens, depth, experts, chain, slots);
  return launched("router_logits_mfma_kernel");
}

// The few tokens of a decode step on finer tiles: 16 tokens x 16 experts a block (v_mfma_f32_16x16x4_f32, the same
// rate a CU as the 32 x 32 form), sixteen wavefronts a share of the depth each. A 32 x 32 tile's block keeps its whole
// product on one CU's four matrix pipes (64 tokens of a 2880 x 32 gate: two blocks, 20 us); four times the blocks
// finish in a quarter of that. Lane l multiplies token l % 16 and expert l % 16 over the depths 4 (l / 16) .. + 3 of a
// 16-deep chunk, one depth an instruction; its four sums are tokens 4 (l / 16) + i of expert column l % 16.
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kShares = kLogitShares;  // the depth's shares, one a wavefront

// Sixteen shares of a short depth take steps of 32: in steps of 64 a depth of 512 leaves half of them without one (a layer's pass over
// 2048 tokens of a 512 x 8 gate 49.4 us, 48.5 with them).
static bool short_shares(int depth) { return depth < 1024; }

// 32 x 32 tiles few enough that sixteen shares of the depth spread them over the CUs. Past 2048 tokens only few experts', whose shares are few
// bytes: a layer's pass (us, finished logits and shares) of 7168 deep gates: 2100 tokens of 8 experts, 66 tiles, 159 and 147, 4096, 128, 258 and 251, 4500, 141, 266
// and 264, 6000, 188, 306 and 307, 8192 294 and 298; of 32 experts, 4096 tokens 229 and 221, 8000 355 and 360; of 512 deep ones of 8 experts 128 tiles 43.7 and
// 42.3, of 32 experts 40.6 and 41.9; of 64 experts, 132 tiles, 7168 deep 200 and 190, 512 deep 39.6 and 41.9.
static bool share_tiles(int tokens, int experts) {
  const long long tiles = static_cast<long long>((tokens + 31) / 32) * ((experts + 31) / 32);
  return tokens <= 2048 ? tiles < 112 : experts <= 32 && tiles <= 128;
}

// The sums of share `share` of the depth for 16 tokens from t0 on and 16 experts from e0 on.
__device__ __forceinline__ f32x4 fine_share(const bf16_t* __restrict__ x, const float* __restrict__ kernel, int tokens, int depth, int experts,
                                            int t0, int e0, int share) {
  const int lane = threadIdx.x % 64;
  const int chunks = depth / 16;
  const int first = static_cast<int>(static_cast<long long>(chunks) * share / kShares);
  const int last = static_cast<int>(static_cast<long long>(chunks) * (share + 1) / kShares);
  const bf16_t* a_src = x + static_cast<size_t>(min(t0 + lane % 16, tokens - 1)) * depth + 4 * (lane / 16);
  const float* b_src = kernel + static_cast<size_t>(4 * (lane / 16)) * experts + min(e0 + lane % 16, experts - 1);
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  // four chunks' loads are in flight while the four before them multiply (a wavefront's walk is a chain of round trips
  // otherwise: 28 chunks of a 7168-deep gate)
  constexpr int kAhead = 4;
  u32x2 words[2][kAhead];
  float b[2][kAhead][4];
  auto load = [&](int set, int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int ahead = 0; ahead < kAhead; ++ahead) {
      const int at = min(chunk + ahead, last - 1);  // (past the share: the last chunk again, which multiplies nothing)
      words[set][ahead] = *reinterpret_cast<const u32x2*>(a_src + at * 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) b[set][ahead][j] = b_src[static_cast<size_t>(at * 16 + j) * experts];
    }
  };
  auto multiply = [&](int set, int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int ahead = 0; ahead < kAhead; ++ahead) {
      if (chunk + ahead >= last) continue;
      const u32x2 w = words[set][ahead];
      const float a[4] = {__uint_as_float(w[0] << 16), __uint_as_float(w[0] & 0xFFFF0000u), __uint_as_float(w[1] << 16),
                          __uint_as_float(w[1] & 0xFFFF0000u)};
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], b[set][ahead][j], acc, 0, 0, 0);
    }
  };
  if (first < last) load(0, first);
  for (int chunk = first; chunk < last; chunk += 2 * kAhead) {
    if (chunk + kAhead < last) load(1, chunk + kAhead);
    multiply(0, chunk);
    if (chunk + 2 * kAhead < last) load(0, chunk + 2 * kAhead);
    if (chunk + kAhead < last) multiply(1, chunk + kAhead);
  }
  return acc;
}

__global__ __launch_bounds__(64 * kShares) void router_logits_fine_kernel(const bf16_t* __restrict__ x, const float* __restrict__ kernel,
                                                                          const float* __restrict__ bias, float* __restrict__ logits,
                                                                          int tokens, int depth, int experts) {
  __shared__ float partial[kShares][4][64];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int t0 = blockIdx.x * 16, e0 = blockIdx.y * 16;
  const f32x4 acc = fine_share(x, kernel, tokens, depth, experts, t0, e0, wave);
#pragma unroll
  for (int i = 0; i < 4; ++i) partial[wave][i][lane] = acc[i];
  __syncthreads();
  if (wave < 4) {  // wavefront i finishes register i of every lane, adding the wavefronts' partial sums in wavefront order
    float sum = partial[0][wave][lane];
#pragma unroll
    for (int w = 1; w < kShares; ++w) sum += partial[w][wave][lane];
    const int t = t0 + 4 * (lane / 16) + wave, e = e0 + lane % 16;
    if (t < tokens && e < experts) logits[static_cast<size_t>(t) * experts + e] = bias ? sum + bias[e] : sum;
  }
}

// The same shares, a block each, left as [share][token][expert] for a launch that adds them in the same order as it reads
// them (route_and_sort_kernel): a decode step's few tokens then spread over 16 times the CUs, with no barrier at the end.
// Measured: one token of a 2048 x 128 gate 6.2 -> 3.4 us, 64 tokens 7.5 -> 5.0, 24 tokens of a 2880 x 32 gate 10.8 -> 4.7.
__global__ __launch_bounds__(64) void router_logit_shares_kernel(const bf16_t* __restrict__ x, const float* __restrict__ kernel,
                                                                 float* __restrict__ partial, int tokens, int depth, int experts) {
  const int lane = threadIdx.x, t0 = blockIdx.x * 16, e0 = blockIdx.y * 16, share = blockIdx.z;
  const f32x4 acc = fine_share(x, kernel, tokens, depth, experts, t0, e0, share);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int t = t0 + 4 * (lane / 16) + i, e = e0 + lane % 16;
    if (t < tokens && e < experts) partial[(static_cast<size_t>(share) * tokens + t) * experts + e] = acc[i];
  }
}

// The shares of router_logits_mfma_kernel<1, 1, 16, 1, CHUNKS> the same way: 32 tokens x 32 experts of one share of the depth a wavefront,
// for the few hundred tokens whose tiles with sixteen wavefronts each leave CUs without one. The partial sums are that kernel's and
// are added in its order: the same bits.
template <int CHUNKS, bool WHOLE>
__global__ __launch_bounds__(64) void router_logit_tile_shares_kernel(const bf16_t* __restrict__ x, const float* __restrict__ kernel,
                                                                      float* __restrict__ partial, int tokens, int depth, int experts) {
  const int lane = threadIdx.x, t0 = blockIdx.x * 32, share = blockIdx.z;
  const int steps = depth / (16 * CHUNKS), first = steps * share / kShares, last = steps * (share + 1) / kShares;
  f32x16 acc[1][1];
  logit_terms<1, 1, 1, CHUNKS, WHOLE>(x, kernel, tokens, depth, experts, t0, min(32 * static_cast<int>(blockIdx.y) + lane % 32, experts - 1), first, last,
                               share == kShares - 1 ? depth : 16 * CHUNKS * last, 1 << 30, nullptr, acc);
  const int e = 32 * blockIdx.y + lane % 32;
  if (e >= experts) return;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int t = t0 + 8 * (i / 4) + 4 * (lane / 32) + i % 4;
    if (t < tokens) partial[(static_cast<size_t>(share) * tokens + t) * experts + e] = acc[0][0][i];
  }
}

// How a layer's gate leaves its logits: in shares, by 16 x 16 tiles as the fine launch's (up to kShareTokens tokens, and wherever
// dew_moe_router_logits takes that launch) or by 32 x 32 tiles as its sixteen wavefronts', or finished. Past some hundred such tiles
// the shares' sixteen times the bytes cost more than the idle CUs do. A layer's pass (us; tiles by the fp32 instruction still): 200 tokens of a 2048 x 8 gate 85.0 -> 81.4,
// 100 of 7168 x 256 (32 tiles) 393 -> 381, 2048 of 512 x 8 (64) 52.0 -> 50.3, 1111 of 2048 x 64 (70) 134.5 -> 131.9, 1000 of 7168 x 128
// (128) 489.5 and 490.4, 600 of 2048 x 256 (152) 284.6 and 288.
LogitShares logit_shares(int tokens, int depth, int experts) {
  if (depth % 16 != 0) return kNoShares;
  if (tokens <= kShareTokens) return kFineShares;
  const long long blocks = static_cast<long long>((tokens + 31) / 32) * ((experts + 31) / 32);
  if (depth < 64 || !share_tiles(tokens, experts)) return kNoShares;
  return blocks < 64 ? kFineShares : kTileShares;
}

int router_logit_shares(const void* x, const float* kernel, float* partial, int tokens, int depth, int experts, hipStream_t stream) {
  if (logit_shares(tokens, depth, experts) == kTileShares) {
    auto routine = short_shares(depth) ? (depth % 32 == 0 ? router_logit_tile_shares_kernel<2, true> : router_logit_tile_shares_kernel<2, false>)
                                       : (depth % 64 == 0 ? router_logit_tile_shares_kernel<4, true> : router_logit_tile_shares_kernel<4, false>);
    hipLaunchKernelGGL(routine, dim3((tokens + 31) / 32, (experts + 31) / 32, kShares), dim3(64), 0, stream,
                       static_cast<const bf16_t*>(x), kernel, partial, tokens, depth, experts);
    return launched("router_logit_tile_shares_kernel");
  }
  hipLaunchKernelGGL(router_logit_shares_kernel, dim3((tokens + 15) / 16, (experts + 15) / 16, kShares), dim3(64), 0, stream,
                     static_cast<const bf16_t*>(x), kernel, partial, tokens, depth, experts);
  return launched("router_logit_shares_kernel");
}

constexpr int LT = 64, LE = 64, LK = 16;

__global__ __launch_bounds__(256) void router_logits_kernel(const bf16_t* __restrict__ x, const float* __restrict__ kernel,
                                                            const float* __restrict__ bias, float* __restrict__ logits,
                                                            int tokens, int depth, int experts) {
  __shared__ float xs[LK][LT + 1];
  __shared__ float ks[LK][LE + 1];
  const int t0 = blockIdx.x * LT, e0 = blockIdx.y * LE;
  const int tx = threadIdx.x % 16, ty = threadIdx.x / 16;  // thread owns tokens ty*4.., experts tx*4..
  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.0f;
  for (int d0 = 0; d0 < depth; d0 += LK) {
    for (int item = threadIdx.x; item < LT * LK; item += 256) {
      const int t = item / LK, d = item % LK;
      xs[d][t] = (t0 + t < tokens && d0 + d < depth) ? bf16_to_f32(x[static_cast<size_t>(t0 + t) * depth + d0 + d]) : 0.0f;
    }
    for (int item = threadIdx.x; item < LK * LE; item += 256) {
      const int d = item / LE, e = item % LE;
      ks[d][e] = (d0 + d < depth && e0 + e < experts) ? kernel[static_cast<size_t>(d0 + d) * experts + e0 + e] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int d = 0; d < LK; ++d) {
      float a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = xs[d][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = ks[d][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int t = t0 + ty * 4 + i, e = e0 + tx * 4 + j;
      // a biased router (GPT-OSS's, src/dew/nn/gpt_oss.py:163-165) adds its fp32 bias to the finished sum
      if (t < tokens && e < experts) logits[static_cast<size_t>(t) * experts + e] = bias ? acc[i][j] + bias[e] : acc[i][j];
    }
}

__global__ __launch_bounds__(64) void group_offsets_kernel(const int32_t* __restrict__ sizes, int32_t* __restrict__ offsets, int experts, int unit) {
  write_group_offsets(sizes, offsets, experts, unit);
}

}  // namespace dew

extern "C" int dew_moe_router_logits(const void* x, const float* kernel, const float* bias, float* logits, int32_t tokens,
                                     int32_t depth, int32_t experts, void* stream) {
  using namespace dew;
  DEW_REQUIRE(tokens >= 0 && depth >= 1 && experts >= 1, "dew_moe_router_logits: tokens %d depth %d experts %d", tokens, depth, experts);
  if (tokens == 0) return DEW_MOE_OK;
  DEW_REQUIRE(x && kernel && logits, "dew_moe_router_logits: x, kernel and logits must not be null");
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int tiles = (experts + 31) / 32;
  if (depth % 16 == 0 && depth >= 64 && (reinterpret_cast<uintptr_t>(x) & 15u) == 0) {
    if (static_cast<long long>((tokens + 31) / 32) * tiles < 64) {  // a decode step: finer tiles, four times the blocks
      hipLaunchKernelGGL(router_logits_fine_kernel, dim3((tokens + 15) / 16, (experts + 15) / 16), dim3(1024), 0, s,
                         static_cast<const bf16_t*>(x), kernel, bias, logits, tokens, depth, experts);
      return launched("router_logits_fine_kernel");
    }
#define DEW_LOGITS(ROWS, TILES, WAVES, AHEAD, CHUNKS) \
  return (depth % (16 * CHUNKS) == 0 ? launch_logits<ROWS, TILES, WAVES, AHEAD, CHUNKS, true> : launch_logits<ROWS, TILES, WAVES, AHEAD, CHUNKS, false>)( \
      static_cast<const bf16_t*>(x), kernel, bias, logits, tokens, depth, experts, s)
    auto blocks = [&](int rows, int beside) { return static_cast<long long>((tokens + 32 * rows - 1) / (32 * rows)) * ((tiles + beside - 1) / beside); };
    // The largest tile that still gives most CUs a block: it reads x and the gate least often and splits a gate value for most rows.
    // us, by 2 x 4, 2 x 2, 2 x 1 and 1 x 1 (rows x tiles, four wavefronts): 8192 x 7168 x 256 (256 blocks of 2 x 4) 101, 141, 168, 207; 4096 x 7168 x 256 (256 of
    // 2 x 2) 87, 69, 84, 102; 3000 x 4096 x 256 (188 of 2 x 2) 49, 41, 50, 48; 2112 x 7168 x 160 (165 of 2 x 1) 80, 61, 41, 51; 5000 x 7168 x 32 (157 of 1 x 1) 81,
    // 67, 48, 35. Up to 2048 tokens eight wavefronts, whose shorter sums keep the error below the fp32 instruction's on sixteen.
    if (share_tiles(tokens, experts)) {  // (whose sums a layer's shares are)
      if (short_shares(depth)) DEW_LOGITS(1, 1, 16, 1, 2);
      else DEW_LOGITS(1, 1, 16, 1, 4);
    } else if (tokens <= 2048 && blocks(2, 1) >= 128) DEW_LOGITS(2, 1, 8, 1, 4);
    else if (tokens <= 2048) DEW_LOGITS(1, 1, 8, 1, 4);
    else if (tiles >= 4 && blocks(2, 4) >= 224) DEW_LOGITS(2, 4, 4, 1, 4);
    else if (tiles >= 2 && blocks(2, 2) >= 160) DEW_LOGITS(2, 2, 4, 2, 4);
    else if (blocks(2, 1) >= 160) DEW_LOGITS(2, 1, 4, 2, 4);
    else DEW_LOGITS(1, 1, 4, 2, 4);
#undef DEW_LOGITS
  }
  const dim3 grid((tokens + LT - 1) / LT, (experts + LE - 1) / LE);
  hipLaunchKernelGGL(router_logits_kernel, grid, dim3(256), 0, s, static_cast<const bf16_t*>(x), kernel, bias, logits, tokens, depth,
                     experts);
  return launched("router_logits_kernel");
}

extern "C" int dew_moe_group_offsets(const int32_t* sizes, int32_t experts, int32_t* offsets, void* stream) {
  using namespace dew;
  DEW_REQUIRE(sizes && offsets && experts >= 1, "dew_moe_group_offsets: sizes, offsets must not be null, experts %d", experts);
  hipLaunchKernelGGL(group_offsets_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), sizes, offsets, experts, 1);
  return launched("group_offsets_kernel");
}

extern "C" int dew_moe_block_offsets(const int32_t* blocks, int32_t groups, int32_t unit, int32_t* offsets, void* stream) {
  using namespace dew;
  DEW_REQUIRE(blocks && offsets && groups >= 1 && unit >= 1, "dew_moe_block_offsets: blocks, offsets must not be null, %d groups in units of %d", groups, unit);
  hipLaunchKernelGGL(group_offsets_kernel, dim3(1), dim3(64), 0, static_cast<hipStream_t>(stream), blocks, offsets, groups, unit);
  return launched("group_offsets_kernel");
}
