// Grouped products of plain bf16 operands, read where they lie: a training step's forward product, its input's gradient and
// its kernel's gradient on unquantized matrices, whose weights are new at every step.
//
//   out[scatter[i], :] = x[gather[i], :] @ w[g(i)]      w [groups, depth, width], either way round
//   out[g] = x[rows of g]^T @ dy[rows of g]             x [rows, depth], dy [rows, width]
//
// The tiled launch of gemm.hip takes its weights in the matrix instruction's own order, which a bank has from its load on. A
// plain operand had to be brought to that order at every call: a pass over all weights each way (110 and 132 us of 347 for 16
// matrices of 2048 x 4096), two transposes for a kernel gradient. Here both operands go to the LDS as they lie in memory, and
// where an operand's rows run across the contraction its fragments are read transposed (ds_read_b64_tr_b16).
//
// A 256-thread block owns a BM x 256 tile and walks the contraction in steps of 32: operands global -> LDS by DMA into a ring of
// three stages (24 KB each at BM = 128, so that two blocks share a CU and one's start and end run under the other's loop; a
// contraction of a few hundred rows, a kernel gradient's, is otherwise half start and end), one barrier a step, wavefronts side
// by side along the columns; where such tiles are few, smaller ones. Sums are taken along the contraction in the tiled launch's order: the same bits.
// Launches that fill the chip with 256 x 256 tiles take those (wide.hip); rows that are gathered or scattered stay here. For them, from
// groups of some thousands of rows on, the weights' pass is the smaller price: an operand whose rows run along the contraction
// gives a step 64 bytes of each of its cache lines, so that K-major matrices cost 10 to 17 % more than natural ones, and the tiled
// launch's 256-row tiles fetch half as much. The caller (gemm.py, with the sizes measured) brings such matrices to order first.
#include <mutex>

#include "dense.h"
#include "gemm.h"

namespace dew {

constexpr int kDepthStep = 32, kRing = 3, kBlock = 256;

__device__ const u32x4_t zero_rows[1] = {u32x4_t{0, 0, 0, 0}};  // what a step reads past a group's last row

__device__ __forceinline__ uint32_t lds_address(const void* p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p));
}

template <int N>
__device__ __forceinline__ void pinned(bf16x8_t (&fragments)[N]) {  // used no earlier than here
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(fragments[i]));
}

// A staged operand. kAcross false: its rows run along the contraction, EXTENT rows of 32 depths (64 bytes, four 16-byte chunks,
// chunk index xor-ed with row / 4 mod 4: the rows a pass of ds_read_b128 serves then lie in different banks). kAcross true: 32
// rows of EXTENT columns, in units of 32 columns (64 bytes) whose index is xor-ed with the row mod 4: the four rows that 16
// lanes of a transposed read take lie in different banks.
template <int EXTENT, bool kAcross>
struct Staged {
  static constexpr int kBytes = EXTENT * kDepthStep * 2;
  static constexpr int kLoads = kBytes / (kBlock * 16);  // 1 KiB DMA loads a wavefront makes
  static constexpr int kRowChunks = kAcross ? EXTENT / 8 : kDepthStep / 8;
  // the row and the chunk of it that lane `lane` of load `load` of wavefront `wave` fetches
  static __device__ __forceinline__ int row(int wave, int load, int lane) { return ((wave * kLoads + load) * 64 + lane) / kRowChunks; }
  static __device__ __forceinline__ int chunk(int row, int lane) {
    const int place = lane % kRowChunks;
    return kAcross ? ((place / 4) ^ (row & 3)) * 4 + place % 4 : place ^ ((row >> 2) & 3);
  }
  // the fragment of rows (columns) 32 tile .. + 31 over depths 16 slice .. + 15: lane l holds row l % 32, depths 8 (l / 32) .. + 7
  template <int slice>
  static __device__ __forceinline__ bf16x8_t fragment(const uint8_t* stage, int tile, int lane) {
    if constexpr (!kAcross) {
      const int row = 32 * tile + lane % 32;
      return __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(stage + row * 64 + (((2 * slice + lane / 32) ^ ((row >> 2) & 3)) * 16)));
    } else {
      // (two reads of four depths each, 16 lanes a group: lane j of a group addresses depth j / 4, columns 4 (j % 4) .., and gets
      // column j over the four depths)
      const int piece = lane % 16;
      const uint32_t at = lds_address(stage) + (8 * (lane / 32) + piece / 4) * (EXTENT * 2) + ((tile ^ (piece / 4)) * 64) + (lane / 16 % 2) * 32 + (piece % 4) * 8;
      typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
      u32x2_t low, high;
      // Written out, with the wait for them stated where they are first used (`arrived`): the compiler takes any LDS-DMA load in
      // flight for a write these reads may depend on, and drains the memory pipeline in front of every step's first one.
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(low) : "v"(at), "n"(slice * 16 * EXTENT * 2));
      asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(high) : "v"(at), "n"((slice * 16 + 4) * EXTENT * 2));
      return __builtin_bit_cast(bf16x8_t, u32x4_t{low[0], low[1], high[0], high[1]});
    }
  }
};

// kAAcross: a kernel gradient (both operands' rows run across the contraction, which is a group's rows). kBAcross: w [.., depth, width].
template <int BM, int kColumns, bool kAAcross, bool kBAcross, bool kOutF32>
__global__ __launch_bounds__(kBlock, 2) void dense_kernel(DenseParams p) {
  using A = Staged<BM, kAAcross>;
  using B = Staged<kColumns, kBAcross>;
  static_assert(!kAAcross || kBAcross, "a kernel gradient's operands both run across");
  constexpr int kStageBytes = A::kBytes + B::kBytes, kLoads = A::kLoads + B::kLoads;
  constexpr int TI = BM / 32, TJ = kColumns / 128;
  extern __shared__ uint8_t stages[];  // the ring; then the finished tile's rows
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);

  // ---- block -> tile, as the tiled launch maps it: chunks of group_m row tiles x 8 strips, dealt round-robin to the XCDs ----
  const int strips = (p.outer_n + kColumns - 1) / kColumns, total = p.m_tiles * strips, chunk_tiles = 8 * p.group_m;
  const int local = blockIdx.x / 8, order = ((local / chunk_tiles) * 8 + blockIdx.x % 8) * chunk_tiles + local % chunk_tiles;
  if (order >= total) return;
  const int band = order / (p.group_m * strips), band_tiles = min(p.group_m, p.m_tiles - band * p.group_m), within = order % (p.group_m * strips);
  const int m_tile = band * p.group_m + within % band_tiles, n0 = (within / band_tiles) * kColumns;

  // ---- the tile's group and rows (every wavefront scans the groups for itself, 64 a round) ----
  auto scanned = [lane](int value) {
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
      const int other = __shfl_up(value, offset, 64);
      if (lane >= offset) value += other;
    }
    return value;
  };
  auto size_of = [&p](int g) { return g >= p.groups ? 0 : p.sizes ? max(p.sizes[g], 0) : max(p.offsets[g + 1] - p.offsets[g], 0); };
  int group = -1, row0 = 0, end = 0, m0 = 0, carried = 0, carried_rows = 0;
  if constexpr (kAAcross) {
    const int tiles = (p.outer_m + BM - 1) / BM;
    group = m_tile / tiles;
    m0 = (m_tile % tiles) * BM;
    if (p.sizes) {
      for (int base = 0; base <= group; base += 64) {
        const int size = size_of(base + lane), rows = scanned(size), at = min(group - base, 63);
        if (group < base + 64) {
          row0 = carried_rows + __builtin_amdgcn_readlane(rows - size, at);
          end = carried_rows + __builtin_amdgcn_readlane(rows, at);
        }
        carried_rows += __builtin_amdgcn_readlane(rows, 63);
      }
    } else {
      row0 = __builtin_amdgcn_readfirstlane(p.offsets[group]);
      end = __builtin_amdgcn_readfirstlane(p.offsets[group + 1]);
    }
    row0 = min(max(row0, 0), p.rows);
    end = min(max(end, row0), p.rows);
  } else {
    for (int base = 0; base < p.groups && group < 0; base += 64) {
      const int size = size_of(base + lane);
      int start = 0;
      if (p.sizes) {
        const int rows = scanned(size);
        start = carried_rows + rows - size;
        carried_rows += __builtin_amdgcn_readlane(rows, 63);
      } else if (base + lane < p.groups) {
        start = p.offsets[base + lane];
      }
      const int tiles = (size + BM - 1) / BM, inclusive = scanned(tiles), first = carried + inclusive - tiles;
      const unsigned long long hit = __ballot(m_tile >= first && m_tile < first + tiles);
      if (hit != 0ull) {
        const int owner = __builtin_ctzll(hit);
        group = base + owner;
        row0 = __builtin_amdgcn_readlane(start + (m_tile - first) * BM, owner);
        end = __builtin_amdgcn_readlane(start + size, owner);
      }
      carried += __builtin_amdgcn_readlane(inclusive, 63);
    }
    if (group < 0) {  // past the last tile: zero the rows of no group
      const int held = p.sizes ? carried_rows : p.offsets[p.groups];
      const int begin = held + (m_tile - carried) * BM, stop = min(begin + BM, p.rows);
      for (int item = threadIdx.x; item < (stop - begin) * (kColumns / 8); item += kBlock) {
        const int sorted = begin + item / (kColumns / 8), column = n0 + item % (kColumns / 8) * 8;
        const int row = p.scatter ? p.scatter[sorted] : sorted;
        if (column < p.outer_n) *reinterpret_cast<u32x4_t*>(static_cast<bf16_t*>(p.out) + static_cast<size_t>(row) * p.outer_n + column) = u32x4_t{0, 0, 0, 0};
      }
      return;
    }
  }
  const int valid_rows = kAAcross ? min(BM, p.outer_m - m0) : min(BM, end - row0);
  const int depth = kAAcross ? end - row0 : p.inner, steps = (depth + kDepthStep - 1) / kDepthStep;

  // ---- where a lane's loads start; they move on by a uniform stride a step ----
  const bf16_t *a_src[A::kLoads], *b_src[B::kLoads];
  int a_row[A::kLoads], b_row[B::kLoads];
#pragma unroll
  for (int i = 0; i < A::kLoads; ++i) {
    a_row[i] = A::row(wave, i, lane);
    const int chunk = A::chunk(a_row[i], lane);
    if constexpr (kAAcross) {
      a_src[i] = p.a + static_cast<size_t>(row0 + a_row[i]) * p.outer_m + min(m0 + 8 * chunk, p.outer_m - 8);
    } else {
      const int sorted = row0 + min(a_row[i], valid_rows - 1);
      a_src[i] = p.a + static_cast<size_t>(p.gather ? p.gather[sorted] : sorted) * p.inner + 8 * chunk;
    }
  }
#pragma unroll
  for (int i = 0; i < B::kLoads; ++i) {
    b_row[i] = B::row(wave, i, lane);
    const int chunk = B::chunk(b_row[i], lane);
    if constexpr (kAAcross) {
      b_src[i] = p.b + static_cast<size_t>(row0 + b_row[i]) * p.outer_n + min(n0 + 8 * chunk, p.outer_n - 8);
    } else {
      const bf16_t* matrix = p.b + static_cast<size_t>(group) * p.inner * p.outer_n;
      b_src[i] = kBAcross ? matrix + static_cast<size_t>(b_row[i]) * p.outer_n + min(n0 + 8 * chunk, p.outer_n - 8)
                          : matrix + static_cast<size_t>(min(n0 + b_row[i], p.outer_n - 1)) * p.inner + 8 * chunk;
    }
  }
  const size_t a_stride = kAAcross ? static_cast<size_t>(kDepthStep) * p.outer_m : kDepthStep;
  const size_t b_stride = kBAcross ? static_cast<size_t>(kDepthStep) * p.outer_n : kDepthStep;
  auto load = [&](int stage, int step) __attribute__((always_inline)) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(3))) void* lds_t;
    uint8_t* to = stages + stage * kStageBytes;
#pragma unroll
    for (int i = 0; i < A::kLoads; ++i) {
      const bf16_t* from = a_src[i] + step * a_stride;
      if (kAAcross && step * kDepthStep + a_row[i] >= depth) from = reinterpret_cast<const bf16_t*>(zero_rows);
      __builtin_amdgcn_global_load_lds(from, (lds_t)(to + (wave * A::kLoads + i) * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < B::kLoads; ++i) {
      const bf16_t* from = b_src[i] + step * b_stride;
      if (kAAcross && step * kDepthStep + b_row[i] >= depth) from = reinterpret_cast<const bf16_t*>(zero_rows);
      __builtin_amdgcn_global_load_lds(from, (lds_t)(to + A::kBytes + (wave * B::kLoads + i) * 1024), 16, 0, 0);
    }
#endif
  };

  f32x16_t acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int q = 0; q < 16; ++q) acc[i][j][q] = 0.0f;
  bf16x8_t a_frag[2][TI], b_frag[2][TJ];
  auto fetch = [&](int stage, auto slice) __attribute__((always_inline)) {
    const uint8_t* from = stages + stage * kStageBytes;
#pragma unroll
    for (int j = 0; j < TJ; ++j) b_frag[slice.value][j] = B::template fragment<decltype(slice)::value>(from + A::kBytes, TJ * wave + j, lane);
#pragma unroll
    for (int i = 0; i < TI; ++i) a_frag[slice.value][i] = A::template fragment<decltype(slice)::value>(from, i, lane);
  };
  // the fragments of `slice` are there once this wavefront's LDS reads are (the wait stands in front of this)
  auto arrived = [&](auto slice) __attribute__((always_inline)) {
    pinned(a_frag[slice.value]);
    pinned(b_frag[slice.value]);
  };
  auto multiply = [&](auto slice) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int j = 0; j < TJ; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a_frag[slice.value][i], b_frag[slice.value][j], acc[i][j], 0, 0, 0);
  };
  constexpr std::integral_constant<int, 0> first{};
  constexpr std::integral_constant<int, 1> second{};
  // vmcnt(n), lgkmcnt(0): everything but this step's own loads has landed, and this wavefront's reads are done
  constexpr int kLanded = (kLoads & 0xF) | (7 << 4) | ((kLoads >> 4) << 14);
  constexpr int kAll = 7 << 4;
  constexpr int kReads = 0xF | (7 << 4) | (3 << 14);  // lgkmcnt(0) alone
  if (steps > 0) {
    load(0, 0);
    load(1, min(1, steps - 1));
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(kLanded);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    fetch(0, first);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(kReads);
    arrived(first);
    __builtin_amdgcn_sched_barrier(0);
    int current = 0;
    __builtin_amdgcn_s_setprio(3);  // a wavefront in its loop goes ahead of one in its start or end (the CU's other block)
    for (int step = 0; step < steps; ++step) {
      const int next = current == kRing - 1 ? 0 : current + 1, fill = next == kRing - 1 ? 0 : next + 1;
      fetch(current, second);
      load(fill, min(step + 2, steps - 1));
      multiply(first);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_waitcnt(kLanded);
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      arrived(second);
      fetch(next, first);
      multiply(second);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_waitcnt(kReads);  // (long back: eight matrix instructions were issued behind them)
      arrived(first);
      __builtin_amdgcn_sched_barrier(0);
      current = next;
    }
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_s_waitcnt(kAll);  // the clamped last loads still target the LDS
  }
  __builtin_amdgcn_s_barrier();  // every wavefront has read its last fragments: the ring is free

  // ---- epilogue: acc[i][j][q] is row 8 (q / 4) + 4 (lane / 32) + q % 4, column lane % 32 of its 32 x 32 tile ----
  float factor = 1.0f;
  if constexpr (kAAcross) factor = (p.factor0 ? *p.factor0 : 1.0f) * (p.factor1 ? *p.factor1 : 1.0f);
  if constexpr (kOutF32) {
    float* out = static_cast<float*>(p.out) + (static_cast<size_t>(group) * p.outer_m + m0) * p.outer_n;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int q = 0; q < 16; ++q) {
        const int row = 32 * i + 8 * (q / 4) + 4 * (lane / 32) + q % 4;
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          const int column = n0 + 32 * (TJ * wave + j) + lane % 32;
          if (row < valid_rows && column < p.outer_n) out[static_cast<size_t>(row) * p.outer_n + column] = acc[i][j][q] * factor;
        }
      }
    return;
  } else {
    // each pair of lanes swaps one value so that a lane holds two neighbouring columns; rows leave the LDS 16 bytes a lane
    constexpr int kRowDwords = kColumns / 2 + 4, kRowPieces = kColumns / 8;
    uint32_t* staged = reinterpret_cast<uint32_t*>(stages);
    const bool odd = lane & 1;
    const uint32_t select = odd ? 0x03020706u : 0x05040100u;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int q = 0; q < 16; q += 2) {
        const int row = 32 * i + 8 * (q / 4) + 4 * (lane / 32) + q % 4 + (odd ? 1 : 0);
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
          const uint32_t mine = pack_bf16(acc[i][j][q] * factor, acc[i][j][q + 1] * factor);
          const uint32_t other = __builtin_amdgcn_mov_dpp(mine, 0xB1, 0xF, 0xF, true);
          staged[row * kRowDwords + (32 * (TJ * wave + j) + (lane % 32 & ~1)) / 2] = __builtin_amdgcn_perm(other, mine, select);
        }
      }
    __syncthreads();
    bf16_t* out = static_cast<bf16_t*>(p.out);
#pragma unroll 4
    for (int item = threadIdx.x; item < BM * kRowPieces; item += kBlock) {
      const int row = item / kRowPieces, column = n0 + item % kRowPieces * 8;
      if (row >= valid_rows || column >= p.outer_n) continue;
      const size_t to = kAAcross ? static_cast<size_t>(group) * p.outer_m + m0 + row : p.scatter ? p.scatter[row0 + row] : row0 + row;
      *reinterpret_cast<u32x4_t*>(out + to * p.outer_n + column) = *reinterpret_cast<const u32x4_t*>(staged + row * kRowDwords + (item % kRowPieces) * 4);
    }
  }
}

template <int BM, int kColumns, bool kAAcross, bool kBAcross, bool kOutF32>
static int launch_dense(const char* who, DenseParams p, hipStream_t stream) {
  constexpr size_t kRingBytes = kRing * (Staged<BM, kAAcross>::kBytes + Staged<kColumns, kBAcross>::kBytes);
  constexpr size_t kStagedBytes = static_cast<size_t>(BM) * (kColumns / 2 + 4) * 4;
  constexpr size_t kShared = kRingBytes > kStagedBytes ? kRingBytes : kStagedBytes;
  auto kernel = dense_kernel<BM, kColumns, kAAcross, kBAcross, kOutF32>;
  static std::once_flag configured;  // dynamic LDS above 64 KiB must be opted into once per kernel
  static hipError_t reserved = hipSuccess;
  std::call_once(configured, [&] {
    reserved = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(kShared));
  });
  if (reserved != hipSuccess) return fail(DEW_MOE_ELAUNCH, "%s: cannot reserve %zu bytes of LDS", who, kShared);
  // every group of rows may end in a partial tile, and the zeroed tail may add one more
  p.m_tiles = kAAcross ? p.groups * ((p.outer_m + BM - 1) / BM) : (p.rows + BM - 1) / BM + p.groups + 1;
  p.group_m = 4;
  const long long total = static_cast<long long>(p.m_tiles) * ((p.outer_n + kColumns - 1) / kColumns);
  const int round = 64 * p.group_m;
  DEW_REQUIRE(total + round < (1ll << 31), "%s: %lld tiles", who, total);
  const int blocks = static_cast<int>((total + round - 1) / round * round);
  hipLaunchKernelGGL(kernel, dim3(blocks), dim3(kBlock), kShared, stream, p);
  return launched(who);
}

constexpr int kFewTiles = 128;
static bool few_tiles(int rows, int groups, int width) {  // about so many of 128 x 256, the groups' last ones half empty
  return (rows / 128 + groups / 2 + 1) * static_cast<long long>((width + 255) / 256) <= kFewTiles;
}

// Whether a product takes 256 x 256 tiles (wide.hip), on groups of at least about half a tile's rows (of 64 to 97 rows 0.82 to 0.98 times as fast):
//  * whole tiles, but where a first round of them is half empty: from 146 on, K-major matrices, which the tiles below read half a cache line at a
//    step, from 129;
//  * quarters, up to one a block, and up to two where the walk is long enough to hide two starts.
// us, the tiles below and here, natural order and K-major. Whole: 4608 rows of 1 x 1024 x 2048, 148 tiles, 32.1 and 25.5 (natural), 4096 of 1 x 4096 x 2048,
// 132, 67.5 and 80.3, 75.6 and 79.9. One quarter a block: 1024 of 1 x 4096 x 4096 63 and 33, 70 and 33, 3127 of 1 x 3584 x 1152, 225 quarters of 65 tiles, 40 and 28,
// 48 and 28. Two: 1536 of 1 x 4096 x 4096 64 and 56, 70 and 54, 2560 of 4 x 1024 x 2048 24 and 19 (K-major). Furthest off: 2205 of 14 x 4928 x 1184, 64 and 76, 64 and 59.
static bool wide_product(int rows, int groups, int depth, int width, bool kmajor) {
  const double tiles = product_tiles(rows, groups, width);
  const int quarters = depth >= (kmajor ? 1024 : 2048) ? 128 : 64;
  return wide_extents(groups, depth, width) && rows / groups >= 112 && (tiles + (groups > 1 ? kGuessed : 0) <= quarters || tiles >= (kmajor ? 129 : 146));
}

// The same of a kernel's gradient, whose tiles are known; groups of fewer than 256 rows, four steps, are all start and end either way:
//  * up to 128 tiles, one quarter a block on groups of 512 rows and more, two where the walk is long (a launch takes two from 1024 rows on; of 1024 to
//    2048 in several groups they are 0.8 to 1.2 times the time, 1.0 in the mean of 152 shapes, of more 0.93, in one group 0.87);
//  * whole ones from over half a round on, and from 1.1, before which groups of fewer than 512 rows lose.
// us, the tiles below and here. One quarter a block: 4096 rows of 2 x 512 x 2048 28.1 and 15.9, 2340 of 3 x 576 x 1952, 72 tiles, 14.3 and 11.1; 813 of 3 x 640 x
// 2176 10.7 and 13.3. Two: 2048 of 1 x 2048 x 4096 41.0 and 35.9, 11 129 of 1 x 2048 x 2432 179 and 139, 16 329 of 2 x 1664 x 1344 137 and 111; 3531 of 4 x 960 x 1368
// 21.2 and 24.0. Whole: 144 tiles of 512 rows 20.1 and 18.4, of 8192 207 and 169. Behind a round: 3364 of 1 x 2432 x 6672, 270 tiles, 141 and 106; 2221 of 5
// x 3200 x 800, 260, 19.9 and 24.3.
static bool wide_gradient(int rows, int groups, int depth, int width) {
  const double tiles = gradient_tiles(groups, depth, width), quarters = gradient_quarters(groups, depth, width);
  if (!wide_extents(groups, depth, width) || rows / groups < 256) return false;
  if (tiles <= 128) return quarters <= 256 ? rows / groups >= 512 : quarters >= 280 && rows / groups >= (groups == 1 ? 1024 : 2048);
  return tiles >= 282 || (tiles >= 141 && tiles <= 256) || (tiles > 256 && rows / groups >= 512);
}

}  // namespace dew

extern "C" int dew_moe_dense_gemm(const void* x, const int32_t* gather, const int32_t* offsets, const int32_t* group_sizes, const void* w,
                                  int32_t kmajor, const int32_t* scatter, void* out, int32_t rows, int32_t groups, int32_t depth,
                                  int32_t width, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_dense_gemm";
  DEW_REQUIRE(rows >= 0 && groups >= 1 && groups <= 4096, "%s: %d rows in %d groups", who, rows, groups);
  DEW_REQUIRE(depth >= 64 && depth % 64 == 0 && width >= 32 && width % 32 == 0, "%s: matrices [%d, %d]: depths are whole 64s, widths whole 32s", who,
              depth, width);
  if (rows == 0) return DEW_MOE_OK;
  DEW_REQUIRE((offsets != nullptr) != (group_sizes != nullptr), "%s: the groups come as offsets [E + 1] or as group_sizes [E], one of them", who);
  DEW_REQUIRE(x && w && out && aligned16(x) && aligned16(w) && aligned16(out), "%s: x, w and out must not be null and must be 16-byte aligned", who);
  DenseParams p{};
  p.a = static_cast<const bf16_t*>(x);
  p.b = static_cast<const bf16_t*>(w);
  p.gather = gather;
  p.scatter = scatter;
  p.offsets = offsets;
  p.sizes = group_sizes;
  p.out = out;
  p.groups = groups;
  p.rows = rows;
  p.inner = depth;
  p.outer_n = width;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (!gather && !scatter && wide_product(rows, groups, depth, width, kmajor != 0)) return launch_wide(who, p, false, kmajor != 0, false, s);
  // Where 128 x 256 tiles would leave half of the chip idle, a quarter of one each: a block's walk down the contraction is what the
  // launch takes then (us: 640 rows of 4 x 1024 x 2048 22 -> 14 and its input's gradient 38 -> 22, 1000 of 8 x 3072 x 1024 57 -> 31, 3000
  // of 8 x 2048 x 1024, 112 tiles, 42 -> 32; at 160 to 220 tiles 3 to 30 % slower).
  if (few_tiles(rows, groups, width))
    return kmajor ? launch_dense<64, 128, false, false, false>(who, p, s) : launch_dense<64, 128, false, true, false>(who, p, s);
  if (rows / groups <= 64)
    return kmajor ? launch_dense<64, 256, false, false, false>(who, p, s) : launch_dense<64, 256, false, true, false>(who, p, s);
  return kmajor ? launch_dense<128, 256, false, false, false>(who, p, s) : launch_dense<128, 256, false, true, false>(who, p, s);
}

extern "C" int dew_moe_dense_gradient(const void* lhs, const void* rhs, const int32_t* offsets, const int32_t* group_sizes, const float* lhs_scale,
                                      const float* rhs_scale, void* out, int32_t out_is_f32, int32_t rows, int32_t groups, int32_t depth, int32_t width, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_dense_gradient";
  DEW_REQUIRE(rows >= 0 && groups >= 1 && groups <= 4096, "%s: %d rows in %d groups", who, rows, groups);
  DEW_REQUIRE(depth >= 8 && depth % 8 == 0 && width >= 8 && width % 8 == 0, "%s: a gradient [%d, %d]: extents are whole 8s", who, depth, width);
  DEW_REQUIRE((offsets != nullptr) != (group_sizes != nullptr), "%s: the groups come as offsets [E + 1] or as group_sizes [E], one of them", who);
  DEW_REQUIRE(out && aligned16(out) && (rows == 0 || (lhs && rhs)) && aligned16(lhs) && aligned16(rhs),
              "%s: out and the operands must not be null; operands and out are 16-byte aligned", who);
  DenseParams p{};
  p.a = static_cast<const bf16_t*>(lhs);
  p.b = static_cast<const bf16_t*>(rhs);
  p.offsets = offsets;
  p.sizes = group_sizes;
  p.out = out;
  p.factor0 = lhs_scale;
  p.factor1 = rhs_scale;
  p.groups = groups;
  p.rows = rows;
  p.outer_m = depth;
  p.outer_n = width;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  if (wide_gradient(rows, groups, depth, width)) return launch_wide(who, p, true, false, out_is_f32 != 0, s);
  // (few tiles: half as wide, 4 groups of 4096 rows, 1024 x 1024, 128 tiles, 96 -> 77 us; 3333 rows, 2 x 640 x 4096, 39 -> 34; at 512
  // tiles 8 to 10 % slower)
  if (static_cast<long long>(groups) * ((depth + 127) / 128) * ((width + 255) / 256) <= 2 * kFewTiles)
    return out_is_f32 ? launch_dense<128, 128, true, true, true>(who, p, s) : launch_dense<128, 128, true, true, false>(who, p, s);
  return out_is_f32 ? launch_dense<128, 256, true, true, true>(who, p, s) : launch_dense<128, 256, true, true, false>(who, p, s);
}
