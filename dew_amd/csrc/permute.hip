// Dispatch bookkeeping: the stable counting sort of routed slots by expert id
// (reference src/dew/nn/moe.py:1101-1128 `_sorted_locally`: argsort(experts), bincount, order // k).
//
// Two stream-ordered launches, no global atomics, so the result is deterministic:
//   count   each block builds an LDS histogram of its run of slots
//   place   each block adds up all blocks' counts, those before its own apart, and scans them over the buckets (block 0 writes sizes and
//           offsets); then each wavefront ranks its slots, 64 at a time, among themselves with ballots (match-any over the id's bits),
//           adds the running count of earlier slots, and writes order[] / rows[]
// A block is sixteen wavefronts of one round each up to 64 blocks, of more beyond. (Four wavefronts of eight rounds, and a launch of one
// block between the two for the scan: 6666 slots of 64 experts 20 us, 11 here; 73 728 of 257
// 33 and 17.)
// Slots whose id is >= experts (a dropped slot's sentinel) sort last, in slot order, outside every group.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "sort.h"

namespace dew {

constexpr int kPermuteThreads = 256;
constexpr int kPermuteWaves = kPermuteThreads / 64;
constexpr int kSlotsPerBlock = 2048;  // what a caller's workspace is sized by: two counts for so many slots and a bucket
constexpr int kMostBlocks = 64;
constexpr int kMaxExperts = 1024;  // buckets = experts + 1 (the sentinel's) <= 1025 handled by loops

template <int THREADS>
__global__ __launch_bounds__(THREADS) void permute_count_kernel(PermuteParams p) {
  extern __shared__ int32_t hist[];  // [buckets]
  for (int b = threadIdx.x; b < p.buckets; b += THREADS) hist[b] = 0;
  __syncthreads();
  const int begin = blockIdx.x * p.slots_a_block;
  const int end = min(begin + p.slots_a_block, p.slots);
  for (int slot = begin + threadIdx.x; slot < end; slot += THREADS) atomicAdd(&hist[bucket_of(p, slot)], 1);
  __syncthreads();
  for (int b = threadIdx.x; b < p.buckets; b += THREADS) p.counts[static_cast<size_t>(blockIdx.x) * p.buckets + b] = hist[b];
}

template <int THREADS>
__global__ __launch_bounds__(THREADS) void permute_place_kernel(PermuteParams p) {
  constexpr int kWaves = THREADS / 64;
  extern __shared__ int32_t running[];  // [kWaves][buckets]: next free position per wave and bucket; then [buckets + 1] totals, [buckets] before
  int32_t *totals = running + kWaves * p.buckets, *before = totals + p.buckets + 1;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  for (int i = threadIdx.x; i < kWaves * p.buckets; i += THREADS) running[i] = 0;
  __syncthreads();
  int32_t* mine = running + wave * p.buckets;
  const int rounds = p.slots_a_block / THREADS, wave_begin = blockIdx.x * p.slots_a_block + wave * rounds * 64;
  for (int round = 0; round < rounds; ++round) {
    const int slot = wave_begin + round * 64 + lane;
    if (slot < p.slots) atomicAdd(&mine[bucket_of(p, slot)], 1);
  }
  for (int b = threadIdx.x; b < p.buckets; b += THREADS) {
    int total = 0, earlier = 0;
#pragma unroll 8
    for (int blk = 0; blk < p.blocks; ++blk) {
      const int count = p.counts[static_cast<size_t>(blk) * p.buckets + b];
      total += count;
      earlier += blk < static_cast<int>(blockIdx.x) ? count : 0;
    }
    totals[b] = total;
    before[b] = earlier;
  }
  __syncthreads();
  if (threadIdx.x < 64) scan_buckets(totals, p.buckets);
  __syncthreads();
  for (int b = threadIdx.x; b < p.buckets; b += THREADS) {
    const int start = totals[b];
    if (blockIdx.x == 0) {
      if (b < p.groups) {
        p.sizes[b] = totals[b + 1] - start;
        p.offsets[b] = start;
      } else {
        p.offsets[p.groups] = start;  // slots routed to a real expert
      }
    }
    int next = start + before[b];
    for (int w = 0; w < kWaves; ++w) {
      const int count = running[w * p.buckets + b];
      running[w * p.buckets + b] = next;
      next += count;
    }
  }
  __syncthreads();
  int bits = 1;
  while ((1 << bits) < p.buckets) ++bits;
  for (int round = 0; round < rounds; ++round) {
    const int slot = wave_begin + round * 64 + lane;
    place_round(p, slot, slot < p.slots ? bucket_of(p, slot) : p.buckets, bits, mine);
  }
}

template <int THREADS>
__global__ __launch_bounds__(THREADS) void permute_small_kernel(PermuteParams p) {
  extern __shared__ int32_t running[];  // [THREADS / 64][buckets] then [buckets + 1] totals
  sort_small<THREADS>(p, running, [&p](int slot) { return p.ids[slot]; });
}

}  // namespace dew

extern "C" size_t dew_moe_permute_workspace_bytes(int32_t slots, int32_t experts) {
  if (slots <= 0 || experts <= 0) return 256;
  const size_t blocks = (static_cast<size_t>(slots) + dew::kSlotsPerBlock - 1) / dew::kSlotsPerBlock;
  return 2 * blocks * (static_cast<size_t>(experts) + 1) * sizeof(int32_t) + 256;
}

namespace dew {

// Capacity dropping (`capacity_positions`, src/dew/nn/moe.py:832-855, applied at :914-919): a block a sequence. Each of a
// sequence's `slots` = length * top_k slots queues at its expert in slot order; a slot whose place in the queue is
// `capacity` or later is dropped: its id becomes `experts`, the sentinel that sorts last and outside every group.
// The place is the slot's rank among its sequence's slots of the same expert: the single block's counting sort above,
// without the scatter.
__global__ __launch_bounds__(kPermuteThreads) void capacity_admit_kernel(const int32_t* __restrict__ ids, int32_t* __restrict__ admitted,
                                                                         int slots, int experts, int capacity) {
  extern __shared__ int32_t running[];  // [kPermuteWaves][buckets]
  const int buckets = experts + 1;
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64;
  const int32_t* mine_ids = ids + static_cast<size_t>(blockIdx.x) * slots;
  int32_t* out = admitted + static_cast<size_t>(blockIdx.x) * slots;
  for (int i = threadIdx.x; i < kPermuteWaves * buckets; i += kPermuteThreads) running[i] = 0;
  __syncthreads();
  int32_t* mine = running + wave * buckets;
  const int segment = ((slots + kPermuteThreads - 1) / kPermuteThreads) * 64;  // contiguous slots per wavefront
  const int rounds = segment / 64, wave_begin = wave * segment;
  auto bucket_at = [&](int slot) {
    const int id = mine_ids[slot];
    return (id < 0 || id >= experts) ? experts : id;
  };
  for (int round = 0; round < rounds; ++round) {
    const int slot = wave_begin + round * 64 + lane;
    if (slot < slots) atomicAdd(&mine[bucket_at(slot)], 1);
  }
  __syncthreads();
  for (int b = threadIdx.x; b < buckets; b += kPermuteThreads) {  // each wavefront's first place in every queue
    int next = 0;
    for (int w = 0; w < kPermuteWaves; ++w) {
      const int count = running[w * buckets + b];
      running[w * buckets + b] = next;
      next += count;
    }
  }
  __syncthreads();
  int bits = 1;
  while ((1 << bits) < buckets) ++bits;
  for (int round = 0; round < rounds; ++round) {
    const int slot = wave_begin + round * 64 + lane;
    const bool valid = slot < slots;
    const int bucket = valid ? bucket_at(slot) : buckets;
    unsigned long long same = __ballot(valid);
    for (int bit = 0; bit < bits; ++bit) {
      const bool set = (bucket >> bit) & 1;
      const unsigned long long vote = __ballot(set);
      same &= set ? vote : ~vote;
    }
    const int rank = __popcll(same & ((1ull << lane) - 1ull));
    const int count = __popcll(same);
    int place = 0;
    if (valid) place = mine[bucket] + rank;
    __syncthreads();
    if (valid && rank == count - 1) mine[bucket] = place + 1;
    __syncthreads();
    if (valid) out[slot] = (bucket < experts && place < capacity) ? bucket : experts;
  }
}

// The sort's launches, given where the per-block counts live (the caller's workspace or the library's own
// scratch array): `counts` holds a bucket's count for every 1024 slots, 256-byte aligned.
static int permute_launches(const int32_t* indices, int32_t tokens, int32_t top_k, int32_t experts, int32_t shared_rows,
                            int32_t* sizes, int32_t* offsets, int32_t* order, int32_t* rows, int32_t* counts, hipStream_t s) {
  const int slots = tokens * top_k + shared_rows;
  PermuteParams p;
  p.ids = indices;
  p.sizes = sizes;
  p.offsets = offsets;
  p.order = order;
  p.rows = rows;
  p.slots = slots;
  p.routed = tokens * top_k;
  p.experts = experts;
  p.groups = experts + (shared_rows > 0 ? 1 : 0);
  p.top_k = top_k;
  p.buckets = p.groups + 1;
  p.counts = counts;
  // one block does it all faster than two launches
  const size_t wide_lds = sizeof(int32_t) * ((kSmallThreads / 64 + 1) * static_cast<size_t>(p.buckets) + 1);
  if (slots <= kSmallSlots && wide_lds <= 65536) {
    hipLaunchKernelGGL(permute_small_kernel<kSmallThreads>, dim3(1), dim3(kSmallThreads), wide_lds, s, p);
    return launched("permute_small_kernel");
  }
  if (slots <= kNarrowSmallSlots) {
    hipLaunchKernelGGL(permute_small_kernel<kPermuteThreads>, dim3(1), dim3(kPermuteThreads),
                       sizeof(int32_t) * ((kPermuteWaves + 1) * p.buckets + 1), s, p);
    return launched("permute_small_kernel");
  }
  auto launch = [&](auto threads) {
    constexpr int kThreads = decltype(threads)::value;
    const int whole = (slots + kMostBlocks * kThreads - 1) / (kMostBlocks * kThreads);
    p.slots_a_block = kThreads * std::max(whole, kSlotsPerBlock / 2 / kThreads);  // (half of what a workspace holds two counts for, at least)
    p.blocks = (slots + p.slots_a_block - 1) / p.slots_a_block;
    hipLaunchKernelGGL(permute_count_kernel<kThreads>, dim3(p.blocks), dim3(kThreads), sizeof(int32_t) * p.buckets, s, p);
    if (int rc = launched("permute_count_kernel")) return rc;
    hipLaunchKernelGGL(permute_place_kernel<kThreads>, dim3(p.blocks), dim3(kThreads), sizeof(int32_t) * ((kThreads / 64 + 2) * p.buckets + 1), s, p);
    return launched("permute_place_kernel");
  };
  if (sizeof(int32_t) * ((kSmallThreads / 64 + 2) * static_cast<size_t>(p.buckets) + 1) <= 65536) return launch(std::integral_constant<int, kSmallThreads>{});
  return launch(std::integral_constant<int, kPermuteThreads>{});
}

static int permute_arguments(const char* who, const int32_t* indices, int32_t tokens, int32_t top_k, int32_t experts,
                             const int32_t* sizes, const int32_t* offsets, const int32_t* order, const int32_t* rows) {
  DEW_REQUIRE(tokens >= 0 && top_k >= 1, "%s: tokens %d top_k %d", who, tokens, top_k);
  DEW_REQUIRE(experts >= 1 && experts <= kMaxExperts, "%s: experts %d (at most %d)", who, experts, kMaxExperts);
  DEW_REQUIRE(static_cast<int64_t>(tokens) * top_k < (1ll << 30), "%s: %d x %d slots overflow int32", who, tokens, top_k);
  DEW_REQUIRE(sizes && offsets, "%s: sizes and offsets must not be null", who);
  DEW_REQUIRE(tokens * top_k == 0 || (indices && order && rows), "%s: indices, order and rows must not be null", who);
  return DEW_MOE_OK;
}

// The library's own scratch for dew_moe_permute_static: the per-block counts of the two-launch sort.
// Every GPU the library runs on holds its own copy of the array until the process ends. The array's name is a
// host-side stand-in for it, not a device address: host code uses the address hipGetSymbolAddress returns for the
// current device, looked up once a device and kept.
constexpr size_t kStaticScratchBytes = DEW_MOE_PERMUTE_STATIC_BYTES;
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
static void* scratch_of_device[kMaxDevices];  // null until the device's first call
static std::mutex scratch_lookup;

static int static_scratch(const char* who, void** out) {
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxDevices)
    return fail(DEW_MOE_EDEVICE, "%s: no HIP device below %d is current", who, kMaxDevices);
  std::lock_guard<std::mutex> hold(scratch_lookup);
  if (scratch_of_device[device] == nullptr) {
    void* address = nullptr;
    const hipError_t status = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
    if (status != hipSuccess || address == nullptr)
      return fail(DEW_MOE_ELAUNCH, "%s: hipGetSymbolAddress of the scratch array on device %d: %s", who, device,
                  hipGetErrorString(status));
    scratch_of_device[device] = address;
  }
  *out = scratch_of_device[device];
  return DEW_MOE_OK;
}

}  // namespace dew

extern "C" int dew_moe_permute(const int32_t* indices, int32_t tokens, int32_t top_k, int32_t experts,
                               int32_t* sizes, int32_t* offsets, int32_t* order, int32_t* rows,
                               void* workspace, size_t workspace_bytes, void* stream) {
  using namespace dew;
  if (int rc = permute_arguments("dew_moe_permute", indices, tokens, top_k, experts, sizes, offsets, order, rows)) return rc;
  const int slots = tokens * top_k;
  DEW_REQUIRE(workspace && workspace_bytes >= dew_moe_permute_workspace_bytes(slots, experts),
              "dew_moe_permute: workspace of %zu bytes, need %zu", workspace_bytes,
              dew_moe_permute_workspace_bytes(slots, experts));
  const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255) & ~static_cast<uintptr_t>(255);
  return permute_launches(indices, tokens, top_k, experts, 0, sizes, offsets, order, rows, reinterpret_cast<int32_t*>(base),
                          static_cast<hipStream_t>(stream));
}

extern "C" int dew_moe_permute_shared(const int32_t* indices, int32_t tokens, int32_t top_k, int32_t experts, int32_t shared_rows,
                                      int32_t* sizes, int32_t* offsets, int32_t* order, int32_t* rows, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_permute_shared";
  if (int rc = permute_arguments(who, indices, tokens, top_k, experts, sizes, offsets, order, rows)) return rc;
  DEW_REQUIRE(shared_rows >= 0 && static_cast<int64_t>(tokens) * top_k + shared_rows < (1ll << 30) && experts < kMaxExperts,
              "%s: %d shared rows beside %d x %d slots, %d experts (a shared group needs one below %d)", who, shared_rows, tokens,
              top_k, experts, kMaxExperts);
  DEW_REQUIRE(shared_rows == 0 || (order && rows), "%s: order and rows must not be null", who);
  const int slots = tokens * top_k + shared_rows;
  const size_t need = dew_moe_permute_workspace_bytes(slots, experts + 1);
  DEW_REQUIRE(workspace && workspace_bytes >= need, "%s: workspace of %zu bytes, need %zu", who, workspace_bytes, need);
  const uintptr_t base = (reinterpret_cast<uintptr_t>(workspace) + 255) & ~static_cast<uintptr_t>(255);
  return permute_launches(indices, tokens, top_k, experts, shared_rows, sizes, offsets, order, rows, reinterpret_cast<int32_t*>(base),
                          static_cast<hipStream_t>(stream));
}

extern "C" int dew_moe_permute_static(const int32_t* indices, int32_t tokens, int32_t top_k, int32_t experts,
                                      int32_t* sizes, int32_t* offsets, int32_t* order, int32_t* rows, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_permute_static";
  if (int rc = permute_arguments(who, indices, tokens, top_k, experts, sizes, offsets, order, rows)) return rc;
  const size_t need = dew_moe_permute_workspace_bytes(tokens * top_k, experts);
  DEW_REQUIRE(need <= kStaticScratchBytes,
              "%s: %d slots over %d experts need %zu bytes of scratch, the library's own array holds %zu; use dew_moe_permute "
              "with a workspace", who, tokens * top_k, experts, need, kStaticScratchBytes);
  void* base = nullptr;
  if (int rc = static_scratch(who, &base)) return rc;
  // every int32 of the counts a call reads is written earlier in the same call: nothing to clear
  return permute_launches(indices, tokens, top_k, experts, 0, sizes, offsets, order, rows, static_cast<int32_t*>(base),
                          static_cast<hipStream_t>(stream));
}

extern "C" int dew_moe_capacity_admit(const int32_t* indices, int32_t sequences, int32_t length, int32_t top_k, int32_t experts,
                                      int32_t capacity, int32_t* admitted, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_capacity_admit";
  DEW_REQUIRE(sequences >= 0 && length >= 0 && top_k >= 1 && capacity >= 0, "%s: %d sequences of %d x %d slots, capacity %d", who,
              sequences, length, top_k, capacity);
  DEW_REQUIRE(experts >= 1 && experts <= kMaxExperts, "%s: experts %d (at most %d)", who, experts, kMaxExperts);
  DEW_REQUIRE(static_cast<int64_t>(sequences) * length * top_k < (1ll << 30), "%s: the slots overflow int32", who);
  if (sequences == 0 || length == 0) return DEW_MOE_OK;
  DEW_REQUIRE(indices && admitted, "%s: indices and admitted must not be null", who);
  hipLaunchKernelGGL(capacity_admit_kernel, dim3(sequences), dim3(kPermuteThreads), sizeof(int32_t) * kPermuteWaves * (experts + 1),
                     static_cast<hipStream_t>(stream), indices, admitted, length * top_k, experts, capacity);
  return launched("capacity_admit_kernel");
}
