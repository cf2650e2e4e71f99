// The stable counting sort of routed slots by expert as one block runs it, shared by the sort's own launch and by the
// router's launch of a decode step.
#pragma once

#include "common.h"

namespace dew {

// offsets[0] = 0, offsets[e + 1] = offsets[e] + unit * sizes[e] by one wavefront, 64 sizes a round, the next round's asked for
// while this one's are added up. (One lane walking the sizes took a memory round trip each few of them: 5 us for 16 groups.)
__device__ __forceinline__ void write_group_offsets(const int32_t* __restrict__ sizes, int32_t* __restrict__ offsets, int experts, int unit) {
  const int lane = threadIdx.x % 64;
  int running = 0, next = lane < experts ? sizes[lane] : 0;
  if (lane == 0) offsets[0] = 0;
  for (int base = 0; base < experts; base += 64) {
    int through = unit * next;
    next = base + 64 + lane < experts ? sizes[base + 64 + lane] : 0;
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
      const int below = __shfl_up(through, offset, 64);
      if (lane >= offset) through += below;
    }
    if (base + lane < experts) offsets[base + lane + 1] = running + through;
    running += __shfl(through, 63, 64);
  }
}

struct PermuteParams {
  const int32_t* ids;  // [slots]
  int32_t* sizes;      // [experts]
  int32_t* offsets;    // [experts + 1]
  int32_t* order;      // [slots]
  int32_t* rows;       // [slots]
  int32_t* counts;     // workspace [blocks][buckets]
  // `slots` sorted positions: the `routed` = tokens * top_k slots of `ids`, then `slots - routed` rows that every token
  // sends to one always-on (shared) expert, which sorts as group `experts`. `groups` = the groups written (experts, or
  // experts + 1 with a shared one); bucket `groups` collects the dropped slots (an id outside [0, experts)), last.
  int slots, routed, experts, groups, top_k, blocks, buckets, slots_a_block;
};

__device__ __forceinline__ int bucket_of_id(const PermuteParams& p, int id) { return (id < 0 || id >= p.experts) ? p.groups : id; }

__device__ __forceinline__ int bucket_of(const PermuteParams& p, int slot) {
  return slot >= p.routed ? p.experts /* a shared expert's row */ : bucket_of_id(p, p.ids[slot]);
}

// The row of the activations a slot reads: its token, or for a shared expert's row the token it is.
__device__ __forceinline__ int row_of(const PermuteParams& p, int slot) {
  return slot < p.routed ? slot / p.top_k : slot - p.routed;
}

// The exclusive scan of `buckets` totals by one wavefront, 64 a round; totals[buckets] is their sum.
__device__ __forceinline__ void scan_buckets(int32_t* totals, int buckets) {
  const int lane = threadIdx.x % 64;
  int carried = 0;
  for (int base = 0; base < buckets; base += 64) {
    const int b = base + lane;
    const int size = b < buckets ? totals[b] : 0;
    int inclusive = size;
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
      const int other = __shfl_up(inclusive, offset, 64);
      if (lane >= offset) inclusive += other;
    }
    if (b < buckets) totals[b] = carried + inclusive - size;
    carried += __shfl(inclusive, 63, 64);
  }
  if (lane == 0) totals[buckets] = carried;
}

// A wavefront's 64 slots to their places: ranked among themselves, behind the wavefront's running positions `mine`. A lane without a slot
// has bucket `buckets`.
__device__ __forceinline__ void place_round(const PermuteParams& p, int slot, int bucket, int bits, int32_t* mine) {
  const int lane = threadIdx.x % 64;
  const bool valid = bucket < p.buckets;
  unsigned long long same = __ballot(valid);
  for (int bit = 0; bit < bits; ++bit) {
    const bool set = (bucket >> bit) & 1;
    const unsigned long long vote = __ballot(set);
    same &= set ? vote : ~vote;
  }
  const int rank = __popcll(same & ((1ull << lane) - 1ull));
  const int count = __popcll(same);
  int position = 0;
  if (valid) position = mine[bucket] + rank;
  // The running positions are the wavefront's own (no other wavefront touches them), so no block barrier is needed,
  // only an order between this wavefront's lanes: every lane's read above before the one lane's write below, and that
  // write before the next round's reads. The wavefront-scope fences state that order to the compiler and the memory
  // model (they cost no instruction: a wavefront's LDS operations are issued and served in order).
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (valid && rank == count - 1) mine[bucket] = position + 1;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (valid) {
    p.order[position] = slot;
    p.rows[position] = row_of(p, slot);
  }
}

// The whole sort in one block for at most kSmallSlots slots (a decode step, a small prefill): the block
// counts, scans and scatters, each wavefront a contiguous run of the slots, with the LDS histogram as the only
// intermediate.
// Measured under graph replay, sixteen wavefronts, of 8, 64 and 256 experts, and the two launches over many blocks beside it: 2048 slots 4.6,
// 5.4 and 6.6 us (four wavefronts: 7.9 to 10.0) and 6.1, 6.8 and 7.9; 4096 slots 6.3, 7.2 and 8.8 and 6.7, 7.7 and 8.8; 5120 slots 7.4, 8.4 and
// 10.3 and 6.7, 8.0 and 9.1; 8192 slots 10.0, 11.1 and 14.2 and 6.3, 7.1 and 8.6.
constexpr int kSmallSlots = 4096;      // where the two meet
constexpr int kSmallThreads = 1024;    // sixteen wavefronts, where their counters fit the LDS a launch may take unasked
constexpr int kNarrowSmallSlots = 2048;  // the four-wavefront form's reach, for more buckets than that
// `running`: LDS, [THREADS / 64][buckets] then [buckets + 1] totals. `id_of(slot)`: a routed slot's expert.
template <int THREADS, class IdOf>
__device__ __forceinline__ void sort_small(const PermuteParams& p, int32_t* running, IdOf id_of) {
  constexpr int kWaves = THREADS / 64;
  int32_t* totals = running + kWaves * p.buckets;
  const int lane = threadIdx.x % 64;
  const int wave = threadIdx.x / 64;
  for (int i = threadIdx.x; i < kWaves * p.buckets; i += THREADS) running[i] = 0;
  __syncthreads();
  int32_t* mine = running + wave * p.buckets;
  const int segment = ((p.slots + THREADS - 1) / THREADS) * 64;  // contiguous slots per wavefront
  const int rounds = segment / 64;
  const int wave_begin = wave * segment;
  // a lane's buckets stay in registers between the count and the scatter (one round trip to the indices, not two)
  constexpr int kMaxRounds = (THREADS == kSmallThreads ? kSmallSlots : kNarrowSmallSlots) / THREADS;
  int kept[kMaxRounds];
#pragma unroll
  for (int round = 0; round < kMaxRounds; ++round) {
    const int slot = wave_begin + round * 64 + lane;
    kept[round] = (round < rounds && slot < p.slots) ? (slot < p.routed ? bucket_of_id(p, id_of(slot)) : p.experts) : p.buckets;
  }
#pragma unroll
  for (int round = 0; round < kMaxRounds; ++round)
    if (kept[round] < p.buckets) atomicAdd(&mine[kept[round]], 1);
  __syncthreads();
  for (int b = threadIdx.x; b < p.buckets; b += THREADS) {
    int sum = 0;
    for (int w = 0; w < kWaves; ++w) sum += running[w * p.buckets + b];
    totals[b] = sum;
  }
  __syncthreads();
  if (threadIdx.x < 64) scan_buckets(totals, p.buckets);
  __syncthreads();
  for (int b = threadIdx.x; b < p.buckets; b += THREADS) {
    const int start = totals[b];
    if (b < p.groups) {
      p.sizes[b] = totals[b + 1] - start;
      p.offsets[b] = start;
    } else {
      p.offsets[p.groups] = start;
    }
    int next = start;
    for (int w = 0; w < kWaves; ++w) {
      const int count = running[w * p.buckets + b];
      running[w * p.buckets + b] = next;
      next += count;
    }
  }
  __syncthreads();
  int bits = 1;
  while ((1 << bits) < p.buckets) ++bits;
#pragma unroll
  for (int round = 0; round < kMaxRounds; ++round) {
    if (round >= rounds) continue;  // (the same for the whole block)
    const int slot = wave_begin + round * 64 + lane;
    place_round(p, slot, kept[round], bits, mine);
  }
}

// The same sort of a few slots, a lane a slot, by a block of any size: no counters, no barrier. A slot's place is the number of slots
// before it in (bucket, slot) order, an offset the number of slots in lower buckets.
constexpr int kFewSlots = 16;  // (at 45 to 60 slots the walks over them take longer than the counting)
template <class IdOf>
__device__ __forceinline__ void sort_few(const PermuteParams& p, IdOf id_of) {
  const int lane = threadIdx.x % 64;
  const int bucket = lane >= p.slots ? p.buckets : lane < p.routed ? bucket_of_id(p, id_of(lane)) : p.experts;
  if (threadIdx.x < 64) {
    int place = 0;
    for (int slot = 0; slot < p.slots; ++slot) {
      const int other = __builtin_amdgcn_readlane(bucket, slot);
      place += other < bucket || (other == bucket && slot < lane) ? 1 : 0;
    }
    if (lane < p.slots) {
      p.order[place] = lane;
      p.rows[place] = row_of(p, lane);
    }
  }
  for (int b = threadIdx.x; b - lane <= p.groups; b += blockDim.x) {  // (whole wavefronts: every lane's slot is read)
    int below = 0, held = 0;
    for (int slot = 0; slot < p.slots; ++slot) {
      const int other = __builtin_amdgcn_readlane(bucket, slot);
      below += other < b ? 1 : 0;
      held += other == b ? 1 : 0;
    }
    if (b <= p.groups) p.offsets[b] = below;
    if (b < p.groups) p.sizes[b] = held;
  }
}

// A decode step's gate and dispatch (layer.hip): the gate's logits as kLogitShares partial sums of the depth,
// [share][token][expert] (logits.hip), where logit_shares says so; a router that adds them (route.hip); and, for at most
// kRouteAndSortTokens tokens, that router and the sort as one launch.
constexpr int kLogitShares = 16;
constexpr int kShareTokens = 64;
constexpr int kRouteAndSortTokens = 16;
enum LogitShares { kNoShares = 0, kFineShares = 1, kTileShares = 2 };
LogitShares logit_shares(int tokens, int depth, int experts);
int router_logit_shares(const void* x, const float* kernel, float* partial, int tokens, int depth, int experts, hipStream_t stream);
int route_shares(const dew_moe_router* router, const float* partial, const float* gate_bias, const float* selection_bias, int tokens,
                 float* weights, int32_t* indices, hipStream_t stream);
// A layer's last two launches as one, for a few tokens (decode.hip, gemm.hip): whether they are, and that launch.
bool combines_few(const dew_moe_bank* down, int tokens, int top_k, bool shared);
int down_and_combine(const char* who, const void* hidden, const int32_t* offsets, const dew_moe_bank* down, const float* bias, const int32_t* order,
                     const float* weights, int tokens, int top_k, bool shared, void* out, hipStream_t stream);
int route_and_sort(const dew_moe_router* router, const float* partial, const float* gate_bias, const float* selection_bias, int tokens,
                   bool shared, float* weights, int32_t* sizes, int32_t* offsets, int32_t* order, int32_t* rows, hipStream_t stream);

}  // namespace dew
