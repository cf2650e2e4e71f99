// Router: scores, (group-limited) selection, top-k and gate weights, one wavefront per token.
// Follows Router.__call__ from the logits on (reference src/dew/nn/moe.py:466-565). Every floating-point
// step is a fixed sequence of IEEE fp32/fp64 operations with contraction off, the same sequence the CPU
// oracle runs, so the chosen experts agree bit for bit.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "sort.h"

#pragma clang fp contract(off)

namespace dew {

constexpr int kWave = 64;
constexpr int kMaxPerLane = 8;   // experts <= 512
constexpr int kRouteWaves = 4;   // tokens per 256-thread block

// DeepSeek V4's score sqrt(softplus(x)) (src/dew/nn/moe.py:303-313), formed in float64 (softplus as max(x, 0) +
// log1p(exp(-|x|)), the square root IEEE) and rounded once to fp32: the CPU oracle's arithmetic for this score.
__device__ __forceinline__ float sqrt_softplus_f32(float x) {
  const double wide = static_cast<double>(x);
  return static_cast<float>(sqrt(fmax(wide, 0.0) + log1p(exp(-fabs(wide)))));
}

// A score that is a function of its own logit alone (every score function but softmax).
__device__ __forceinline__ float pointwise_score(int score_function, float logit) {
  return score_function == DEW_MOE_SCORE_SQRTSOFTPLUS ? sqrt_softplus_f32(logit) : 1.0f / (1.0f + exp_f32(-logit));
}

// The wavefront's largest value, in every lane: maxima within quads, half rows and rows of 16 lanes by DPP moves (one
// instruction each, no LDS crossbar), then lane 15 of each row into the next row and lane 31 into the upper half, so that
// lane 63 holds the maximum of all 64, which a lane read hands to everyone. (A maximum does not depend on the order it
// is taken in, so this is the butterfly's result; the sums below keep their fixed order.)
__device__ __forceinline__ float wave_max(float v) {
  auto moved = [](float value, auto control, auto rows) {
    const int bits = __builtin_bit_cast(int, value);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(bits, bits, decltype(control)::value, decltype(rows)::value, 0xF, false));
  };
  using std::integral_constant;
  v = fmaxf(v, moved(v, integral_constant<int, 0xB1>{}, integral_constant<int, 0xF>{}));   // quad_perm [1,0,3,2]
  v = fmaxf(v, moved(v, integral_constant<int, 0x4E>{}, integral_constant<int, 0xF>{}));   // quad_perm [2,3,0,1]
  v = fmaxf(v, moved(v, integral_constant<int, 0x141>{}, integral_constant<int, 0xF>{}));  // row_half_mirror
  v = fmaxf(v, moved(v, integral_constant<int, 0x140>{}, integral_constant<int, 0xF>{}));  // row_mirror
  v = fmaxf(v, moved(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{}));  // row_bcast15 into rows 1, 3
  v = fmaxf(v, moved(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{}));  // row_bcast31 into rows 2, 3
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Sum rounded once: fp64 partials per lane, then a butterfly over lanes 32, 16, 8, 4, 2 and 1 apart; every lane ends with the same value.
// (Both halves of a swap are added where a lane would add its own and the other's, and once lanes 8 apart hold the same, four lanes on in a
// row of 16 is four apart: the same additions as exchanges through the LDS crossbar, without its six round trips.)
__device__ __forceinline__ float wave_sum_once(double v) {
  auto words = [](double value) { return __builtin_bit_cast(uint64_t, value); };
  auto of = [](uint32_t low, uint32_t high) { return __builtin_bit_cast(double, static_cast<uint64_t>(high) << 32 | low); };
  {
    const uint32_t low = static_cast<uint32_t>(words(v)), high = static_cast<uint32_t>(words(v) >> 32);
    const auto lows = __builtin_amdgcn_permlane32_swap(low, low, false, false), highs = __builtin_amdgcn_permlane32_swap(high, high, false, false);
    v = of(lows[0], highs[0]) + of(lows[1], highs[1]);
  }
  {
    const uint32_t low = static_cast<uint32_t>(words(v)), high = static_cast<uint32_t>(words(v) >> 32);
    const auto lows = __builtin_amdgcn_permlane16_swap(low, low, false, false), highs = __builtin_amdgcn_permlane16_swap(high, high, false, false);
    v = of(lows[0], highs[0]) + of(lows[1], highs[1]);
  }
  auto add_moved = [&](auto control) {
    const uint32_t low = static_cast<uint32_t>(words(v)), high = static_cast<uint32_t>(words(v) >> 32);
    v = v + of(__builtin_amdgcn_mov_dpp(low, decltype(control)::value, 0xF, 0xF, true), __builtin_amdgcn_mov_dpp(high, decltype(control)::value, 0xF, 0xF, true));
  };
  add_moved(std::integral_constant<int, 0x128>{});  // row_ror 8
  add_moved(std::integral_constant<int, 0x124>{});  // row_ror 4
  add_moved(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  add_moved(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  return static_cast<float>(v);
}

// A float as an unsigned key of the same order (-inf lowest of the non-NaN), never 0.
__device__ __forceinline__ uint32_t ordered_key(float v) {
  const uint32_t bits = __float_as_uint(v);
  return (bits & 0x80000000u) ? ~bits : bits | 0x80000000u;
}

__device__ __forceinline__ float from_ordered_key(uint32_t key) {
  if (key == 0u) return -__builtin_inff();  // no token wrote here
  return __uint_as_float((key & 0x80000000u) ? key & 0x7fffffffu : ~key);
}

// A selection as it competes: by its value, either zero the same, NaN as -inf; 0, below them all, is none.
__device__ __forceinline__ uint32_t competing_key(float v) { return ordered_key(v == v ? v + 0.0f : -__builtin_inff()); }

// The wavefront's largest key, the same register in every lane: as wave_max, an instruction a move.
__device__ __forceinline__ uint32_t wave_max_key(uint32_t v) {
  auto moved = [](uint32_t value, auto control, auto rows) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, value, decltype(control)::value, decltype(rows)::value, 0xF, false));
  };
  using std::integral_constant;
  v = max(v, moved(v, integral_constant<int, 0xB1>{}, integral_constant<int, 0xF>{}));   // quad_perm [1,0,3,2]
  v = max(v, moved(v, integral_constant<int, 0x4E>{}, integral_constant<int, 0xF>{}));   // quad_perm [2,3,0,1]
  v = max(v, moved(v, integral_constant<int, 0x141>{}, integral_constant<int, 0xF>{}));  // row_half_mirror
  v = max(v, moved(v, integral_constant<int, 0x140>{}, integral_constant<int, 0xF>{}));  // row_mirror
  v = max(v, moved(v, integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{}));  // row_bcast15 into rows 1, 3
  v = max(v, moved(v, integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{}));  // row_bcast31 into rows 2, 3
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// The best of the wavefront's keys (key[i] of a lane is number lane + 64 i), ties to the lower number, taken out: its number, the same
// register in every lane. One of them is not 0.
// Bound by its chain: seven vector instructions one after another, a ballot a register and scalar ones. As values and numbers compared lane by
// lane before a butterfly of float maxima (four instructions a move) a round of 128 experts took some 0.4 us, a wavefront alone on its SIMD. A launch's us with
// that, sums through the LDS crossbar and a round trip of the gate's shares for every 64 experts, and now: one token of 128 experts, top 8, sorted too
// 6.5 -> 4.7, 64 tokens 5.9 -> 4.6, 1111 of 64, top 6, 5.75 -> 5.05, 2048 of 8, top 2, 5.0 -> 4.4, 8192 of 256 in 8 groups, top 8, 30 -> 27.
template <int kCount>
__device__ __forceinline__ int take_best(uint32_t (&key)[kCount]) {
  const int lane = threadIdx.x % kWave;
  uint32_t mine = key[0];
#pragma unroll
  for (int i = 1; i < kCount; ++i) mine = max(mine, key[i]);
  const uint32_t top = wave_max_key(mine);
  int best = 0;
#pragma unroll
  for (int i = kCount - 1; i >= 0; --i) {
    const unsigned long long holders = __ballot(key[i] == top);
    if (holders != 0ull) best = kWave * i + __builtin_ctzll(holders);
  }
#pragma unroll
  for (int i = 0; i < kCount; ++i) key[i] = lane + kWave * i == best ? 0u : key[i];
  return best;
}

struct RouteParams {
  const float* logits;
  const float* bias;
  float* weights;
  int32_t* indices;
  int tokens, experts, top_k, score_function, normalize, expert_groups, groups_per_token;
  int group_by_max;  // a group's score is its best selection (`group_score='max'`), not the sum of its two best
  float scaling;
  float* scores;  // nullable [T, E]: the activated scores, as the router sows them for the balance statistics
  float* log_z;   // nullable [T]: logsumexp of the logits (the z-loss's log partition)
  int bias_in_weights;   // the weights are the chosen scores + bias
  float sum_epsilon, sum_min;
  int fill_excluded;     // an expert outside the kept groups competes at `excluded` rather than -inf
  float excluded;
  float softcap;         // above 0: every logit is read as softcap * tanh(logit / softcap)
  const int32_t* given;    // nullable [T, k]: the experts to use in place of the router's own choice (a replayed record, a hash table's)
  const uint8_t* covered;  // nullable [T]: with `given`, the tokens it covers; the others keep the router's choice
  const float* media_bias; // nullable [E]: the bias a media token's experts are chosen by, in place of `bias`
  const uint8_t* media;    // nullable [T]: the media tokens
  // Block routing (`Router.block_mask`, src/dew/nn/moe.py:566-585): tokens are `rows` x `length`, each in the block of its
  // row that `blocks` numbers (negative: padding, a block of its own); a token chooses among its block's shortlist.
  const int32_t* blocks;   // nullable [T]
  int length;              // tokens a row
  uint32_t* block_keys;    // [rows x (length + 1), E]: a block's best selection for every expert, as ordered keys (0: none yet)
  const uint8_t* allowed;  // [rows x (length + 1), 64]: bit i of byte `lane` set where expert lane + 64 i is on the block's shortlist
  int gather_blocks;       // this launch only gathers the blocks' best selections into block_keys
  const float* gate_bias;  // nullable [E]: still due to logits that come in shares
};

// The block a token routes with: its row's blocks are numbered from 0, padding (or an id past the row) is block `length`.
__device__ __forceinline__ size_t block_of(const RouteParams& p, int token) {
  const int id = p.blocks[token];
  return static_cast<size_t>(token / p.length) * (p.length + 1) + ((id < 0 || id > p.length) ? p.length : id);
}

// Laguna's capped gate logit (`capped_logits`, src/dew/nn/precision.py:2086-2092): cap * tanh(logit / cap) in fp32.
__device__ __forceinline__ float capped(float logit, float cap) { return cap > 0.0f ? cap * tanhf(logit / cap) : logit; }

// A token's logits, expert lane + 64 i in logit[i]: as they are, or added up from the gate's shares of the depth in the order the
// gate's own launch adds them.
template <int kPerLane, bool SHARES>  // SHARES: p.logits are kLogitShares partial sums of them, [share][T][E] (logits.hip)
__device__ __forceinline__ void read_logits(const RouteParams& p, int token, float (&logit)[kPerLane]) {
  const int lane = threadIdx.x % kWave;
  const float* row = p.logits + static_cast<size_t>(token) * p.experts;
  if constexpr (SHARES) {
    constexpr int kAtOnce = kPerLane < 4 ? kPerLane : 4;
#pragma unroll
    for (int first = 0; first < kPerLane; first += kAtOnce) {
      float share[kAtOnce][kLogitShares];
      auto expert = [&](int i) { return min(lane + kWave * (first + i), p.experts - 1); };
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i)
#pragma unroll
        for (int s = 0; s < kLogitShares; ++s) share[i][s] = row[static_cast<size_t>(s) * p.tokens * p.experts + expert(i)];
      __builtin_amdgcn_sched_barrier(0);  // (all of them asked for before the first is waited for)
#pragma unroll
      for (int i = 0; i < kAtOnce; ++i) {
        float value = share[i][0];
#pragma unroll
        for (int s = 1; s < kLogitShares; ++s) value += share[i][s];
        if (p.gate_bias != nullptr) value = value + p.gate_bias[expert(i)];
        logit[first + i] = value;
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) logit[i] = row[min(lane + kWave * i, p.experts - 1)];
  }
#pragma unroll
  for (int i = 0; i < kPerLane; ++i)
    if (lane + kWave * i >= p.experts) logit[i] = -__builtin_inff();
}

// One token of a wavefront, from its logits (expert lane + 64 i in logit[i], -inf past the experts) to its experts and weights:
// lane j < top_k returns the j-th. `mine`: the wavefront's own LDS, p.experts floats, where there are expert groups.
struct Chosen {
  float weight;
  int expert;
};
template <int kPerLane>  // experts <= 64 * kPerLane
__device__ __forceinline__ Chosen routed_token(const RouteParams& p, int token, bool active, float (&logit)[kPerLane], float* mine) {
  const int lane = threadIdx.x % kWave;
  const float ninf = -__builtin_inff();
  float score[kPerLane], select[kPerLane];
  if (p.softcap > 0.0f) {  // (a branch of its own: the cap's hyperbolic tangent stays out of the routers that have none)
#pragma unroll
    for (int i = 0; i < kPerLane; ++i)
      if (lane + kWave * i < p.experts) logit[i] = capped(logit[i], p.softcap);
  }

  float top = ninf, denom = 1.0f;
  if (p.score_function == DEW_MOE_SCORE_SOFTMAX) {
    float m = ninf;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) m = fmaxf(m, logit[i]);
    top = wave_max(m);
    double partial = 0.0;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int e = lane + kWave * i;
      score[i] = e < p.experts ? exp_f32(logit[i] - top) : 0.0f;
      partial = partial + static_cast<double>(score[i]);
    }
    denom = wave_sum_once(partial);
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) score[i] = score[i] / denom;
  } else {
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) score[i] = pointwise_score(p.score_function, logit[i]);
  }

  // What the router sows beside its choices (src/dew/nn/moe.py:474-479): the scores, and the log partition
  // max + log(sum exp(logit - max)) of the logits whatever the score function.
  if (p.scores != nullptr && active) {
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int e = lane + kWave * i;
      if (e < p.experts) p.scores[static_cast<size_t>(token) * p.experts + e] = score[i];
    }
  }
  if (p.log_z != nullptr) {
    float m = ninf;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) m = fmaxf(m, logit[i]);
    m = wave_max(m);
    double partial = 0.0;
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int e = lane + kWave * i;
      if (e < p.experts) partial = partial + static_cast<double>(exp_f32(logit[i] - m));
    }
    const float total = wave_sum_once(partial);
    if (active && lane == 0) p.log_z[token] = m + logf(total);
  }

  const bool by_media = p.media != nullptr && p.media[token] != 0;  // DeepSeek-V4.1's image-span tokens (one token a wavefront)
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const int e = lane + kWave * i;
    float s = score[i];
    if (e < p.experts) {
      if (by_media) s = s + p.media_bias[e];
      else if (p.bias != nullptr) s = s + p.bias[e];
    }
    // A NaN selection (a NaN in the bias or the logits) is never preferred: it competes as -inf, so every round still
    // finds an expert in range (no comparison with NaN holds, and a round without a candidate would name no expert).
    select[i] = (e < p.experts && s == s) ? s : ninf;
  }

  if (p.blocks != nullptr) {  // (a block router has no expert groups: no barrier lies ahead of the early return)
    const size_t block = block_of(p, token);
    if (p.gather_blocks) {
      if (active) {
#pragma unroll
        for (int i = 0; i < kPerLane; ++i) {
          const int e = lane + kWave * i;
          if (e < p.experts) atomicMax(p.block_keys + block * p.experts + e, ordered_key(select[i]));
        }
      }
      return Chosen{0.0f, 0};
    }
    const unsigned shortlist = p.allowed[block * kWave + lane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i)
      if (!((shortlist >> i) & 1u)) select[i] = ninf;
  }

  if (p.expert_groups > 1) {
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int e = lane + kWave * i;
      if (e < p.experts) mine[e] = select[i];
    }
    // (the selections are the wavefront's own: an order between its lanes is all the reads below need)
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int per_group = p.experts / p.expert_groups;
    // lane g scores group g: the sum of its two best selections
    float group_score = ninf;
    if (lane < p.expert_groups) {
      float first = ninf, second = ninf;
      for (int j = 0; j < per_group; ++j) {
        const float v = mine[lane * per_group + j];
        if (v > first) {
          second = first;
          first = v;
        } else if (v > second) {
          second = v;
        }
      }
      group_score = p.group_by_max ? first : first + second;
    }
    unsigned long long kept = 0ull;
    uint32_t group_key[1] = {lane < p.expert_groups && group_score == group_score ? competing_key(group_score) : 0u};
    for (int round = 0; round < p.groups_per_token; ++round) {
      if (__ballot(group_key[0] != 0u) == 0ull) break;  // (a group whose two best are infinities of either sign has no score)
      kept |= 1ull << take_best(group_key);
    }
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) {
      const int e = lane + kWave * i;
      if (e < p.experts && !((kept >> (e / per_group)) & 1ull)) select[i] = p.fill_excluded ? p.excluded : ninf;
    }
  }

  // A token whose experts are given takes them as they come; the wavefront is one token, so the branch is uniform. A given
  // id outside [0, experts) (a dropped slot's sentinel in a replayed record) is written back as it came, with weight zero
  // and no part in the other slots' normalization: the reference passes such ids through (`chosen_experts`,
  // src/dew/nn/moe.py:202-224) and its sort drops the slot. Its reads below go to the nearest expert, to stay in range.
  const bool replayed = p.given != nullptr && (p.covered == nullptr || p.covered[token] != 0);
  // top-k: k rounds of a wave-wide argmax, ties to the lower index
  int my_choice = 0, given_id = 0;
  bool in_range = true;
  if (replayed && lane < p.top_k) {
    given_id = p.given[static_cast<size_t>(token) * p.top_k + lane];
    in_range = given_id >= 0 && given_id < p.experts;
    my_choice = min(max(given_id, 0), p.experts - 1);
  }
  if (!replayed) {
    uint32_t key[kPerLane];
#pragma unroll
    for (int i = 0; i < kPerLane; ++i) key[i] = lane + kWave * i < p.experts ? competing_key(select[i]) : 0u;
    for (int round = 0; round < p.top_k; ++round) {
      const int best = take_best(key);
      if (lane == round) my_choice = best;
    }
  }

  // gate weights: lane j < k owns the j-th choice
  const bool owner = lane < p.top_k && in_range;
  float chosen_logit = ninf;  // (read from the lane that holds it: no round trip to the logits)
#pragma unroll
  for (int i = 0; i < kPerLane; ++i) {
    const float held = __shfl(logit[i], my_choice % kWave, kWave);
    if (owner && my_choice / kWave == i) chosen_logit = held;
  }
  float weight = 0.0f;
  if (p.score_function == DEW_MOE_SCORE_SOFTMAX && p.normalize && !p.bias_in_weights && !(p.sum_min != 0.0f)) {
    const float m = wave_max(chosen_logit);
    const float shifted = owner ? exp_f32(chosen_logit - m) : 0.0f;
    const float total = wave_sum_once(static_cast<double>(shifted));
    weight = shifted / total;
  } else {
    if (owner) {
      weight = p.score_function == DEW_MOE_SCORE_SOFTMAX ? exp_f32(chosen_logit - top) / denom
                                                         : pointwise_score(p.score_function, chosen_logit);
      if (p.bias_in_weights) weight = weight + p.bias[my_choice];
    }
    if (p.normalize) {
      auto of_lane = [&](int j) { return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(weight), j)); };
      float total = of_lane(0);
      for (int j = 1; j < p.top_k; ++j) total = total + of_lane(j);
      total = total + p.sum_epsilon;
      if (p.sum_min != 0.0f) total = fmaxf(total, p.sum_min);
      weight = weight / total;
    }
  }
  weight = weight * p.scaling;
  return Chosen{in_range ? weight : 0.0f, replayed ? given_id : my_choice};
}

// (SHARES apart: the shares in flight take 98 registers of more than 128 experts' launches, four wavefronts a SIMD, where logits as they are take 42 and
// eight. Of few tokens, each a chain alone, that costs nothing; in one launch for both forms the many tokens that come without shares paid for it: 32 768 of 256
// experts in 8 groups, top 1, 47 us, apart 33, 16 384 of 192 22 and 16.)
template <int kPerLane, bool SHARES>
__global__ __launch_bounds__(kWave* kRouteWaves) void route_kernel(RouteParams p) {
  extern __shared__ float shared[];  // [kRouteWaves][experts] selections, for the group scores
  const int lane = threadIdx.x % kWave;
  const int wave = threadIdx.x / kWave;
  const int token_raw = blockIdx.x * kRouteWaves + wave;
  const bool active = token_raw < p.tokens;
  const int token = active ? token_raw : p.tokens - 1;
  float logit[kPerLane];
  read_logits<kPerLane, SHARES>(p, token, logit);
  const Chosen chosen = routed_token<kPerLane>(p, token, active, logit, shared + wave * p.experts);
  if (p.gather_blocks) return;
  if (active && lane < p.top_k) {
    p.weights[static_cast<size_t>(token) * p.top_k + lane] = chosen.weight;
    p.indices[static_cast<size_t>(token) * p.top_k + lane] = chosen.expert;
  }
}

// The router and the sort of up to sixteen tokens in one block: a wavefront routes a token and leaves its experts in the LDS,
// where the whole block then sorts them. They are two launches of 4 to 5 us otherwise, most of either its own latency. (More
// tokens, several a wavefront, are slower than two launches: some 750 instructions a token on one CU's four SIMDs.)
// Measured, one token of 128 experts, top 8: 8.8 us with the sort that counts, 6.8 with the one of few slots, 4.7 with rounds of keys (take_best).
constexpr int kSortWaves = kSmallThreads / kWave;
template <int kPerLane>
__global__ __launch_bounds__(kSmallThreads) void route_and_sort_kernel(RouteParams p, PermuteParams sort) {
  extern __shared__ int32_t scratch[];  // the sort's counters (before them the group scores' selections), then the slots' experts
  int32_t* ids = scratch + max(kSortWaves * p.experts, (kSortWaves + 1) * sort.buckets + 1);
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  if (wave < p.tokens) {  // a wavefront a token; the others wait for the sort
    float logit[kPerLane];
    read_logits<kPerLane, true>(p, wave, logit);
    const Chosen chosen = routed_token<kPerLane>(p, wave, true, logit, reinterpret_cast<float*>(scratch) + wave * p.experts);
    if (lane < p.top_k) {
      p.weights[wave * p.top_k + lane] = chosen.weight;
      ids[wave * p.top_k + lane] = chosen.expert;
    }
  }
  __syncthreads();
  auto id_of = [ids](int slot) { return ids[slot]; };
  if (sort.slots <= kFewSlots)
    sort_few(sort, id_of);
  else
    sort_small<kSmallThreads>(sort, scratch, id_of);
}

// Each block's shortlist: the `count` best of its best selections (ties to the lower index), one wavefront a block.
__global__ __launch_bounds__(kWave* kRouteWaves) void block_shortlist_kernel(const uint32_t* __restrict__ keys, uint8_t* __restrict__ allowed,
                                                                             int blocks, int experts, int count) {
  const int lane = threadIdx.x % kWave;
  const int block = blockIdx.x * kRouteWaves + threadIdx.x / kWave;
  if (block >= blocks) return;
  uint32_t key[kMaxPerLane];
#pragma unroll
  for (int i = 0; i < kMaxPerLane; ++i) {
    const int e = lane + kWave * i;
    key[i] = e < experts ? competing_key(from_ordered_key(keys[static_cast<size_t>(block) * experts + e])) : 0u;
  }
  unsigned taken = 0u;
  for (int round = 0; round < count; ++round) {
    const int best = take_best(key);
    if (best % kWave == lane) taken |= 1u << (best / kWave);
  }
  allowed[static_cast<size_t>(block) * kWave + lane] = static_cast<uint8_t>(taken);
}

__global__ __launch_bounds__(256) void clear_words_kernel(uint32_t* __restrict__ words, size_t count) {
  for (size_t i = blockIdx.x * 256ull + threadIdx.x; i < count; i += static_cast<size_t>(gridDim.x) * 256) words[i] = 0u;
}

}  // namespace dew

extern "C" int dew_moe_route(const float* logits, const float* bias, int32_t tokens, int32_t experts,
                             int32_t top_k, int32_t score_function, int32_t normalize, float scaling,
                             int32_t expert_groups, int32_t groups_per_token, float* weights,
                             int32_t* indices, void* stream) {
  return dew_moe_route_sown(logits, bias, tokens, experts, top_k, score_function, normalize, scaling, expert_groups,
                            groups_per_token, weights, indices, nullptr, nullptr, stream);
}

extern "C" int dew_moe_route_sown(const float* logits, const float* bias, int32_t tokens, int32_t experts,
                                  int32_t top_k, int32_t score_function, int32_t normalize, float scaling,
                                  int32_t expert_groups, int32_t groups_per_token, float* weights,
                                  int32_t* indices, float* scores, float* log_z, void* stream) {
  const dew_moe_router router{experts, top_k, score_function, normalize, scaling, expert_groups, groups_per_token,
                              DEW_MOE_GROUP_TOP2, 0, DEW_MOE_WEIGHT_SUM_EPSILON, 0.0f, 0, 0.0f, 0.0f};
  return dew_moe_route_with(&router, logits, bias, tokens, weights, indices, scores, log_z, stream);
}

extern "C" int dew_moe_route_with(const dew_moe_router* router, const float* logits, const float* bias, int32_t tokens,
                                  float* weights, int32_t* indices, float* scores, float* log_z, void* stream) {
  return dew_moe_route_call(router, logits, bias, nullptr, nullptr, nullptr, nullptr, tokens, weights, indices, scores, log_z, stream);
}

namespace dew {
struct BlockRouting {
  const int32_t* blocks = nullptr;
  int length = 0;
  uint32_t* keys = nullptr;
  const uint8_t* allowed = nullptr;
  int gather = 0;
};
static int route_launch(const dew_moe_router* router, const float* logits, const float* bias, const float* media_bias,
                        const uint8_t* media, const int32_t* given, const uint8_t* covered, const BlockRouting& by_block,
                        int32_t tokens, float* weights, int32_t* indices, float* scores, float* log_z, void* stream);
}  // namespace dew

extern "C" int dew_moe_route_call(const dew_moe_router* router, const float* logits, const float* bias,
                                  const float* media_bias, const uint8_t* media, const int32_t* given,
                                  const uint8_t* covered, int32_t tokens, float* weights, int32_t* indices, float* scores,
                                  float* log_z, void* stream) {
  return dew::route_launch(router, logits, bias, media_bias, media, given, covered, dew::BlockRouting{}, tokens, weights, indices,
                           scores, log_z, stream);
}

namespace dew {

static int check_router(const dew_moe_router* router, const float* bias, int32_t tokens) {
  DEW_REQUIRE(router, "dew_moe_route: the router's description must not be null");
  const int experts = router->experts, top_k = router->top_k, score_function = router->score_function;
  const int expert_groups = router->expert_groups, groups_per_token = router->groups_per_token;
  DEW_REQUIRE(tokens >= 0 && experts >= 1, "dew_moe_route: tokens %d experts %d", tokens, experts);
  DEW_REQUIRE(experts <= kWave * kMaxPerLane, "dew_moe_route: at most %d experts, got %d", kWave * kMaxPerLane,
              experts);
  DEW_REQUIRE(top_k >= 1 && top_k <= experts && top_k <= kWave, "dew_moe_route: top_k %d of %d experts (at most %d)",
              top_k, experts, kWave);
  DEW_REQUIRE(score_function == DEW_MOE_SCORE_SOFTMAX || score_function == DEW_MOE_SCORE_SIGMOID || score_function == DEW_MOE_SCORE_SQRTSOFTPLUS,
              "dew_moe_route: score_function %d is none of softmax (0), sigmoid (1), sqrtsoftplus (2)", score_function);
  DEW_REQUIRE(router->group_score == DEW_MOE_GROUP_TOP2 || router->group_score == DEW_MOE_GROUP_MAX,
              "dew_moe_route: group_score %d is neither top2 (0) nor max (1)", router->group_score);
  DEW_REQUIRE(expert_groups >= 1 && expert_groups <= kWave && experts % expert_groups == 0,
              "dew_moe_route: %d experts do not split into %d groups (at most %d)", experts, expert_groups, kWave);
  if (expert_groups > 1) {
    DEW_REQUIRE(groups_per_token >= 1 && groups_per_token <= expert_groups,
                "dew_moe_route: groups_per_token %d of %d groups", groups_per_token, expert_groups);
    DEW_REQUIRE(experts / expert_groups >= 2 || router->group_score == DEW_MOE_GROUP_MAX,
                "dew_moe_route: a group's score sums its two best experts, got %d a group", experts / expert_groups);
    DEW_REQUIRE(top_k <= groups_per_token * (experts / expert_groups),
                "dew_moe_route: top_k %d exceeds the %d experts of the kept groups", top_k,
                groups_per_token * (experts / expert_groups));
  }
  DEW_REQUIRE(!router->bias_in_weights || bias, "dew_moe_route: bias_in_weights gates on the balancing bias, which is null");
  DEW_REQUIRE(router->weight_sum_epsilon >= 0.0f && router->weight_sum_min >= 0.0f,
              "dew_moe_route: weight_sum_epsilon %g and weight_sum_min %g bound a sum from below: neither is negative",
              static_cast<double>(router->weight_sum_epsilon), static_cast<double>(router->weight_sum_min));
  DEW_REQUIRE(router->logit_softcap >= 0.0f, "dew_moe_route: logit_softcap %g is a positive cap, or 0 for none",
              static_cast<double>(router->logit_softcap));
  return DEW_MOE_OK;
}

static RouteParams route_params(const dew_moe_router* router, const float* logits, const float* bias, const float* media_bias, const uint8_t* media,
                                const int32_t* given, const uint8_t* covered, const BlockRouting& by_block, int32_t tokens, float* weights,
                                int32_t* indices, float* scores, float* log_z) {
  return RouteParams{logits, bias, weights, indices, tokens, router->experts, router->top_k, router->score_function, router->normalize ? 1 : 0,
                router->expert_groups, router->groups_per_token, router->group_score == DEW_MOE_GROUP_MAX ? 1 : 0, router->scaling, scores, log_z,
                router->bias_in_weights ? 1 : 0, router->weight_sum_epsilon, router->weight_sum_min,
                router->fill_excluded ? 1 : 0, router->excluded_group_score, router->logit_softcap, given, covered, media_bias, media,
                by_block.blocks, by_block.length, by_block.keys, by_block.allowed, by_block.gather, nullptr};
}

// (Kernels lie in the library in the order of their first use here. With the four kernels of whole logits ahead of the four of shares the same instructions cost a
// pass that takes shares more: 2048 tokens of 512 x 1024, 2 of 8 experts, replayed, 47.7 us, as here 46.9. With all four of shares first 22 tokens of 256 experts take 0.3 more.)
static int launch_route(const RouteParams& p, bool shares, hipStream_t s) {
  const size_t shared = p.expert_groups > 1 ? sizeof(float) * kRouteWaves * p.experts : 0;
  const dim3 grid((p.tokens + kRouteWaves - 1) / kRouteWaves), block(kWave * kRouteWaves);
  auto kernel = p.experts <= 64    ? (shares ? route_kernel<1, true> : route_kernel<1, false>)
                : p.experts <= 128 ? (shares ? route_kernel<2, true> : route_kernel<2, false>)
                : p.experts <= 256 ? (shares ? route_kernel<4, true> : route_kernel<4, false>)
                                   : (shares ? route_kernel<kMaxPerLane, true> : route_kernel<kMaxPerLane, false>);
  hipLaunchKernelGGL(kernel, grid, block, shared, s, p);
  return launched("route_kernel");
}

}  // namespace dew

int dew::route_launch(const dew_moe_router* router, const float* logits, const float* bias, const float* media_bias,
                             const uint8_t* media, const int32_t* given, const uint8_t* covered, const BlockRouting& by_block,
                             int32_t tokens, float* weights, int32_t* indices, float* scores, float* log_z, void* stream) {
  DEW_REQUIRE(given || !covered, "dew_moe_route: a coverage without the experts it covers");
  DEW_REQUIRE((media == nullptr) == (media_bias == nullptr), "dew_moe_route: the media tokens and the bias that chooses for them come together");
  if (int rc = check_router(router, bias, tokens)) return rc;
  DEW_REQUIRE(tokens == 0 || (logits && weights && indices), "dew_moe_route: logits, weights and indices must not be null");
  if (tokens == 0) return DEW_MOE_OK;
  const RouteParams p = route_params(router, logits, bias, media_bias, media, given, covered, by_block, tokens, weights, indices, scores, log_z);
  return launch_route(p, false, static_cast<hipStream_t>(stream));
}

int dew::route_shares(const dew_moe_router* router, const float* partial, const float* gate_bias, const float* selection_bias, int tokens,
                      float* weights, int32_t* indices, hipStream_t stream) {
  if (int rc = check_router(router, selection_bias, tokens)) return rc;
  RouteParams p = route_params(router, partial, selection_bias, nullptr, nullptr, nullptr, nullptr, BlockRouting{}, tokens, weights, indices, nullptr,
                               nullptr);
  p.gate_bias = gate_bias;
  return launch_route(p, true, stream);
}

int dew::route_and_sort(const dew_moe_router* router, const float* partial, const float* gate_bias, const float* selection_bias, int tokens,
                        bool shared, float* weights, int32_t* sizes, int32_t* offsets, int32_t* order, int32_t* rows, hipStream_t stream) {
  if (int rc = check_router(router, selection_bias, tokens)) return rc;
  const int experts = router->experts, slots = tokens * router->top_k + (shared ? tokens : 0);
  DEW_REQUIRE(tokens >= 1 && tokens <= kRouteAndSortTokens && slots <= kSmallSlots, "route_and_sort: %d tokens, %d slots", tokens, slots);
  RouteParams p = route_params(router, partial, selection_bias, nullptr, nullptr, nullptr, nullptr, BlockRouting{}, tokens, weights, nullptr, nullptr,
                               nullptr);
  p.gate_bias = gate_bias;
  const int groups = experts + (shared ? 1 : 0);
  const PermuteParams sort{nullptr, sizes, offsets, order, rows, nullptr, slots, tokens * router->top_k, experts, groups, router->top_k, 1, groups + 1, slots};
  const size_t lds = sizeof(int32_t) * (static_cast<size_t>(std::max(kSortWaves * experts, (kSortWaves + 1) * sort.buckets + 1)) + sort.routed);
  static_assert(sizeof(int32_t) * ((kSortWaves + 1) * (kWave * kMaxPerLane + 2) + 1 + kSmallSlots) <= 65536, "the block's LDS");
  // (few slots are sorted by any block: a wavefront a token, and four at least for the offsets)
  const dim3 grid(1), block(slots <= kFewSlots ? kWave * std::max(tokens, 4) : kSmallThreads);
  if (experts <= 64) {
    hipLaunchKernelGGL(route_and_sort_kernel<1>, grid, block, lds, stream, p, sort);
  } else if (experts <= 128) {
    hipLaunchKernelGGL(route_and_sort_kernel<2>, grid, block, lds, stream, p, sort);
  } else if (experts <= 256) {
    hipLaunchKernelGGL(route_and_sort_kernel<4>, grid, block, lds, stream, p, sort);
  } else {
    hipLaunchKernelGGL(route_and_sort_kernel<kMaxPerLane>, grid, block, lds, stream, p, sort);
  }
  return launched("route_and_sort_kernel");
}

extern "C" size_t dew_moe_route_blocks_workspace_bytes(int32_t rows, int32_t length, int32_t experts) {
  if (rows <= 0 || length <= 0 || experts <= 0) return 0;
  const size_t blocks = static_cast<size_t>(rows) * (static_cast<size_t>(length) + 1);
  return blocks * experts * sizeof(uint32_t) + blocks * dew::kWave;
}

extern "C" int dew_moe_route_blocks(const dew_moe_router* router, const float* logits, const float* bias,
                                    const int32_t* blocks, int32_t rows, int32_t length, int32_t block_experts,
                                    void* workspace, size_t workspace_bytes, float* weights, int32_t* indices, float* scores,
                                    float* log_z, void* stream) {
  using namespace dew;
  DEW_REQUIRE(router, "dew_moe_route_blocks: the router's description must not be null");
  DEW_REQUIRE(rows >= 0 && length >= 1 && static_cast<long long>(rows) * length <= 0x7fffffffLL,
              "dew_moe_route_blocks: %d rows of %d tokens", rows, length);
  DEW_REQUIRE(router->expert_groups == 1, "dew_moe_route_blocks: block routing limits a token to its block's experts, so it has no expert groups");
  DEW_REQUIRE(block_experts >= router->top_k && block_experts <= router->experts,
              "dew_moe_route_blocks: block_experts %d must hold the top_k of %d and at most the %d experts", block_experts,
              router->top_k, router->experts);
  if (rows == 0) return DEW_MOE_OK;
  DEW_REQUIRE(blocks, "dew_moe_route_blocks: the tokens' blocks must not be null");
  const size_t needed = dew_moe_route_blocks_workspace_bytes(rows, length, router->experts);
  DEW_REQUIRE(workspace && workspace_bytes >= needed && reinterpret_cast<uintptr_t>(workspace) % 4 == 0,
              "dew_moe_route_blocks: the workspace holds %zu bytes of the %zu needed (dew_moe_route_blocks_workspace_bytes), 4-byte aligned",
              workspace ? workspace_bytes : size_t{0}, needed);
  const int tokens = rows * length;
  const size_t segments = static_cast<size_t>(rows) * (static_cast<size_t>(length) + 1);
  const size_t words = segments * router->experts;
  uint32_t* keys = static_cast<uint32_t*>(workspace);
  uint8_t* allowed = reinterpret_cast<uint8_t*>(keys + words);
  hipStream_t s = static_cast<hipStream_t>(stream);
  // (a kernel, not a memset: a caller may capture these launches in a graph)
  hipLaunchKernelGGL(clear_words_kernel, dim3(static_cast<unsigned>(std::min<size_t>((words + 255) / 256, 4096))), dim3(256), 0, s, keys, words);
  BlockRouting by_block;
  by_block.blocks = blocks, by_block.length = length, by_block.keys = keys, by_block.allowed = allowed, by_block.gather = 1;
  int status = route_launch(router, logits, bias, nullptr, nullptr, nullptr, nullptr, by_block, tokens, weights, indices, nullptr, nullptr, stream);
  if (status != DEW_MOE_OK) return status;
  hipLaunchKernelGGL(block_shortlist_kernel, dim3(static_cast<unsigned>((segments + kRouteWaves - 1) / kRouteWaves)), dim3(kWave * kRouteWaves),
                     0, s, keys, allowed, static_cast<int>(segments), router->experts, block_experts);
  by_block.gather = 0;
  return route_launch(router, logits, bias, nullptr, nullptr, nullptr, nullptr, by_block, tokens, weights, indices, scores, log_z, stream);
}

namespace dew {

// The aux-loss-free balancing step on the selection bias (src/dew/nn/moe.py:271-300 `load_balance_update`, applied
// as src/dew/objectives/routing.py:342-345): an expert that took more slots than the average loses `rate`, one that
// took fewer gains it, one exactly at the floor of the average gains it only if the average has a remainder.
__global__ __launch_bounds__(256) void balance_bias_kernel(const int32_t* __restrict__ counts, float* __restrict__ bias,
                                                           float rate, int experts) {
  __shared__ long long partial[256];
  long long sum = 0;
  for (int e = threadIdx.x; e < experts; e += 256) sum += counts[e];
  partial[threadIdx.x] = sum;
  __syncthreads();
  for (int half = 128; half >= 1; half >>= 1) {
    if (threadIdx.x < half) partial[threadIdx.x] += partial[threadIdx.x + half];
    __syncthreads();
  }
  const long long total = partial[0];
  const long long average = total / experts, remainder = total % experts;
  for (int e = threadIdx.x; e < experts; e += 256) {
    const long long count = counts[e];
    const float direction = count > average ? -1.0f : (count < average || remainder > 0) ? 1.0f : 0.0f;
    bias[e] = bias[e] + rate * direction;
  }
}

}  // namespace dew

extern "C" int dew_moe_balance_bias(const int32_t* counts, float* bias, float rate, int32_t experts, void* stream) {
  using namespace dew;
  DEW_REQUIRE(experts >= 1, "dew_moe_balance_bias: experts %d", experts);
  DEW_REQUIRE(counts && bias, "dew_moe_balance_bias: counts and bias must not be null");
  hipLaunchKernelGGL(balance_bias_kernel, dim3(1), dim3(256), 0, static_cast<hipStream_t>(stream), counts, bias, rate, experts);
  return launched("balance_bias_kernel");
}
