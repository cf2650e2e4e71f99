// A sparse expert layer's whole forward pass as one call: gate logits, routing, the dispatch sort, the expert products and
// the combine, on one workspace. The launches are the ones the separate entry points make, in the same order on the same
// stream, so the same bits; what the one call saves is the host's work between them. Two pairs of launches are one launch each that has no entry point of
// its own, where a step is bound by its launches: a few tokens' router and sort (route_and_sort, route.hip), and small experts' down product and
// combine (down_and_combine, gemm.hip), which form every sum in the separate launches' order.
// Measured on one token of 128 experts of 2048 x 768 (FP8 blocks), where the launches' own time is 51 us: 123 us a pass
// through the separate entry points, each with its own checks, allocations and foreign call.
#include "common.h"
#include "sort.h"

namespace dew {

struct LayerWorkspace {
  size_t logits, weights, indices, sizes, offsets, order, rows, sort, x_rows, x_scale, hidden, slots, split, bytes;
  size_t sort_bytes, split_bytes;
};

// What the products of `rows` sorted rows run on: the same rules as the separate calls'.
enum LayerForm { kRowsBf16 = 0, kRowsF16 = 1, kRowsSplit = 2 };

static LayerForm layer_form(const dew_moe_layer* layer, const dew_moe_bank* gate, const dew_moe_bank* up, const dew_moe_bank* down,
                            int32_t rows, int32_t split_terms, int32_t f16_rows_from) {
  if (layer->gating == DEW_MOE_GATE_INTERLEAVED) return kRowsBf16;
  if (split_terms >= 0 && dew_moe_prefers_split_rows(gate, up, down, rows)) return kRowsSplit;
  if (f16_rows_from >= 0 && gate->format == DEW_MOE_W_NVFP4 && up->format == DEW_MOE_W_NVFP4 &&
      rows >= static_cast<int64_t>(f16_rows_from) * gate->experts)
    return kRowsF16;
  return kRowsBf16;
}

static LayerWorkspace layer_workspace(const dew_moe_layer* layer, const dew_moe_bank* gate, const dew_moe_bank* down, int64_t tokens,
                                      LayerForm form) {
  const int64_t slots = tokens * layer->router.top_k, rows = slots + (layer->shared ? tokens : 0);
  const int64_t groups = layer->router.experts + (layer->shared ? 1 : 0);
  const int64_t depth = gate->depth, hidden_width = down->depth, width = down->width;
  LayerWorkspace w{};
  size_t at = 0;
  auto take = [&at](int64_t bytes) {
    const size_t here = at;
    at += (static_cast<size_t>(bytes) + 255) / 256 * 256;
    return here;
  };
  w.logits = take(tokens * layer->router.experts * 4 * (logit_shares(static_cast<int>(tokens), gate->depth, layer->router.experts) ? kLogitShares : 1));
  w.weights = take(slots * 4);
  w.indices = take(slots * 4);
  w.sizes = take(groups * 4);
  w.offsets = take((groups + 1) * 4);
  w.order = take(rows * 4);
  w.rows = take(rows * 4);
  w.sort_bytes = dew_moe_permute_workspace_bytes(static_cast<int32_t>(rows), static_cast<int32_t>(groups));
  w.sort = take(w.sort_bytes);
  if (form == kRowsF16) {
    w.x_rows = take(tokens * depth * 2);
    w.x_scale = take(tokens);
  }
  if (form == kRowsSplit) {
    w.split_bytes = dew_moe_swiglu_mlp_split_workspace_bytes(static_cast<int32_t>(tokens), static_cast<int32_t>(rows), gate->depth,
                                                             gate->width, gate->experts);
    w.split = take(w.split_bytes);
  } else {
    w.hidden = take(rows * hidden_width * 2);
  }
  w.slots = take(rows * width * 2);
  w.bytes = at + 256;  // room to align the caller's base
  return w;
}

static int check_layer(const char* who, const dew_moe_layer* layer, const dew_moe_bank* gate, const dew_moe_bank* up,
                       const dew_moe_bank* down, int32_t tokens) {
  DEW_REQUIRE(layer && gate && down, "%s: the layer and its banks must not be null", who);
  const bool interleaved = layer->gating == DEW_MOE_GATE_INTERLEAVED;
  DEW_REQUIRE(interleaved || layer->gating == DEW_MOE_GATE_SILU || layer->gating == DEW_MOE_GATE_GELU_TANH, "%s: gating %d", who, layer->gating);
  DEW_REQUIRE(interleaved == (up == nullptr), "%s: interleaved experts have one gate_up bank, the others a gate and an up bank", who);
  DEW_REQUIRE(!interleaved || !layer->shared, "%s: interleaved experts have no shared expert", who);
  DEW_REQUIRE(tokens >= 0 && layer->router.top_k >= 1 && layer->router.experts >= 1, "%s: %d tokens, %d of %d experts", who, tokens,
              layer->router.top_k, layer->router.experts);
  const int64_t rows = static_cast<int64_t>(tokens) * (layer->router.top_k + (layer->shared ? 1 : 0));
  DEW_REQUIRE(rows < (1ll << 30), "%s: %lld rows overflow int32", who, static_cast<long long>(rows));
  const int groups = layer->router.experts + (layer->shared ? 1 : 0);
  DEW_REQUIRE(gate->experts == groups && down->experts == groups, "%s: banks of %d and %d experts for %d groups", who, gate->experts,
              down->experts, groups);
  const int hidden_width = interleaved ? gate->width / 2 : gate->width;
  DEW_REQUIRE(down->depth == hidden_width && down->width == gate->depth, "%s: down [%d, %d] does not follow gate [%d, %d]", who, down->depth,
              down->width, gate->depth, gate->width);
  DEW_REQUIRE(!interleaved || gate->width % 64 == 0, "%s: interleaved columns %d are not whole atoms of pairs", who, gate->width);
  DEW_REQUIRE(down->width % 8 == 0, "%s: outputs %d wide", who, down->width);
  return DEW_MOE_OK;
}

}  // namespace dew

extern "C" size_t dew_moe_layer_workspace_bytes(const dew_moe_layer* layer, const dew_moe_bank* gate, const dew_moe_bank* up,
                                                const dew_moe_bank* down, int32_t tokens, int32_t split_terms, int32_t f16_rows_from) {
  using namespace dew;
  if (check_layer("dew_moe_layer_workspace_bytes", layer, gate, up, down, tokens) != DEW_MOE_OK) return 0;
  const int rows = tokens * (layer->router.top_k + (layer->shared ? 1 : 0));
  return layer_workspace(layer, gate, down, tokens, layer_form(layer, gate, up, down, rows, split_terms, f16_rows_from)).bytes;
}

extern "C" int dew_moe_layer_forward(const dew_moe_layer* layer, const void* x, const float* gate_kernel, const float* gate_bias,
                                     const float* selection_bias, const dew_moe_bank* gate, const dew_moe_bank* up, const dew_moe_bank* down,
                                     const float* up_bias, const float* down_bias, int32_t tokens, int32_t split_terms,
                                     int32_t f16_rows_from, void* out, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace dew;
  const char* who = "dew_moe_layer_forward";
  if (int rc = check_layer(who, layer, gate, up, down, tokens)) return rc;
  if (tokens == 0) return DEW_MOE_OK;
  const int experts = layer->router.experts, top_k = layer->router.top_k;
  const int slots_count = tokens * top_k, rows = slots_count + (layer->shared ? tokens : 0);
  const LayerForm form = layer_form(layer, gate, up, down, rows, split_terms, f16_rows_from);
  const LayerWorkspace w = layer_workspace(layer, gate, down, tokens, form);
  DEW_REQUIRE(x && gate_kernel && out, "%s: x, the gate kernel and out must not be null", who);
  DEW_REQUIRE(workspace && workspace_bytes >= w.bytes, "%s: workspace of %zu bytes, need %zu (dew_moe_layer_workspace_bytes)", who,
              workspace_bytes, w.bytes);
  uint8_t* base = reinterpret_cast<uint8_t*>((reinterpret_cast<uintptr_t>(workspace) + 255) & ~static_cast<uintptr_t>(255));
  auto words = [base](size_t at) { return reinterpret_cast<int32_t*>(base + at); };
  float* logits = reinterpret_cast<float*>(base + w.logits);
  float* weights = reinterpret_cast<float*>(base + w.weights);
  int32_t *indices = words(w.indices), *sizes = words(w.sizes), *offsets = words(w.offsets), *order = words(w.order), *gather = words(w.rows);
  // a decode step's or a short prompt's gate leaves its logits in shares, which spread over more CUs and which its router adds up
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const bool in_shares = logit_shares(tokens, gate->depth, experts) != kNoShares && aligned16(x);
  if (int rc = in_shares ? router_logit_shares(x, gate_kernel, logits, tokens, gate->depth, experts, s)
                         : dew_moe_router_logits(x, gate_kernel, gate_bias, logits, tokens, gate->depth, experts, stream))
    return rc;
  if (in_shares && tokens <= kRouteAndSortTokens && rows <= kSmallSlots) {
    if (int rc = route_and_sort(&layer->router, logits, gate_bias, selection_bias, tokens, layer->shared != 0, weights, sizes, offsets, order, gather, s))
      return rc;
  } else {
    if (int rc = in_shares ? route_shares(&layer->router, logits, gate_bias, selection_bias, tokens, weights, indices, s)
                           : dew_moe_route_with(&layer->router, logits, selection_bias, tokens, weights, indices, nullptr, nullptr, stream))
      return rc;
    if (int rc = layer->shared ? dew_moe_permute_shared(indices, tokens, top_k, experts, tokens, sizes, offsets, order, gather, base + w.sort,
                                                        w.sort_bytes, stream)
                               : dew_moe_permute(indices, tokens, top_k, experts, sizes, offsets, order, gather, base + w.sort, w.sort_bytes, stream))
      return rc;
  }
  uint8_t* slots = base + w.slots;
  if (form == kRowsSplit) {
    if (int rc = dew_moe_gated_mlp_split(x, tokens, gather, offsets, nullptr, gate, up, down, layer->gating, layer->limit, order, slots, rows,
                                         split_terms, base + w.split, w.split_bytes, stream))
      return rc;
  } else {
    uint8_t* hidden = base + w.hidden;
    if (layer->gating == DEW_MOE_GATE_INTERLEAVED) {
      if (int rc = dew_moe_gateup_interleaved(x, gather, offsets, gate, up_bias, layer->limit, hidden, rows, stream)) return rc;
    } else if (form == kRowsF16) {
      uint8_t* x_rows = base + w.x_rows;
      uint8_t* x_scale = base + w.x_scale;
      if (int rc = dew_moe_rows_f16(x, x_rows, x_scale, tokens, gate->depth, stream)) return rc;
      if (int rc = dew_moe_gateup_gated_f16(x_rows, x_scale, gather, offsets, nullptr, gate, up, layer->gating, layer->limit, hidden, rows, stream))
        return rc;
    } else {
      if (int rc = dew_moe_gateup_gated(x, gather, offsets, nullptr, gate, up, layer->gating, layer->limit, hidden, rows, stream)) return rc;
    }
    if (combines_few(down, tokens, top_k, layer->shared != 0))
      return down_and_combine(who, hidden, offsets, down, down_bias, order, weights, tokens, top_k, layer->shared != 0, out, s);
    if (int rc = dew_moe_grouped_gemm_param_bias(hidden, nullptr, offsets, nullptr, down, down_bias, order, slots, rows, stream)) return rc;
  }
  const void* addend = layer->shared ? slots + static_cast<size_t>(slots_count) * down->width * 2 : nullptr;
  return dew_moe_combine(slots, weights, addend, out, tokens, top_k, down->width, stream);
}
