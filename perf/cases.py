"""The work a program built on this package has it do, as cases that can be timed: an expert layer's forward pass when a model
serves (one token to a long prompt, every weight format), and the grouped products of a training step, forward and both
gradients, in each recipe. Everything goes through the package's public entry points with the operands such a program holds:
activations and gate kernels as they are, expert banks in their checkpoint's format with their one-time layout made at load.

`listed()` names the fixed cases, `draw(rng)` gives another one of the same ranges; `prepare` makes a case's inputs on the GPU,
`run` is one pass, `work` what a pass cannot do without and `tolerance` what another correct implementation may differ by."""

import math

import torch

from dew_amd import codecs, formats, gemm, gpt_oss, moe, projections

DEEPSEEK_ROUTER = dict(score_function="sigmoid", routed_scaling_factor=2.5, expert_groups=8, groups_per_token=4, expert_bias=True)
MOST_FLOPS = 12.0e12
"""No drawn case does more than the largest listed ones."""
MOST_WEIGHTS = {"layer": 1.5e9, "gpt_oss": 1.5e9, "train": 4.7e8}


def listed():
    return [
        # Serving, decode: one sequence's next token through a layer of many small experts. Launches and host work.
        layer("decode, 1 token, fp8", tokens=1, model=2048, hidden=768, experts=128, top_k=8, quant="fp8_block"),
        # Serving, decode: a batch of sequences on the same layer; nearly every expert is read for half a dozen rows.
        layer("decode, 64 tokens, fp8", tokens=64, model=2048, hidden=768, experts=128, top_k=8, quant="fp8_block"),
        # Serving, decode: GPT-OSS's layer (biased router, interleaved gate and up, 2880 wide) on a checkpoint's MXFP4 bytes.
        oss("decode, 24 tokens, gpt-oss mxfp4", tokens=24, model=2880, hidden=2880, experts=32, top_k=4),
        # Serving, a prompt on a small model's experts, one scale a channel.
        layer("prompt, 2048 tokens, small fp8", tokens=2048, model=512, hidden=1024, experts=8, top_k=2, quant="fp8_channel"),
        # Serving, a chunk of a prompt of no round length on unquantized experts.
        layer("prompt, 1111 tokens, bf16", tokens=1111, model=2048, hidden=1408, experts=64, top_k=6, quant="bf16"),
        # Serving, long prompts on large experts: MXFP4, DeepSeek-V3's layer (group-limited router, shared expert), NVFP4.
        layer("prompt, 16384 tokens, mxfp4", tokens=16384, model=4096, hidden=14336, experts=8, top_k=2, quant="mxfp4"),
        layer("prompt, 8192 tokens, deepseek fp8", tokens=8192, model=7168, hidden=2048, experts=256, top_k=8, quant="fp8_block",
              router="deepseek", shared=True),
        layer("prompt, 4096 tokens, nvfp4", tokens=4096, model=4096, hidden=14336, experts=8, top_k=2, quant="nvfp4"),
        # Training: one expert projection, forward and both gradients, groups of any sizes on unquantized matrices ...
        step("train, bf16", recipe="bf16", tokens=10007, depth=2048, width=4096, groups=16),
        # ... and in the low-precision recipes, whose matrices are new (and quantized anew) at every step.
        step("train, blockwise fp8", recipe="blockwise_fp8", tokens=32768, depth=7168, width=2048, groups=32),
        step("train, mxfp8", recipe="mxfp8", tokens=32768, depth=4096, width=14336, groups=8),
        step("train, nvfp4", recipe="nvfp4", tokens=8192, depth=2048, width=4096, groups=8),
    ]


def layer(name, *, tokens, model, hidden, experts, top_k, quant, router="softmax", shared=False):
    return dict(name=name, kind="layer", tokens=tokens, model=model, hidden=hidden, experts=experts, top_k=top_k, quant=quant,
                router=router, shared=shared)


def oss(name, *, tokens, model, hidden, experts, top_k):
    return dict(name=name, kind="gpt_oss", tokens=tokens, model=model, hidden=hidden, experts=experts, top_k=top_k)


def step(name, *, recipe, tokens, depth, width, groups):
    return dict(name=name, kind="train", recipe=recipe, tokens=tokens, depth=depth, width=width, groups=groups)


def draw(rng):
    """A case of the listed ones' ranges: 1 to 16384 tokens in a layer of 8 to 256 experts 512 to 7168 wide, any format; or a
    training step of 512 to 32768 tokens in 1 to 64 groups, any recipe."""
    def spread(low, high, unit=1):
        return max(low, min(high, unit * round(math.exp(rng.uniform(math.log(low), math.log(high))) / unit)))

    while True:
        kind = rng.choices(("layer", "gpt_oss", "train"), (6, 1, 3))[0]
        if kind == "train":
            recipe = rng.choice(("bf16", "blockwise_fp8", "mxfp8", "nvfp4"))
            unit = 256 if recipe == "nvfp4" else 128     # (NVFP4's block stages; both extents are a depth in one of the products)
            case = step("", recipe=recipe, tokens=spread(512, 32768, 1 if recipe == "bf16" else 128), depth=spread(512, 7168, unit),
                        width=spread(512, 14336, unit), groups=spread(1, 64))
        else:
            experts = rng.choice((8, 16, 32, 64, 128, 256))
            sizes = dict(tokens=spread(1, 16384), experts=experts, top_k=rng.randint(1, min(8, experts // 2)))
            if kind == "gpt_oss":
                case = oss("", model=spread(512, 4096, 64), hidden=spread(512, 4096, 64), **sizes)
            else:
                quant = rng.choice(("fp8_channel", "fp8_block", "mxfp4", "nvfp4", "bf16"))
                unit = 256 if quant == "nvfp4" else 128
                router = rng.choice(("softmax", "softmax", "deepseek")) if experts >= 64 else "softmax"
                case = layer("", quant=quant, router=router, shared=router == "deepseek" and rng.random() < 0.5,
                             model=spread(512, 7168, unit), hidden=spread(512, 14336, unit), **sizes)
        del case["name"]
        if work(case)["flops"] <= MOST_FLOPS and weights(case) <= MOST_WEIGHTS[kind]:
            return case


def weights(case):
    """The elements of a case's matrices."""
    if case["kind"] == "train":
        return case["groups"] * case["depth"] * case["width"]
    return 3 * (case["experts"] + bool(case.get("shared"))) * case["model"] * case["hidden"]


# ---- inputs -----------------------------------------------------------------------------------------------


def prepare(case, seed):
    device = torch.device("cuda")
    generator = torch.Generator(device=device).manual_seed(seed)

    def normal(*shape, scale=1.0):
        return torch.randn(shape, generator=generator, device=device, dtype=torch.float32).mul_(scale)

    if case["kind"] == "train":
        return prepare_step(case, normal, generator)
    tokens, model, hidden, experts = case["tokens"], case["model"], case["hidden"], case["experts"]
    # Hidden states share a mean, so that a gate favours some experts (by half a logit, one standard deviation) as trained ones do.
    x = (normal(tokens, model) + normal(1, model, scale=0.5)).to(torch.bfloat16)
    gate = normal(model, experts, scale=model ** -0.5)

    def bank(count, depth, width, quant):
        at_once = max(1, int(6e7 // (depth * width)))
        parts = [quantized(normal(min(at_once, count - first), depth, width, scale=0.02), quant) for first in range(0, count, at_once)]
        return joined(parts)

    if case["kind"] == "gpt_oss":
        mlp = gpt_oss.GptOssMLP(model, hidden, experts, case["top_k"])
        banks = {"gate_up_proj": bank(experts, model, 2 * hidden, "mxfp4"), "down_proj": bank(experts, hidden, model, "mxfp4")}
        for held in banks.values():
            gemm.prepared(held)
        variables = {"params": {"router": {"kernel": gate, "bias": normal(experts, scale=0.1)},
                                "experts": {"gate_up_proj_bias": normal(experts, 2 * hidden, scale=0.02),
                                            "down_proj_bias": normal(experts, model, scale=0.02)}},
                     "quantization": {"experts": banks}}
        return dict(case=case, layer=mlp, variables=variables, x=x)

    deepseek = case["router"] == "deepseek"
    mlp = moe.SparseMLP(num_experts=experts, top_k=case["top_k"], hidden_features=hidden, out_features=model,
                        shared=hidden if case["shared"] else None, **(DEEPSEEK_ROUTER if deepseek else {}))
    shapes = {"gate_proj": (model, hidden), "up_proj": (model, hidden), "down_proj": (hidden, model)}
    routed = {name: bank(experts, *shape, case["quant"]) for name, shape in shapes.items()}
    held = {"experts": {name: {"kernel": b} for name, b in routed.items()}}
    if case["shared"]:
        shared = {name: bank(1, *shape, case["quant"]) for name, shape in shapes.items()}
        held["shared_experts"] = {name: {"kernel": b} for name, b in shared.items()}
        moe.with_shared_expert(tuple(routed.values()), tuple(shared.values()))
    else:
        for b in routed.values():
            gemm.prepared(b)
    variables = {"params": {"gate": {"kernel": gate}}, "quantization": held}
    if deepseek:
        variables["moe"] = {"gate": {"e_score_correction_bias": normal(experts, scale=0.05)}}
    return dict(case=case, layer=mlp, variables=variables, x=x)


def prepare_step(case, normal, generator):
    tokens, depth, width, groups = case["tokens"], case["depth"], case["width"], case["groups"]
    # The groups' shares of the rows vary as a router's choices do; a recipe's groups are padded to whole 128-row blocks.
    rows = 1 if case["recipe"] == "bf16" else 128
    share = torch.softmax(torch.randn(groups, generator=generator, device="cuda") * 0.3, 0)
    ends = (share.cumsum(0) * (tokens // rows)).round().to(torch.int32)
    ends[-1] = tokens // rows
    sizes = torch.diff(ends, prepend=ends.new_zeros(1)).contiguous()
    w = torch.empty((groups, depth, width), dtype=torch.bfloat16, device="cuda")
    for g in range(groups):
        w[g] = normal(depth, width, scale=0.02)
    return dict(case=case, x=normal(tokens, depth).to(torch.bfloat16), w=w, dy=normal(tokens, width, scale=0.1).to(torch.bfloat16), sizes=sizes)


def quantized(weight, quant):
    if quant == "fp8_block":
        return formats.Fp8Blocks.quantized(weight)
    if quant == "fp8_channel":
        return formats.Fp8Channels.quantized(weight)
    if quant == "nvfp4":
        return formats.NvFp4.quantized(weight)
    if quant == "mxfp4":
        return formats.Mxfp4Blocks(*codecs.quantize_mxfp4(weight))
    return formats.Bf16(weight.to(torch.bfloat16))


def joined(parts):
    return parts[0] if len(parts) == 1 else formats.stacked(parts)


# ---- a pass -----------------------------------------------------------------------------------------------


GRADIENTS = {"blockwise_fp8": (projections.blockwise_fp8_projection, projections.blockwise_fp8_gradients),
             "mxfp8": (projections.mxfp8_projection, projections.mxfp8_gradients),
             "nvfp4": (projections.nvfp4_projection, projections.nvfp4_gradients)}


def run(state):
    case, x = state["case"], state["x"]
    if case["kind"] != "train":
        return state["layer"].apply(state["variables"], x)
    w, dy, sizes = state["w"], state["dy"], state["sizes"]
    if case["recipe"] == "bf16":
        return gemm.gemm(x, w, sizes), gemm.gemm(dy, w.transpose(1, 2), sizes), gemm.gemm_t(x, dy, sizes)
    forward, gradients = GRADIENTS[case["recipe"]]
    return forward(x, w, sizes), *gradients(x, w, dy, sizes)


BYTES_A_WEIGHT = {"fp8_block": 1.0, "fp8_channel": 1.0, "mxfp4": 0.5 + 1 / 32, "nvfp4": 0.5 + 1 / 16, "bf16": 2.0}


def work(case):
    if case["kind"] == "train":
        tokens, depth, width = case["tokens"], case["depth"], case["width"]
        operands = 2.0 * (tokens * depth + tokens * width + weights(case))
        return {"bytes": 2 * operands, "flops": 3 * 2.0 * tokens * depth * width}      # x, dy, w in; d_x, y, d_w out
    tokens, model, hidden, experts, top_k = (case[k] for k in ("tokens", "model", "hidden", "experts", "top_k"))
    shared = 1 if case.get("shared") else 0
    touched = experts * (1 - (1 - top_k / experts) ** tokens) + shared
    a_weight = BYTES_A_WEIGHT["mxfp4" if case["kind"] == "gpt_oss" else case["quant"]]
    return {"bytes": touched * 3 * model * hidden * a_weight + 2 * tokens * model * 2 + model * experts * 4,
            "flops": 6.0 * tokens * (top_k + shared) * model * hidden + 2.0 * tokens * model * experts}


def tolerance(case):
    """Operands and results in bf16 (the recipes' products included): one rounding of the result, and in a layer the hidden rows'."""
    return {"rel": 1e-2}
