"""A layer's pass as one foreign call against its separate calls, bit for bit: the same launches on the same operands, but that a few tokens' router
and sort, and small experts' down product and combine, are one launch each there, which form every sum in the same order."""

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = {
    "fp8 blocks, one token": dict(tokens=1, experts=16, top_k=3, quant="fp8_block"),
    "fp8 blocks, one token, every expert": dict(tokens=1, experts=8, top_k=8, quant="fp8_block"),
    "fp8 channels": dict(tokens=77, experts=8, top_k=5, quant="fp8_channel"),
    "fp8 blocks, past the small sort": dict(tokens=1500, experts=64, top_k=7, quant="fp8_block"),
    "bf16, geglu, clamped": dict(tokens=130, experts=8, top_k=2, quant="bf16", activation="geglu", swiglu_limit=1.5),
    "nvfp4, bf16 rows": dict(tokens=20, experts=8, top_k=2, quant="nvfp4"),
    "nvfp4, f16 rows": dict(tokens=300, experts=8, top_k=4, quant="nvfp4"),
    "mxfp4, split rows": dict(tokens=1600, experts=8, top_k=2, quant="mxfp4"),
    "groups, bias, shared": dict(tokens=33, experts=64, top_k=8, quant="fp8_block", score_function="sigmoid", routed_scaling_factor=2.5,
                                 expert_groups=8, groups_per_token=4, expert_bias=True, shared=256),
    "groups, bias, shared, 16 tokens": dict(tokens=16, experts=64, top_k=8, quant="fp8_block", score_function="sigmoid",
                                            expert_groups=8, groups_per_token=4, expert_bias=True, shared=256),
    "groups, bias, shared, 65 tokens": dict(tokens=65, experts=64, top_k=8, quant="fp8_block", score_function="sigmoid",
                                            expert_groups=8, groups_per_token=4, expert_bias=True, shared=256),
    # the gate's shares by tiles: 105 of 32 x 32, neither extent whole; and one tile short of, at and past the lines at 64 and 112
    "shares by tiles": dict(tokens=1111, experts=70, top_k=2, quant="fp8_block"),
    "shares, 63 tiles": dict(tokens=2016, experts=32, top_k=2, quant="fp8_block"),
    "shares, 111 tiles": dict(tokens=1184, experts=96, top_k=1, quant="fp8_block"),
    "no shares, 112 tiles": dict(tokens=1792, experts=64, top_k=1, quant="fp8_block"),
    # the down product and the combine in one launch, in every format, with a shared expert, at the most slots and tokens
    "combined, fp8 channels, 16 tokens": dict(tokens=16, experts=8, top_k=8, quant="fp8_channel"),
    "combined, bf16, shared": dict(tokens=3, experts=8, top_k=3, quant="bf16", shared=256),
    "combined, mxfp4, one slot": dict(tokens=5, experts=16, top_k=1, quant="mxfp4"),
    "combined, nvfp4, shared, 70 experts": dict(tokens=16, experts=70, top_k=7, quant="nvfp4", shared=256),
    # ... and through whole rounds of its weight registers: from 1024 depths on in FP8 and FP4, 768 in bf16
    "combined, fp8 blocks, two slots, 16 steps": dict(tokens=3, experts=8, top_k=2, quant="fp8_block", hidden=1024),
    "combined, fp8 channels, one slot, 36 steps": dict(tokens=7, experts=8, top_k=1, quant="fp8_channel", hidden=2304),
    "combined, bf16, one slot, 17 steps": dict(tokens=5, experts=8, top_k=1, quant="bf16", hidden=1088),
    "combined, mxfp4, one slot, 67 steps": dict(tokens=5, experts=8, top_k=1, quant="mxfp4", hidden=4288),
    "combined, nvfp4, shared, 20 steps": dict(tokens=4, experts=8, top_k=2, quant="nvfp4", hidden=1280, shared=1280),
    "300 experts": dict(tokens=64, experts=300, top_k=6, quant="fp8_block"),
}
DEPTH, HIDDEN = 512, 256


def bank(experts, depth, width, quant, generator):
    from dew_amd import codecs, formats

    w = torch.randn((experts, depth, width), generator=generator, device="cuda") * 0.05
    if quant == "mxfp4":
        return formats.Mxfp4Blocks(*codecs.quantize_mxfp4(w))
    if quant == "bf16":
        return formats.Bf16(w.to(torch.bfloat16))
    return {"fp8_block": formats.Fp8Blocks, "fp8_channel": formats.Fp8Channels, "nvfp4": formats.NvFp4}[quant].quantized(w)


@pytest.mark.parametrize("name", CASES)
def test_one_call_returns_the_separate_calls_bits(name):
    from dew_amd import _lib, gemm, moe

    case = dict(CASES[name])
    tokens, experts, top_k, quant = (case.pop(key) for key in ("tokens", "experts", "top_k", "quant"))
    hidden = case.pop("hidden", HIDDEN)
    layer = moe.SparseMLP(num_experts=experts, top_k=top_k, hidden_features=hidden, out_features=DEPTH, **case)
    generator = torch.Generator("cuda").manual_seed(7)
    shapes = {"gate_proj": (DEPTH, hidden), "up_proj": (DEPTH, hidden), "down_proj": (hidden, DEPTH)}
    held = {"experts": {n: {"kernel": bank(experts, *s, quant, generator)} for n, s in shapes.items()}}
    if case.get("shared"):
        held["shared_experts"] = {n: {"kernel": bank(1, *s, quant, generator)} for n, s in shapes.items()}
    if name.startswith("combined"):
        assert _lib.library().dew_moe_combines_few(gemm.prepared(held["experts"]["down_proj"]["kernel"]).descriptor, tokens, top_k, "shared" in case) == 1
    variables = {"params": {"gate": {"kernel": torch.randn((DEPTH, experts), generator=generator, device="cuda") * DEPTH ** -0.5}},
                 "moe": {"gate": {"e_score_correction_bias": torch.randn(experts, generator=generator, device="cuda") * 0.05}},
                 "quantization": held}
    x = torch.randn((tokens, DEPTH), generator=generator, device="cuda").to(torch.bfloat16)
    want = layer._bound(variables, ())(x)
    got = layer._applied(variables, x)
    assert got is not None and torch.equal(got, want) and bool(got.any())
    shaped = x[None].expand(2, -1, -1)                                     # (not contiguous: the separate calls answer)
    assert layer._applied(variables, shaped) is None
    separate = layer._bound(variables, ())
    assert torch.equal(layer.apply(variables, shaped), separate(torch.stack((x, x))))
    # twice the tokens take other tiles, which sum alike: the same bits from the same logits (whose own sums' order, in the gate, goes by
    # the number of tokens)
    logits = separate.gate.logits(x)
    assert torch.equal(layer.apply(variables, shaped, logits=torch.stack((logits, logits))), torch.stack((want, want)))


@pytest.mark.parametrize("tokens,hidden", ((1, 192), (24, 192), (700, 192), (3, 1024)))     # (the last: 16 steps of the combined launch)
def test_gpt_oss_in_one_call(tokens, hidden):
    from dew_amd import gpt_oss

    generator = torch.Generator("cuda").manual_seed(8)
    depth, experts = 320, 8
    layer = gpt_oss.GptOssMLP(depth, hidden, experts, 4)
    normal = lambda *shape: torch.randn(shape, generator=generator, device="cuda")
    variables = {"params": {"router": {"kernel": normal(depth, experts) * 0.1, "bias": normal(experts) * 0.1},
                            "experts": {"gate_up_proj_bias": normal(experts, 2 * hidden) * 0.1, "down_proj_bias": normal(experts, depth) * 0.1}},
                 "quantization": {"experts": {"gate_up_proj": bank(experts, depth, 2 * hidden, "mxfp4", generator),
                                              "down_proj": bank(experts, hidden, depth, "mxfp4", generator)}}}
    x = normal(tokens, depth).to(torch.bfloat16)
    want = layer._bound(variables, ())(x)
    got = layer._applied(variables, x)
    assert got is not None and torch.equal(got, want) and bool(got.any())


def test_what_the_one_call_does_not_cover_goes_to_the_separate_calls():
    from dew_amd import moe, selection

    layer = moe.SparseMLP(num_experts=8, top_k=2, hidden_features=HIDDEN, out_features=DEPTH)
    assert layer._one_call is not None
    for option in (dict(capacity_factor=1.0), dict(fused=False), dict(scale_inputs=True), dict(implementation="hip"), dict(activation="relu2"),
                   dict(shared=128), dict(shared_gate=True, shared=HIDDEN), dict(latent_features=128)):
        assert moe.SparseMLP(**{**dict(num_experts=8, top_k=2, hidden_features=HIDDEN, out_features=DEPTH), **option})._one_call is None
    generator = torch.Generator("cuda").manual_seed(9)
    held = {"experts": {n: {"kernel": bank(8, *s, "fp8_block", generator)} for n, s in
                        {"gate_proj": (DEPTH, HIDDEN), "up_proj": (DEPTH, HIDDEN), "down_proj": (HIDDEN, DEPTH)}.items()}}
    variables = {"params": {"gate": {"kernel": torch.randn((DEPTH, 8), generator=generator, device="cuda")}}, "quantization": held}
    x = torch.randn((4, DEPTH), generator=generator, device="cuda")
    assert layer._applied(variables, x) is None and layer._applied(variables, x.to(torch.bfloat16)[:, :256].contiguous()) is None
    with selection.chosen(grouped_matmul="hip"):
        assert layer._applied(variables, x.to(torch.bfloat16)) is None
    with pytest.raises(RuntimeError, match="bfloat16"):
        layer.apply(variables, x)          # fp32 tokens: refused by the separate calls, by name
