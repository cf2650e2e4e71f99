"""A recipe's weight matrices quantized straight into their prepared bank, against the same matrices quantized by the
whole-tensor rules (which the oracle's tests pin) and then prepared: the same bytes."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dew_amd import ops

    ops.device_check()
    return ops


def by_whole_tensors(recipe, w):
    from dew_amd import formats, projections

    quantized = {"blockwise_fp8": projections.blocks_quantized, "mxfp8": formats.MxFp8.quantized, "nvfp4": projections.nvfp4_matrices}
    return quantized[recipe](w)


@pytest.mark.parametrize("turned", [False, True], ids=["natural", "kmajor"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("recipe", ["blockwise_fp8", "mxfp8", "nvfp4"])
@pytest.mark.parametrize("shape", [(1, 256, 128), (3, 512, 384), (2, 256, 1152)])   # one tile of columns; several; more tiles than a row of them
def test_the_bank_is_the_quantized_matrices_prepared(ops, recipe, dtype, turned, shape):
    experts, depth, width = shape
    generator = torch.Generator(device="cuda").manual_seed(depth + width)
    w = torch.randn((experts, depth, width), generator=generator, device="cuda") * torch.exp2(
        torch.randint(-12, 6, (experts, depth // 16, width), generator=generator, device="cuda").float()).repeat_interleave(16, 1)
    w[0, :128, :128] = 0.0                      # a block of zeros, signed zeros beside values, a block of subnormals
    w[-1, 128:144, ::3] = -0.0
    w[-1, 144:176, 5] = 2.0 ** -133
    w = w.to(dtype)
    got = ops.quantize_matrices(w.transpose(1, 2).contiguous().transpose(1, 2) if turned else w, recipe)
    want = ops.prepare(by_whole_tensors(recipe, w))
    assert got.shape == want.shape == shape
    elements = experts * depth * width
    compared = elements // 2 + elements // 16 if recipe == "nvfp4" else want.keep[0].numel()
    assert torch.equal(got.keep[0][:compared], want.keep[0][:compared])
    if recipe == "nvfp4":
        assert torch.equal(got.keep[2], want.keep[2])


@pytest.mark.parametrize("recipe", ["blockwise_fp8", "mxfp8", "nvfp4"])
def test_a_nan_in_the_matrices_reaches_the_product(ops, recipe):
    from dew_amd import projections

    w = torch.ones((1, 256, 256), dtype=torch.bfloat16, device="cuda")
    w[0, 37, 200] = float("nan")
    x = torch.ones((128, 256), dtype=torch.bfloat16, device="cuda")
    out = projections.recipe_projection(x, w, recipe=recipe)
    assert out[:, 200].isnan().all()


@pytest.mark.parametrize("groups", [1, 63, 64, 65, 1000])
def test_block_offsets(ops, groups):
    blocks = torch.randint(0, 9, (groups,), generator=torch.Generator().manual_seed(groups), dtype=torch.int32).cuda()
    want = torch.cat([torch.zeros(1, dtype=torch.int64), blocks.cpu().long().cumsum(0) * 128])
    assert torch.equal(ops.block_offsets(blocks, 128).cpu().long(), want)
    assert torch.equal(ops.group_offsets(blocks).cpu().long() * 128, want)


def test_what_cannot_be_quantized_is_refused(ops):
    for w, recipe in ((torch.zeros((1, 128, 64), dtype=torch.bfloat16, device="cuda"), "mxfp8"),
                      (torch.zeros((1, 128, 128), dtype=torch.float16, device="cuda"), "mxfp8"),
                      (torch.zeros((1, 128, 128), dtype=torch.bfloat16, device="cuda"), "fp8"),
                      (torch.zeros((1, 128, 128), dtype=torch.bfloat16), "mxfp8")):
        with pytest.raises(ops.KernelError):
            ops.quantize_matrices(w, recipe)
