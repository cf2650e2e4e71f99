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


@pytest.mark.parametrize("turned", [False, True], ids=["natural", "kmajor"])
def test_matrices_that_no_cache_holds(ops, turned):
    """NVFP4's loads are others past 256 MB: every copy of a matrix has the codes and scales that it has alone."""
    one = torch.randn((1, 2048, 2048), generator=torch.Generator("cuda").manual_seed(1), device="cuda").to(torch.bfloat16)
    quantized = lambda w: ops.quantize_matrices(w.transpose(1, 2).contiguous().transpose(1, 2) if turned else w, "nvfp4").keep[0]
    alone, bytes_of = quantized(one), one.numel() // 2
    for copies in (32, 33):
        got = quantized(one.expand(copies, -1, -1).contiguous())
        assert bool((got[:copies * bytes_of].view(copies, -1) == alone[:bytes_of]).all())
        assert bool((got[copies * bytes_of:copies * bytes_of * 9 // 8].view(copies, -1) == alone[bytes_of:bytes_of * 9 // 8]).all())


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


@pytest.mark.parametrize("groups", [1, 64, 65, 1000])
@pytest.mark.parametrize("recipe", ["blockwise_fp8", "mxfp8", "nvfp4"])
@pytest.mark.parametrize("turned", [False, True])
def test_a_steps_launch_leaves_its_groups_offsets(ops, recipe, groups, turned):
    blocks = torch.randint(0, 9, (groups,), generator=torch.Generator().manual_seed(groups), dtype=torch.int32).cuda()
    w = torch.randn((3, 256, 512), device="cuda", generator=torch.Generator("cuda").manual_seed(groups)).to(torch.bfloat16)
    w = w.transpose(1, 2).contiguous().transpose(1, 2) if turned else w
    of_x, of_w, of_wide = ops.nvfp4_largest_of(w[0].contiguous() * 3, w, w.float())
    assert torch.equal(of_w, ops.nvfp4_largest(w.contiguous() if not turned else w.transpose(1, 2))) and int(of_wide.max()) == int(of_w.max())
    assert int(of_x.max()) == int(ops.nvfp4_largest(w[0].contiguous() * 3).max())
    bank, offsets = ops.quantize_matrices(w, recipe, largest=of_w if recipe == "nvfp4" else None, blocks=blocks)
    assert torch.equal(offsets, ops.block_offsets(blocks, 128))
    want = ops.quantize_matrices(w, recipe)
    compared = w.numel() // 2 + w.numel() // 16 if recipe == "nvfp4" else want.keep[0].numel()     # (behind NVFP4's codes and scales: partials)
    assert torch.equal(bank.keep[0][:compared], want.keep[0][:compared])
    if recipe == "nvfp4":
        assert torch.equal(bank.keep[2], want.keep[2])


def test_what_cannot_be_quantized_is_refused(ops):
    for w, recipe in ((torch.zeros((1, 128, 64), dtype=torch.bfloat16, device="cuda"), "mxfp8"),
                      (torch.zeros((1, 128, 128), dtype=torch.float16, device="cuda"), "mxfp8"),
                      (torch.zeros((1, 128, 128), dtype=torch.bfloat16, device="cuda"), "fp8"),
                      (torch.zeros((1, 128, 128), dtype=torch.bfloat16), "mxfp8")):
        with pytest.raises(ops.KernelError):
            ops.quantize_matrices(w, recipe)


@pytest.mark.parametrize("exponent", [0, -79, 60, -100], ids=["ones", "least", "large", "past"])   # the tensor scale in and (2^-100) out of the range of the short form
def test_every_significand_against_every_tensor_scale(ops, exponent):
    """NVFP4's quotients of bf16 values come from reciprocals and a Newton step. Every significand of the largest magnitude (21 / 16
    and its like, whose tensor scales make most thresholds exact ties) with every significand as a block's largest, and values of
    every significand and a dozen binades below, in each of the four launches that choose codes."""
    from dew_amd import codecs

    e2m1 = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, -0.0, -0.5, -1, -1.5, -2, -3, -4, -6], device="cuda")
    generator = torch.Generator(device="cuda").manual_seed(exponent + 200)
    significands = 1 + torch.arange(128, device="cuda") / 128
    for first in range(0, 128, 8):
        for largest in significands[first:first + 8].tolist():
            tops = largest * torch.exp2(-torch.randint(0, 11, (64, 128), generator=generator, device="cuda").float())
            tops = torch.minimum(tops * significands / 2, torch.tensor(largest, device="cuda"))
            values = tops[:, :, None] * torch.exp2(-torch.randint(0, 12, (64, 128, 16), generator=generator, device="cuda").float())
            values *= significands[torch.randint(0, 128, (64, 128, 16), generator=generator, device="cuda")] / 2
            values *= torch.randint(0, 2, (64, 128, 16), generator=generator, device="cuda") * 2 - 1
            values[:, :, 3] = tops
            values[0, 0, 3] = largest
            x = (values.reshape(256, 512) * 2.0 ** exponent).to(torch.bfloat16)     # [tokens or width, depth], blocks of 16 along the depth
            w = x.t()[None]                                                         # [1, 512, 256], held K-major
            want = ops.prepare(by_whole_tensors("nvfp4", w))
            compared = x.numel() // 2 + x.numel() // 16
            for held in (w, w.contiguous()):
                got = ops.quantize_matrices(held, "nvfp4")
                assert torch.equal(got.keep[0][:compared], want.keep[0][:compared]) and torch.equal(got.keep[2], want.keep[2])
            codes, scales, _ = codecs.nvfp4_coded(w[0].float())
            decoded = (e2m1[codes.long()] * scales.view(torch.float8_e4m3fn).float().repeat_interleave(16, 0)).t()
            rows, scale = ops.quantize_rows_nvfp4(x.contiguous())
            assert scale.item() == want.keep[2][0].item() and torch.equal(rows.float(), decoded)
            columns, scale = ops.transpose_columns(x.t().contiguous(), nvfp4=True, as_bank=False)
            assert scale.item() == want.keep[2][0].item() and torch.equal(columns.float(), decoded)


def test_nans_and_infinities_among_nvfp4_operands(ops):
    """An operand that holds a NaN has the tensor scale 1. In the rows' and columns' blocks the NaN itself reads as a zero and the rest
    as ever, an infinity as the block's largest code under the largest scale; a block of matrices with a NaN has no scale."""
    from dew_amd import codecs

    nan, inf, e2m1 = float("nan"), float("inf"), torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, -0.0, -0.5, -1, -1.5, -2, -3, -4, -6], device="cuda")
    generator = torch.Generator(device="cuda").manual_seed(11)
    x = torch.randn((128, 256), generator=generator, device="cuda").to(torch.bfloat16)
    x[0, 160], x[5, 16:32], x[7, 3], x[7, 4], x[9, 40], x[11, 50] = nan, nan, inf, nan, -inf, inf
    finite = torch.where(x.isnan(), 0.0, x.float()).clamp(-1e30, 1e30)
    blocks = finite.reshape(-1, 16).t()                                            # the rule on finite values, under the scale 1
    ratio = blocks.abs().amax(dim=0) / 6
    nearest = codecs.e4m3_bytes(ratio.clamp(max=448.0)).to(torch.int32)
    each = codecs.e4m3_values(torch.where(codecs.e4m3_values(nearest.to(torch.uint8)) < ratio, (nearest + 1).clamp(max=0x7E), nearest).to(torch.uint8))
    codes = codecs._e2m1_rne(torch.where(each > 0, blocks / torch.where(each > 0, each, 1.0), 0.0))
    want = (e2m1[codes.long()] * each).t().reshape(x.shape)
    rows, scale = ops.quantize_rows_nvfp4(x)
    assert scale.item() == 1.0 and torch.equal(rows.float(), want)
    columns, scale = ops.transpose_columns(x.t().contiguous(), nvfp4=True, as_bank=False)
    assert scale.item() == 1.0 and torch.equal(columns.float(), want)
    w = x.t()[None]
    prepared = ops.prepare(by_whole_tensors("nvfp4", w))
    compared = x.numel() // 2 + x.numel() // 16
    for held in (w, w.contiguous()):
        got = ops.quantize_matrices(held, "nvfp4")
        assert torch.equal(got.keep[0][:compared], prepared.keep[0][:compared]) and torch.equal(got.keep[2], prepared.keep[2])
