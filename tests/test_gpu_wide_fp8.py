"""The recipes' products in 256 x 256 tiles on blocks that stay, at the edges of tiles, steps, scale groups and windows, against the launch
of one tile a block (the same order of sums: the same bits)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# Groups of rows (ragged ones too: the product finds its tiles from the offsets) and a width that fills the CUs with their tiles.
SIZES = {"edges": ([0, 1, 255, 256, 257, 513, 0, 640], 256 * 20 + 128), "many": ([112, 160] * 48, 896), "most": ([113] * 256, 640), "one": ([4000], 3328)}


def tiled(call):
    """The call on the launch of one tile a block."""
    from dew_amd import ops

    with ops.tile_rows(256):
        return call()


def operands(sizes, depth, width, extra=300):
    generator = torch.Generator("cuda").manual_seed(4)
    # rows of many magnitudes, so that a scale of another row, column or depth shows
    normal = lambda *shape: torch.randn(shape, generator=generator, device="cuda") * torch.randn(shape[:-1] + (1,), generator=generator, device="cuda").mul_(3).exp2_()
    rows = sum(sizes) + extra
    w = torch.randn((len(sizes), depth, width), generator=generator, device="cuda") * torch.randn((len(sizes), depth // 128, 1, width // 128, 1), generator=generator,
                                                                                              device="cuda").mul_(2).exp2_().expand(-1, -1, 128, -1, 128).reshape(len(sizes), depth, width)
    return normal(rows, depth).to(torch.bfloat16), w.to(torch.bfloat16), torch.tensor(sizes, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("depth", (512, 640, 1152, 2176))     # 4, 5, 9 and 17 steps: whole and ragged groups of a scale load
@pytest.mark.parametrize("name", SIZES)
@pytest.mark.parametrize("recipe", ("blockwise_fp8", "mxfp8"))
def test_products(recipe, name, depth):
    from dew_amd import ops, projections

    sizes, width = SIZES[name]
    x, w, counts = operands(sizes, depth, width)
    offsets, held = ops.group_offsets(counts), sum(sizes)
    bank = ops.quantize_matrices(w, recipe)
    codes, scales = ops.quantize_rows_mxfp8(x) if recipe == "mxfp8" else ops.quantize_rows_fp8(x)
    product = ops.grouped_gemm_mxfp8_rows if recipe == "mxfp8" else ops.grouped_gemm_fp8_rows
    got, want = product(codes, scales, bank, offsets), tiled(lambda: product(codes, scales, bank, offsets))
    assert torch.equal(got, want) and not bool(got[held:].any()) and bool(torch.isfinite(got).all()) and bool(got[:held].any(1).all())


def test_a_scale_that_is_no_power_of_two_writes_nan_where_it_is_met():
    from dew_amd import formats, gemm, ops

    sizes, depth, width = [300, 400, 500], 640, 256 * 20 + 128
    x, w, counts = operands(sizes, depth, width)
    offsets = ops.group_offsets(counts)
    codes = (w.float() / 64).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8).contiguous()
    factors = torch.ones((3, depth // 128, width // 128), device="cuda")
    factors[1, 2, 3] = 1.5
    bank = gemm.prepared(formats.Fp8Blocks(codes, factors))
    rows, scales = ops.quantize_rows_fp8(x)
    got = ops.grouped_gemm_fp8_rows(rows, scales, bank, offsets)
    hit = torch.isnan(got)
    assert bool(hit[300:700, 384:512].all()) and int(hit.sum()) == 400 * 128
    want = tiled(lambda: ops.grouped_gemm_fp8_rows(rows, scales, bank, offsets))
    assert torch.equal(got[~hit & ~torch.isnan(want)], want[~hit & ~torch.isnan(want)])


@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
@pytest.mark.parametrize("mx", (True, False))
@pytest.mark.parametrize("blocks,depth,width", (([0, 1, 5, 3, 4], 640, 256 * 20 + 128), ([9, 0, 0, 2], 896, 4096), ([1] * 33, 512, 1152)))
def test_gradients(blocks, depth, width, mx, out_dtype):
    from dew_amd import ops

    x, _, _ = operands([128 * sum(blocks)], depth, 128, extra=0)
    dy, _, _ = operands([128 * sum(blocks)], width, 128, extra=0)
    offsets = ops.block_offsets(torch.tensor(blocks, dtype=torch.int32, device="cuda"), 128)
    codes, scales = ops.quantize_columns(x, mx=mx, as_bank=False)
    bank = ops.quantize_columns(dy, mx=mx, as_bank=True)
    got = ops.kernel_gradient_mxfp8_banks(ops.quantize_columns(x, mx=mx, as_bank=True), bank, offsets, out_dtype=out_dtype)
    want = ops.kernel_gradient_mxfp8(codes, scales, bank, offsets, out_dtype=out_dtype)
    assert torch.equal(got, want) and got.dtype == out_dtype
    for g, count in enumerate(blocks):
        assert bool(got[g].any()) == (count > 0)


@pytest.mark.parametrize("blocks", ([9, 2, 0], [4, 7, 0, 0], [11] + [0] * 5))
@pytest.mark.parametrize("not_a_number", (False, True))
def test_gradients_of_empty_groups_behind_the_last_token(blocks, not_a_number):
    """Such a group has no step and no scales of its own: its gradient is zero, also beside other groups' scales that are NaN."""
    from dew_amd import ops

    depth, width = 896, 4096
    x, _, _ = operands([128 * sum(blocks)], depth, 128, extra=0)
    dy, _, _ = operands([128 * sum(blocks)], width, 128, extra=0)
    offsets, tokens = ops.block_offsets(torch.tensor(blocks, dtype=torch.int32, device="cuda"), 128), x.shape[0]
    lhs, rhs = (ops.quantize_columns(operand, mx=True, as_bank=True) for operand in (x, dy))
    codes, scales = ops.quantize_columns(x, mx=True, as_bank=False)
    want = ops.kernel_gradient_mxfp8(codes, scales, rhs, offsets)
    if not_a_number:     # the last 128 tokens' scale bytes, in every column of both operands
        for bank, columns in ((lhs, depth), (rhs, width)):
            bank.keep[0][tokens * columns:][:tokens // 32 * columns].view(columns // 32, tokens // 128, 128)[:, -1] = 0xFF
    got = ops.kernel_gradient_mxfp8_banks(lhs, rhs, offsets)
    last = max(g for g, count in enumerate(blocks) if count)
    for g, count in enumerate(blocks):
        if not count:
            assert not bool(got[g].any())
        elif not_a_number and g == last:
            assert bool(torch.isnan(got[g]).all())
        else:
            assert torch.equal(got[g], want[g]) and bool(got[g].any())
