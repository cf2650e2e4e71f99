"""Plain bf16 operands' products in 256 x 256 tiles, at the edges of tiles, steps and groups, against the launch of smaller tiles that
gathered rows take (the same order of sums: the same bits)."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = {"edges": [0, 1, 255, 256, 257, 513, 0, 640], "tails": [129, 1000, 383, 700], "many": [112, 160] * 48, "most": [113] * 256, "one": [4000]}
WIDTHS = {"edges": 8 * 600 + 32, "tails": 256 * 20 + 96, "many": 1056, "most": 288, "one": 3296}     # (tiles over the CUs: three quarters of a round at least)


def operands(sizes, depth, width, extra=300):
    generator = torch.Generator("cuda").manual_seed(9)
    normal = lambda *shape: torch.randn(shape, generator=generator, device="cuda").to(torch.bfloat16)
    rows = sum(sizes) + extra
    return normal(rows, depth), normal(len(sizes), depth, width) * 0.05, normal(rows, width), torch.tensor(sizes, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("depth", (64, 128, 192, 448))     # one step, two, an odd number, more than either ring holds
@pytest.mark.parametrize("name", SIZES)
def test_products(name, depth):
    from dew_amd import ops

    x, w, _, sizes = operands(SIZES[name], depth, WIDTHS[name])
    x[sum(SIZES[name]):] = float("nan")                     # rows of no group: never read into a sum, zero in the result
    offsets, held = ops.group_offsets(sizes), sum(SIZES[name])
    as_they_lie = torch.arange(x.shape[0], dtype=torch.int32, device="cuda")
    want = ops.dense_gemm(x, w, offsets, gather=as_they_lie)
    plain = ops.dense_gemm(x, w, offsets)
    assert torch.equal(plain, want) and not bool(plain[held:].any()) and bool(torch.isfinite(plain).all())
    assert torch.equal(ops.dense_gemm(x, w, None, sizes=sizes), want)
    kmajor = w.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(ops.dense_gemm(x, kmajor, offsets), want) and torch.equal(ops.dense_gemm(x, kmajor, None, sizes=sizes), want)


@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
@pytest.mark.parametrize("sizes,depth,width", (([0, 1, 63, 64, 65, 1500], 264, 5152), ([257, 300, 1, 700], 520, 5384), ([257, 300, 1, 700], 520, 5896), ([2, 4000, 5, 0], 1032, 2568)))
def test_gradients(sizes, depth, width, out_dtype):
    from dew_amd import gemm, ops

    x, _, dy, counts = operands(sizes, depth, width)
    x[sum(sizes):] = float("nan")
    scale = torch.tensor([0.5], device="cuda")
    got = gemm.gemm_t(x, dy, counts, out_dtype=out_dtype)
    assert got.dtype == out_dtype
    assert torch.equal(got, gemm.gemm_t(x, dy, gemm.GroupSizes(counts, ops.group_offsets(counts)), out_dtype=out_dtype))
    assert torch.equal(got * 0.5, ops.dense_gradient(x, dy, None, sizes=counts, lhs_scale=scale, out_dtype=out_dtype))
    # with so many groups of no rows behind them that they have fewer than 256 rows each, the launch of smaller tiles (the same order of sums)
    many = torch.cat([counts, counts.new_zeros(x.shape[0] // 255)])
    assert x.shape[0] // many.numel() < 256
    tiled = ops.dense_gradient(x, dy, None, sizes=many, out_dtype=out_dtype)
    assert torch.equal(got, tiled[:len(sizes)]) and not bool(tiled[len(sizes):].any())
    begin = 0
    for g, size in enumerate(sizes):
        want = x[begin:begin + size].float().T @ dy[begin:begin + size].float()
        # sums of `size` products of unit normals in another order: 2^-24 a term and step; bf16 outputs round once more
        bound = 1e-5 * max(size, 1) + (2.0 ** -8 * want.abs() if out_dtype == torch.bfloat16 else 0.0)
        assert bool(((got[g].float() - want).abs() <= bound).all())
        begin += size


def test_a_nan_stays_in_its_group():
    """What a tile's loads fetch past its own rows, columns and groups is not part of any sum."""
    from dew_amd import gemm, ops

    x, w, dy, sizes = operands([300, 500, 700, 900], 768, 5152)
    x[300:800], dy[800:1500], w[3] = float("nan"), float("inf"), float("nan")
    y, d_w = ops.dense_gemm(x, w, None, sizes=sizes), gemm.gemm_t(x, dy, sizes)
    assert bool(torch.isfinite(y[:300]).all()) and bool(torch.isfinite(y[800:1500]).all()) and bool(torch.isnan(y[300:800]).all()) and bool(torch.isnan(y[1500:2400]).all())
    finite = torch.isfinite(d_w).flatten(1)
    assert bool(finite[0].all()) and bool(finite[3].all()) and not bool(finite[1].any()) and not bool(finite[2].any())
