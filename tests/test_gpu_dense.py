"""Plain bf16 operands' grouped products, read where they lie, against the tiled launches on prepared banks (the same order of sums:
the same bits) and against fp32 products in PyTorch."""

import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = {"ragged": [0, 1, 31, 33, 200, 0, 129, 64], "one": [130], "tall": [300, 520], "many": [2] * 70, "empty": [0, 0, 0]}


def inputs(sizes, depth, width, extra=7):
    generator = torch.Generator("cuda").manual_seed(5)
    normal = lambda *shape: torch.randn(shape, generator=generator, device="cuda").to(torch.bfloat16)
    rows = sum(sizes) + extra
    return normal(rows, depth), normal(len(sizes), depth, width) * 0.05, normal(rows, width), torch.tensor(sizes, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("depth,width", ((128, 128), (192, 288), (640, 512), (576, 160)))
@pytest.mark.parametrize("name", SIZES)
def test_products_of_plain_matrices(name, depth, width):
    from dew_amd import formats, gemm, ops

    sizes_list = SIZES[name]
    x, w, _, sizes = inputs(sizes_list, depth, width)
    rows = x.shape[0]
    generator = torch.Generator("cuda").manual_seed(6)
    gather = torch.randint(0, rows, (rows,), generator=generator, device="cuda", dtype=torch.int32)
    scatter = torch.randperm(rows, generator=generator, device="cuda").to(torch.int32)
    bank = ops.prepare(formats.Bf16(w))
    offsets = ops.group_offsets(sizes)
    plain = gemm.gemm(x, w, sizes)
    assert torch.equal(plain, ops.grouped_gemm(x, bank, offsets)) and not bool(plain[sum(sizes_list):].any())
    moved = gemm.gemm(x, w, gemm.GroupSizes(sizes, offsets), gather=gather, scatter=scatter)
    assert torch.equal(moved, ops.grouped_gemm(x, bank, offsets, gather=gather, scatter=scatter))
    kmajor = w.transpose(1, 2).contiguous().transpose(1, 2)
    assert torch.equal(gemm.gemm(x, kmajor, sizes), plain)
    begin = 0
    for g, size in enumerate(sizes_list):
        want = x[begin:begin + size].float() @ w[g].float()
        # one bf16 rounding of an fp32 sum: 2^-8 of the value, and the sums' own order, 2^-20 of their terms' scale
        assert bool(((plain[begin:begin + size].float() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())
        begin += size


@pytest.mark.parametrize("depth,width", ((128, 128), (192, 288), (136, 520), (8, 24)))
@pytest.mark.parametrize("name", SIZES)
@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
def test_kernel_gradients_of_plain_rows(name, depth, width, out_dtype):
    from dew_amd import gemm, ops

    sizes_list = SIZES[name]
    x, _, dy, sizes = inputs(sizes_list, depth, width)
    x[sum(sizes_list):] = float("nan")                     # rows of no group: never part of a sum
    got = gemm.gemm_t(x, dy, sizes, out_dtype=out_dtype)
    assert torch.equal(got, gemm.gemm_t(x, dy, gemm.GroupSizes(sizes, ops.group_offsets(sizes)), out_dtype=out_dtype))
    begin = 0
    for g, size in enumerate(sizes_list):
        want = x[begin:begin + size].float().T @ dy[begin:begin + size].float()
        # sums of `size` products of unit normals in another order: 2^-24 a term and step; bf16 outputs round once more
        bound = 1e-5 * max(size, 1) + (2.0 ** -8 * want.abs() if out_dtype == torch.bfloat16 else 0.0)
        assert got.dtype == out_dtype and bool(((got[g].float() - want).abs() <= bound).all())
        begin += size
    scale = torch.tensor([0.5], device="cuda")
    assert torch.equal(ops.dense_gradient(x, dy, None, sizes=sizes, lhs_scale=scale, out_dtype=out_dtype), got * 0.5)


# (a launch of few tiles takes a quarter of one each, a gradient's half: these are many, the last one's columns past the width)
@pytest.mark.parametrize("name", ("ragged", "tall", "many"))
def test_products_of_many_tiles(name):
    test_products_of_plain_matrices(name, 192, 5152)


@pytest.mark.parametrize("name", ("ragged", "many"))
@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
def test_kernel_gradients_of_many_tiles(name, out_dtype):
    test_kernel_gradients_of_plain_rows(name, 264, 5152, out_dtype)


@pytest.mark.parametrize("turned", (False, True), ids=("natural", "kmajor"))
@pytest.mark.parametrize("offset", (1, 4))                # elements: off by two bytes, and by eight
def test_matrices_that_begin_anywhere(offset, turned):
    """A view into a flat buffer of parameters need not begin on 16 bytes."""
    from dew_amd import gemm

    x, w, _, sizes = inputs(SIZES["ragged"], 192, 288)
    held = w.transpose(1, 2).contiguous() if turned else w
    flat = torch.empty(w.numel() + 8, dtype=torch.bfloat16, device="cuda")
    view = flat[offset:offset + w.numel()].view(held.shape)
    view.copy_(held)
    assert view.data_ptr() % 16 == 2 * offset and view.is_contiguous()
    assert torch.equal(gemm.gemm(x, view.transpose(1, 2) if turned else view, sizes), gemm.gemm(x, w, sizes))


# (groups, rows a group, depth, width, turned): on the lines from which the matrices are laid out first, and just short of each
LINES = [(1, 8192, 2048, 1536, False), (1, 8191, 2048, 1536, False), (1, 4096, 2048, 3072, True), (1, 4095, 2048, 3072, True), (1, 4096, 1984, 3072, True),
         (2, 3000, 4096, 2048, True), (2, 2999, 4096, 2048, True), (2, 3000, 4096, 1920, True), (1, 8192, 2048, 1312, False), (1, 8192, 2048, 1568, True)]


@pytest.mark.parametrize("groups,rows,depth,width,turned", LINES)
def test_matrices_laid_out_first_return_the_same_bits(groups, rows, depth, width, turned):
    from dew_amd import gemm, ops

    x, w, _, sizes = inputs([rows + 5 * (1 - 2 * (g % 2)) * (groups > 1) for g in range(groups)], depth, width, extra=0)
    if turned:
        w = w.transpose(1, 2).contiguous().transpose(1, 2)
    average, tiles = rows, (groups * rows // 128 + groups // 2 + 1) * -(-width // 256)
    laid = tiles >= 384 and depth >= 2048 and average >= (8192 if not turned else 3000 if depth >= 4096 else 4096) and (not turned or width % 128 == 0)
    assert gemm._relaid_first(w, x.shape[0]) == laid
    scatter = torch.randperm(x.shape[0], device="cuda").to(torch.int32)
    assert torch.equal(gemm.gemm(x, w, sizes, scatter=scatter), ops.dense_gemm(x, w, ops.group_offsets(sizes), scatter=scatter))
