"""The NVFP4 recipe's operands: the partial largest magnitudes, rows and tokens from one read, and a step's products, against the
quantizers of one operand at a time."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def drawn(*shape, seed=0):
    generator = torch.Generator("cuda").manual_seed(seed)
    return (torch.randn(shape, generator=generator, device="cuda") * torch.randn(shape[:-1] + (1,), generator=generator, device="cuda").mul_(4).exp2_()).to(torch.bfloat16)


@pytest.mark.parametrize("shape", ((128, 128), (128, 2176), (640, 384), (8320, 256)))     # one block of threads, a part of one, rows past one a wavefront
@pytest.mark.parametrize("value", (None, 0.0, float("nan"), float("inf"), 3e38, 1e-38))    # (the last four keep the division)
def test_rows_and_tokens_from_one_read(shape, value):
    from dew_amd import ops

    x = drawn(*shape)
    if value is not None:
        x[:] = torch.where(torch.arange(shape[1], device="cuda") % 7 == 3, torch.tensor(value, device="cuda"), x) if value else 0.0
    largest = ops.nvfp4_largest(x)
    bits = x.view(torch.int16).to(torch.int32) & 0x7FFF
    assert int(largest.max()) == int(bits.max()) << 16
    by_row, by_token, scale, none = ops.quantize_nvfp4(x, largest, rows=True, tokens=True)
    want, want_scale = ops.quantize_rows_nvfp4(x)
    want_tokens, _ = ops.transpose_columns(x, nvfp4=True, as_bank=False)
    same = lambda a, b: torch.equal(a.view(torch.int16), b.view(torch.int16))
    assert none is None and torch.equal(scale.view(torch.int32), want_scale.view(torch.int32))
    assert same(by_row, want) and same(by_token, want_tokens.t().contiguous())
    only_rows = ops.quantize_nvfp4(x, largest, rows=True, tokens=False)
    only_tokens = ops.quantize_nvfp4(x, largest, rows=False, tokens=True)
    assert same(only_rows[0], want) and only_rows[1] is None and same(only_tokens[1], by_token) and only_tokens[0] is None


@pytest.mark.parametrize("shape", ((128, 16), (2, 128, 384), (9, 1024, 1032)))     # a part of a block, of the grid, several rounds
def test_largest_magnitude(shape):
    from dew_amd import ops

    x = drawn(*shape, seed=1)
    x.view(-1)[-1] = -3.0e38
    for operand in (x, x.float()):
        assert float(ops.nvfp4_largest(operand).view(torch.float32).max()) == float(operand.abs().max())


@pytest.mark.parametrize("blocks,depth,width", (([1], 256, 256), ([3, 0, 2, 4], 512, 768), ([5, 6, 7, 6], 1024, 2560), ([49], 256, 512)))    # (the last walks its tokens in transposed copies)
@pytest.mark.parametrize("cached", (True, False))     # magnitudes of all operands from one launch, or of each right before it is quantized
def test_a_step_is_its_operands_products(blocks, depth, width, cached, monkeypatch):
    from dew_amd import ops, projections

    if not cached:
        monkeypatch.setattr(projections, "CACHED_BYTES", 0)
    counts = torch.tensor(blocks, dtype=torch.int32, device="cuda")
    tokens = 128 * sum(blocks)
    x, w, dy = drawn(tokens, depth, seed=4), drawn(len(blocks), depth, width, seed=5), drawn(tokens, width, seed=6)
    offsets = ops.block_offsets(counts, 128)
    product = lambda rows, matrices: projections.nvfp4_block_product(projections.nvfp4_rows(rows), ops.quantize_matrices(matrices, "nvfp4"), projections._groups(counts, "cuda"))
    assert torch.equal(projections.nvfp4_projection(x, w, counts), product(x, w))
    d_x, d_w = projections.nvfp4_gradients(x, w, dy, counts)
    assert torch.equal(d_x, product(dy, w.transpose(1, 2)))
    rows, rows_scale = ops.transpose_columns(x, nvfp4=True, as_bank=False)
    bank, bank_scale = ops.transpose_columns(dy, nvfp4=True, as_bank=True)
    assert torch.equal(d_w, ops.kernel_gradient_bf16(rows, bank, offsets, lhs_scale=rows_scale, rhs_scale=bank_scale))
