"""Tiles of up to 256 rows on eight wavefronts (csrc/tall.hip) against the 64-row tiles' launch, bit for bit (every sum is formed in the same
order): every number of 32-row tiles a group can end in, groups of several tiles, empty ones, rows past the last group, gathers, scatters,
depths that are no whole rounds of the weight registers, a last strip of fewer columns."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = {"fp8": [0, 1, 31, 32, 33, 64, 65, 96, 97, 128, 161, 192, 193, 224, 256, 257],     # 114 rows a group
         "nvfp4": [0, 1, 33, 64, 97, 128, 161, 192, 225, 256, 257, 300, 513, 129, 224, 290],  # 179
         "several tiles": [3, 290, 513, 256, 700, 40, 515, 320]}                               # 329


def banks(form, experts, depth, width, count):
    from dew_amd import formats

    quantized = {"block": formats.Fp8Blocks.quantized, "channel": formats.Fp8Channels.quantized, "nvfp4": formats.NvFp4.quantized,
                 "bf16": lambda w: formats.Bf16(w.to(torch.bfloat16))}[form]
    generator = torch.Generator(device="cuda").manual_seed(depth + width)
    return [formats.stacked([quantized(torch.randn(1, depth, width, device="cuda", generator=generator) * 0.02 * (e % 3 + 1)) for e in range(experts)])
            for _ in range(count)]


@pytest.mark.parametrize("form,sizes,depth,width,paired,limit", [
    ("block", "fp8", 3200, 3328, True, None),       # 50 steps
    ("block", "fp8", 2048, 3200, False, None),      # a last strip of 128 columns
    ("block", "fp8", 3072, 3328, True, 0.75),
    ("channel", "fp8", 2432, 3200, False, None),    # 38 steps
    ("block", "several tiles", 3584, 16640, True, None),
    ("nvfp4", "nvfp4", 2304, 8064, False, None),   # a last strip of 128 columns
    ("bf16", "fp8", 2560, 1568, True, None),        # 40 steps; a last strip of 32 columns; tiles of at most 224 rows
    ("bf16", "fp8", 2880, 1664, True, 0.75),        # 45 steps
    ("bf16", "fp8", 1344, 3232, False, None),       # 21 steps; a last strip of 160 columns
    ("bf16", "nvfp4", 1472, 5216, False, None),     # 23 steps; a last strip of 96 columns
])
def test_tall_tiles_return_the_shorter_tiles_bits(form, sizes, depth, width, paired, limit):
    from dew_amd import gemm, ops

    sizes = SIZES[sizes]
    rows, experts = sum(sizes), len(sizes)
    held = [gemm.prepared(b) for b in banks(form, experts, depth, width, 2 if paired else 1)]
    rng = np.random.default_rng(depth)
    x = torch.from_numpy(rng.standard_normal((rows + 31, depth)).astype(np.float32)).to(torch.bfloat16).cuda()
    padded = rows + 300                                  # sorted positions past the last group: zero rows
    gather = torch.from_numpy(rng.integers(0, rows + 31, size=padded).astype(np.int32)).cuda()
    scatter = torch.from_numpy(rng.permutation(padded).astype(np.int32)).cuda()
    counts = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    offsets = torch.tensor(np.concatenate([[0], np.cumsum(sizes)]), dtype=torch.int32, device="cuda")

    def product(plain):
        if paired:
            return gemm.gemm(x, held[0], counts, paired=held[1], gather=gather, epilogue="swiglu", epilogue_operands=() if limit is None else (limit,))
        if plain:
            return gemm.gemm(x, held[0], counts, gather=gather, epilogue="plus_bias", epilogue_operands=(bias,))
        return ops.grouped_gemm(x, held[0], offsets, gather=gather, scatter=scatter)

    bias = torch.from_numpy(rng.standard_normal((experts, width)).astype(np.float32)).cuda()
    for plain in (False, True):
        got = product(plain)
        with ops.tile_rows(64):
            expected = product(plain)
        assert bool(torch.isfinite(expected.float()).all()) and torch.equal(got, expected)
