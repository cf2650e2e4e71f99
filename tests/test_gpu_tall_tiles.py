"""Tiles of up to 256 rows on eight wavefronts (csrc/tall.hip) against the 64-row tiles' launch, bit for bit (every sum is formed in the same
order): every number of 32-row tiles a group can end in, groups of several tiles, empty ones, rows past the last group, gathers, scatters,
depths that are no whole rounds of the weight registers, a last strip of fewer columns."""

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = {"fp8": [0, 1, 31, 32, 33, 64, 65, 96, 97, 128, 161, 192, 193, 224, 256, 257],     # 114 rows a group
         "nvfp4": [0, 1, 33, 64, 97, 128, 161, 192, 225, 256, 257, 300, 513, 129, 224, 290],  # 179
         "several tiles": [3, 290, 513, 256, 700, 40, 515, 320],                              # 329
         "two rounds of the search": [(37 * g) % 261 for g in range(72)]}                     # 130: groups past the 64th, some empty
PAST = 300                                                                                    # sorted positions past the last group


def banks(form, experts, depth, width, count):
    from dew_amd import formats

    quantized = {"block": formats.Fp8Blocks.quantized, "channel": formats.Fp8Channels.quantized, "nvfp4": formats.NvFp4.quantized,
                 "bf16": lambda w: formats.Bf16(w.to(torch.bfloat16))}[form]
    generator = torch.Generator(device="cuda").manual_seed(depth + width)
    return [formats.stacked([quantized(torch.randn(1, depth, width, device="cuda", generator=generator) * 0.02 * (e % 3 + 1)) for e in range(experts)])
            for _ in range(count)]


PRODUCTS = [                                        # (format, sizes, depth, width, the gating of a pair: its activation and clamp)
    ("block", "fp8", 3200, 3328, ("swiglu", None)),       # 50 steps
    ("block", "fp8", 2048, 3200, None),                   # a last strip of 128 columns
    ("block", "fp8", 3072, 3328, ("swiglu", 0.75)),
    ("block", "fp8", 3072, 3328, ("geglu", None)),
    ("channel", "fp8", 2432, 3200, None),                 # 38 steps
    ("block", "several tiles", 3584, 16640, ("swiglu", None)),
    ("block", "two rounds of the search", 3072, 640, ("geglu", 1.5)),
    ("nvfp4", "nvfp4", 2304, 8064, None),                 # a last strip of 128 columns
    ("nvfp4", "two rounds of the search", 2304, 2048, None),
    ("bf16", "fp8", 2560, 1568, ("swiglu", None)),        # 40 steps; a last strip of 32 columns; tiles of at most 224 rows
    ("bf16", "fp8", 2880, 1664, ("swiglu", 0.75)),        # 45 steps
    ("bf16", "two rounds of the search", 2560, 768, ("geglu", None)),
    ("bf16", "fp8", 1344, 3232, None),                    # 21 steps; a last strip of 160 columns
    ("bf16", "nvfp4", 1472, 5216, None),                  # 23 steps; a last strip of 96 columns
]


@pytest.mark.parametrize("form,sizes,depth,width,gating", PRODUCTS)
def test_tall_tiles_return_the_shorter_tiles_bits(form, sizes, depth, width, gating):
    from dew_amd import _lib, gemm, ops

    sizes = SIZES[sizes]
    rows, experts = sum(sizes), len(sizes)
    held = [gemm.prepared(b) for b in banks(form, experts, depth, width, 2 if gating else 1)]
    rng = np.random.default_rng(depth)
    x = torch.from_numpy(rng.standard_normal((rows + 31, depth)).astype(np.float32)).to(torch.bfloat16).cuda()
    padded = rows + PAST                                  # (the rows past the last group are zero)
    assert _lib.library().dew_moe_takes_tall_tiles(held[0].descriptor, gating is not None, padded) == 1
    gather = torch.from_numpy(rng.integers(0, rows + 31, size=padded).astype(np.int32)).cuda()
    scatter = torch.from_numpy(rng.permutation(padded).astype(np.int32)).cuda()
    counts = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    offsets = torch.tensor(np.concatenate([[0], np.cumsum(sizes)]), dtype=torch.int32, device="cuda")
    bias = torch.from_numpy(rng.standard_normal((experts, width)).astype(np.float32)).cuda()

    def product(by_sizes):
        if gating:
            activation, limit = gating
            groups = dict(offsets=None, sizes=counts) if by_sizes else dict(offsets=offsets)
            return ops.gateup_swiglu(x, *held, gather=gather, activation=activation, limit=limit, **groups)
        if by_sizes:
            return gemm.gemm(x, held[0], counts, gather=gather, epilogue="plus_bias", epilogue_operands=(bias,))
        return ops.grouped_gemm(x, held[0], offsets, gather=gather, scatter=scatter)

    for by_sizes in (False, True):
        got = product(by_sizes)
        with ops.tile_rows(64):
            assert _lib.library().dew_moe_takes_tall_tiles(held[0].descriptor, gating is not None, padded) == 0
            expected = product(by_sizes)
        assert bool(torch.isfinite(expected.float()).all()) and torch.equal(got, expected)
        past = got[scatter[rows:].long()] if not (gating or by_sizes) else got[rows:]
        assert past.shape[0] == PAST and not bool(past.any()) and bool(got.any())
