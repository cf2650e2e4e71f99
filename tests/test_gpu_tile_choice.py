"""The tile that a launch takes by itself, on both sides of the lines the rules draw: every tile sums a product's depth in the same
order, so the outputs are the other tiles' bit for bit."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from dew_amd import ops

    ops.device_check()
    return ops


def groups(experts, average, seed):
    """Sizes that a gate's preferences spread: an empty group, one of a single row, the rest of anything around the average."""
    generator = torch.Generator().manual_seed(seed)
    share = torch.softmax(torch.randn(experts, generator=generator) * 0.5, 0)
    ends = (share.cumsum(0) * average * experts).round().int()
    ends[0], ends[1], ends[-1] = 0, 1, average * experts
    return torch.cat([torch.zeros(1, dtype=torch.int32), ends.cummax(0).values]).cuda()


# (experts, rows a group, depth, width): unquantized banks' lines at 26, 48, 76, 96 and 512 rows and at 160 and 640 blocks;
# FP8 between 128 and 184 rows; NVFP4 at 212 rows and 1000 blocks; the two launches of 3072 strips
CASES = [("bf16", 8, 27, 256, 1024), ("bf16", 8, 40, 896, 768), ("bf16", 8, 49, 512, 384), ("bf16", 16, 75, 256, 1152),
         ("bf16", 16, 77, 256, 1312), ("bf16", 32, 97, 2048, 1408), ("bf16", 32, 140, 1792, 2048), ("bf16", 4, 512, 256, 640),
         ("fp8_block", 32, 140, 256, 1664), ("fp8_channel", 16, 180, 384, 2560), ("nvfp4", 16, 213, 256, 2560), ("nvfp4", 16, 280, 512, 3200),
         ("fp8_block", 128, 260, 256, 3072), ("mxfp4", 48, 390, 256, 2048)]


@pytest.mark.parametrize("quant,experts,average,depth,width", CASES)
def test_the_chosen_tile_returns_the_others_bits(ops, quant, experts, average, depth, width):
    from dew_amd import codecs, formats, gemm

    generator = torch.Generator(device="cuda").manual_seed(depth + width + average)
    w = torch.randn((experts, depth, width), generator=generator, device="cuda") * 0.05
    makers = {"bf16": lambda: formats.Bf16(w.to(torch.bfloat16)), "fp8_block": lambda: formats.Fp8Blocks.quantized(w),
              "fp8_channel": lambda: formats.Fp8Channels.quantized(w), "nvfp4": lambda: formats.NvFp4.quantized(w),
              "mxfp4": lambda: formats.Mxfp4Blocks(*codecs.quantize_mxfp4(w))}
    bank = gemm.prepared(makers[quant]())
    del w
    offsets = groups(experts, average, seed=average)
    rows = experts * average
    x = torch.randn((rows, depth), generator=generator, device="cuda").to(torch.bfloat16)
    scatter = torch.randperm(rows, generator=generator, device="cuda").int()
    plain, paired = ops.grouped_gemm(x, bank, offsets, scatter=scatter), ops.gateup_swiglu(x, bank, bank, offsets)
    assert plain.isfinite().all() and plain.abs().amax() > 0
    for tile in (64, 128):
        with ops.tile_rows(tile):
            assert torch.equal(ops.grouped_gemm(x, bank, offsets, scatter=scatter), plain), tile
            assert torch.equal(ops.gateup_swiglu(x, bank, bank, offsets), paired), tile
