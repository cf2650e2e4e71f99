"""256 x 256 tiles on the lines from which they are taken: so few that half of the blocks have none, and a second round just begun. The
comparisons are those of test_gpu_wide.py and test_gpu_wide_fp8.py, with the launches of smaller tiles (the same bits; a bf16 gradient's is the
one of as many groups that each has fewer than 256 rows) and of gradients with products in fp32."""

import pytest
import test_gpu_wide
import test_gpu_wide_fp8
import torch

pytestmark = pytest.mark.gpu


# (those files add 300 rows of no group: 148, 266 and 292 tiles by the launch's guess, of which K-major matrices take all and natural ones
# the first and the last; blocks without a tile clear rows all the same)
@pytest.mark.parametrize("sizes,width", (([940, 1000, 1100, 900], 2048), ([1900, 2050, 2000, 1750], 2048), ([1900, 1850, 2000, 1750], 2304)))
def test_products(monkeypatch, sizes, width):
    monkeypatch.setitem(test_gpu_wide.SIZES, "lines", sizes)
    monkeypatch.setitem(test_gpu_wide.WIDTHS, "lines", width)
    test_gpu_wide.test_products("lines", 320)


@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
@pytest.mark.parametrize("sizes,depth,width", (([257, 300, 700, 0, 500, 299, 301, 302, 400], 1032, 1000), ([300] * 9, 1024, 2048)))     # 180 tiles, 288
def test_gradients(sizes, depth, width, out_dtype):
    test_gpu_wide.test_gradients(sizes, depth, width, out_dtype)


# Quarters: a launch of nothing else (with a group of no rows and one of a row; whole quarters past a group's rows and past the width), two a
# block, and behind a whole round, one a block and two; the depths are one step, an odd number and more than the ring holds.
@pytest.mark.parametrize("depth,sizes,width", ((64, [129, 1000, 0, 383, 1, 700], 800), (320, [129, 1000, 383, 700], 800), (448, [600], 160),
                                               (2112, [2100, 1900], 1504), (448, [4000], 4384), (1088, [3800, 200], 5472),
                                               # (at most one quarter a block, though the tiles have more than 256: 80 and 240 real ones, 66 and 242)
                                               (2112, [1, 127, 128, 129, 255, 256, 257, 0] * 5, 480), (2112, [1310], 2816)))
def test_products_in_quarters(monkeypatch, depth, sizes, width):
    monkeypatch.setitem(test_gpu_wide.SIZES, "quarters", sizes)
    monkeypatch.setitem(test_gpu_wide.WIDTHS, "quarters", width)
    test_gpu_wide.test_products("quarters", depth)


@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
@pytest.mark.parametrize("sizes,depth,width", (([600, 513, 1, 800], 264, 1032), ([3000, 1800], 1032, 2568), ([700, 800], 2056, 4104), ([1500, 900], 2504, 4400),
                                               ([1348], 2624, 1496), ([600, 1513, 0, 1], 576, 1416)))     # (66 tiles, 252 real quarters; 72, 240)
def test_gradients_in_quarters(sizes, depth, width, out_dtype):
    test_gpu_wide.test_gradients(sizes, depth, width, out_dtype)


@pytest.mark.parametrize("sizes", ([480, 600, 700, 500], [1900, 2050, 2100, 1950]))     # 97 tiles by the launch's guess, 275
@pytest.mark.parametrize("recipe", ("blockwise_fp8", "mxfp8"))
def test_recipes_products(monkeypatch, recipe, sizes):
    monkeypatch.setitem(test_gpu_wide_fp8.SIZES, "lines", (sizes, 2048))
    test_gpu_wide_fp8.test_products(recipe, "lines", 640)


@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
@pytest.mark.parametrize("mx", (True, False))
@pytest.mark.parametrize("blocks,depth,width", (([1, 2, 0, 3, 1, 1, 2, 1, 4], 1024, 1024), ([1] * 9, 1024, 2048)))     # 144 tiles, 288
def test_recipes_gradients(blocks, depth, width, mx, out_dtype):
    test_gpu_wide_fp8.test_gradients(blocks, depth, width, mx, out_dtype)


# (whole and ragged groups of a scale load; one quarter a block and two, alone and behind a whole round)
@pytest.mark.parametrize("depth,sizes,width", ((512, [129, 1000, 0, 383, 1, 700], 896), (640, [129, 1000, 383, 700], 896), (2176, [2100, 1900], 1408),
                                               (640, [4000], 4480), (2176, [3800, 200], 5504),
                                               (2176, [1, 127, 128, 129, 255, 256, 257, 0] * 5, 512), (2176, [1310], 2816)))
@pytest.mark.parametrize("recipe", ("blockwise_fp8", "mxfp8"))
def test_recipes_products_in_quarters(monkeypatch, recipe, depth, sizes, width):
    monkeypatch.setitem(test_gpu_wide_fp8.SIZES, "quarters", (sizes, width))
    test_gpu_wide_fp8.test_products(recipe, "quarters", depth)


@pytest.mark.parametrize("out_dtype", (torch.bfloat16, torch.float32))
@pytest.mark.parametrize("mx", (True, False))
@pytest.mark.parametrize("blocks,depth,width", (([0, 1, 5, 3, 4], 640, 640), ([9, 2, 0], 640, 896), ([40, 1], 896, 4096), ([5, 4], 2176, 4096),
                                              ([1, 0, 2, 1, 3, 1, 0, 2], 640, 640)))     # (72 tiles, 200 real quarters)
def test_recipes_gradients_in_quarters(blocks, depth, width, mx, out_dtype):
    test_gpu_wide_fp8.test_gradients(blocks, depth, width, mx, out_dtype)


def test_a_quarter_writes_nan_where_it_meets_a_scale_that_is_no_power_of_two():
    from dew_amd import formats, gemm, ops

    sizes, depth, width = [300, 400, 500], 640, 896
    x, w, counts = test_gpu_wide_fp8.operands(sizes, depth, width)
    factors = torch.ones((3, depth // 128, width // 128), device="cuda")
    factors[1, 4, 3] = 1.5
    bank = gemm.prepared(formats.Fp8Blocks((w.float() / 64).clamp(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8).contiguous(), factors))
    got = ops.grouped_gemm_fp8_rows(*ops.quantize_rows_fp8(x), bank, ops.group_offsets(counts))
    assert bool(torch.isnan(got[300:700, 384:512]).all()) and int(torch.isnan(got).sum()) == 400 * 128


def test_no_block_waits_a_turn_for_quarters_past_the_rows_and_columns():
    """68 tiles of 768 rows, whose 204 real quarters are one a block, take what 64 tiles do (39 and 22 us where they took two turns)."""
    from dew_amd import ops

    def fastest(width):
        x, w, counts = test_gpu_wide_fp8.operands([384, 384], 5376, width, extra=0)
        rows, bank, offsets = ops.quantize_rows_fp8(x), ops.quantize_matrices(w, "blockwise_fp8"), ops.group_offsets(counts)
        times = []
        for _ in range(6):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(10):
                ops.grouped_gemm_fp8_rows(*rows, bank, offsets)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    assert fastest(4352) <= 1.4 * fastest(4096)
