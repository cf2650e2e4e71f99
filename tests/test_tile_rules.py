"""Which products take tiles of up to 256 rows on eight wavefronts (dew_moe_takes_tall_tiles), and which layers' down product and combine are one
launch (dew_moe_combines_few): rules (csrc/gemm.hip) that can be asked without a GPU. The shapes are ones where both forms were timed; times in us,
the shorter tiles' and the tall ones', or two launches' and one's."""

import pytest

from dew_amd import _lib

BLOCK, CHANNEL, NVFP4, MXFP4, BF16 = _lib.W_FP8_BLOCK, _lib.W_FP8_CHANNEL, _lib.W_NVFP4, _lib.W_MXFP4, _lib.W_BF16


def taken(form, experts, rows, depth, width, paired=False, layout=_lib.LAYOUT_PREPARED):
    return bool(_lib.library().dew_moe_takes_tall_tiles(_lib.Bank(form, layout, experts, depth, width, None, None, None), paired, experts * rows))


@pytest.mark.parametrize("experts,rows,depth,width", [
    (128, 265, 3328, 896),     # 213 -> 277
    (64, 194, 3584, 2176),     # 203 -> 265
    (128, 284, 3968, 896),     # 267 -> 345
    (32, 239, 4352, 7168)])
def test_mxfp4_banks_stay_on_the_shorter_tiles(experts, rows, depth, width):
    assert not taken(MXFP4, experts, rows, depth, width)
    assert not taken(MXFP4, experts, rows, depth, width, paired=True)


@pytest.mark.parametrize("experts,rows,depth,width,tall", [
    (24, 95, 3968, 2688, False),      # 103 -> 142
    (16, 91, 4608, 4608, False),      # 117 -> 154
    (32, 170, 2944, 1664, False),     # 83 -> 109
    (64, 145, 2560, 640, False),      # 48 -> 63: three strips, the third half empty
    (256, 186, 2560, 512, False),     # 170 -> 189
    (16, 150, 2560, 4352, False),     # 272 tiles of 256 CUs'
    (8, 145, 2944, 7040, True),       # 97 -> 64
    (24, 148, 2816, 2304, True),      # 97 -> 67
    (32, 197, 2944, 1536, True),      # 101 -> 72
    (8, 150, 6912, 7168, True)])      # 216 -> 146
def test_one_fp8_bank_takes_them_where_the_last_round_is_mostly_full(experts, rows, depth, width, tall):
    assert taken(BLOCK, experts, rows, depth, width) == tall
    assert taken(CHANNEL, experts, rows, depth, width) == tall


@pytest.mark.parametrize("experts,rows,depth,width,tall", [
    (24, 132, 2048, 1792, False),     # 66 -> 86
    (128, 105, 3968, 768, False),     # 239 -> 288
    (64, 103, 6016, 768, False),      # 176 -> 223
    (48, 96, 3840, 1024, False),      # 118 -> 141
    (64, 322, 2048, 2560, False),     # 464 -> 475
    (8, 147, 5376, 6400, True),       # 284 -> 193
    (64, 132, 5120, 1024, True),      # 296 -> 202
    (48, 142, 5632, 1280, True),      # 315 -> 226
    (114, 298, 5120, 2048, True)])    # 1560 -> 1495
def test_fp8_block_pairs_take_them_where_deep_and_where_the_shorter_rounds_are_not_full(experts, rows, depth, width, tall):
    assert taken(BLOCK, experts, rows, depth, width, paired=True) == tall


@pytest.mark.parametrize("experts,rows,depth,width", [
    (128, 105, 2560, 1152),    # 204 -> 251
    (64, 91, 2688, 896),       # 85 -> 106
    (32, 157, 3072, 1664),     # 135 -> 152
    (64, 320, 4096, 3072),
    (8, 147, 5376, 6400)])
def test_pairs_of_channel_scaled_banks_stay_on_the_shorter_tiles(experts, rows, depth, width):
    assert not taken(CHANNEL, experts, rows, depth, width, paired=True)


def test_channel_scaled_banks_of_large_groups_stay_on_the_shorter_tiles():
    assert not taken(CHANNEL, 128, 286, 2048, 7168) and not taken(CHANNEL, 64, 201, 4096, 7168)
    assert taken(CHANNEL, 8, 147, 4480, 6912)                        # 149 -> 87


@pytest.mark.parametrize("experts,rows,depth,width,tall", [
    (64, 533, 3328, 1280, False),     # 284 -> 331
    (48, 844, 2304, 1536, False),     # 270 -> 306
    (64, 268, 3072, 1536, False),     # 170 -> 217
    (8, 1024, 14336, 4096, False),    # 839 -> 839
    (32, 216, 3072, 4096, False),
    (128, 156, 3072, 1024, True),     # 194 -> 138
    (64, 161, 3072, 2048, True),      # 195 -> 142
    (16, 207, 2304, 8192, True)])     # 174 -> 128
def test_nvfp4_banks_take_them_where_a_group_is_one_tile(experts, rows, depth, width, tall):
    assert taken(NVFP4, experts, rows, depth, width) == tall
    assert not taken(NVFP4, experts, rows, depth, width, paired=True)


@pytest.mark.parametrize("experts,rows,depth,width,paired,tall", [
    (24, 263, 1664, 1536, False, False),    # 55 -> 76
    (8, 287, 4096, 4352, False, False),     # 118 -> 156
    (24, 49, 1152, 6528, False, False),     # 78 -> 83
    (64, 104, 2048, 1408, True, False),     # with its down product 301 -> 318
    (24, 112, 7040, 2432, False, True),     # 233 -> 148
    (48, 73, 6656, 1280, False, True),      # 219 -> 141
    (128, 97, 3200, 512, False, True),      # 130 -> 84
    (32, 162, 2560, 1536, True, True),      # 156 -> 128
    (25, 29, 4864, 4864, True, True)])      # 458 -> 380
def test_unquantized_banks_take_them_in_whole_rounds_of_groups_of_one_tile(experts, rows, depth, width, paired, tall):
    assert taken(BF16, experts, rows, depth, width, paired) == tall


def test_what_is_no_prepared_bank_or_has_no_rows_takes_none():
    assert taken(BF16, 24, 112, 7040, 2432)                          # 233 -> 148
    assert not taken(BF16, 24, 0, 7040, 2432) and not taken(BF16, 24, -112, 7040, 2432)
    assert not taken(BF16, 24, 112, 7040, 2432, layout=_lib.LAYOUT_REFERENCE)
    assert _lib.library().dew_moe_takes_tall_tiles(None, 0, 100) == 0


@pytest.mark.parametrize("form,tokens,top_k,experts,depth,width,combined", [
    (MXFP4, 11, 6, 32, 512, 1024, False),     # 23.1 -> 27.8
    (NVFP4, 15, 6, 32, 512, 768, False),      # 26.9 -> 31.4
    (NVFP4, 4, 5, 64, 768, 2304, False),      # 36.0 -> 39.4
    (BLOCK, 2, 2, 16, 1024, 4480, False),     # 30.6 -> 32.2
    (BLOCK, 8, 3, 8, 640, 2048, False),       # 26.2 -> 27.5
    (BLOCK, 1, 8, 128, 768, 2048, False),     # 26.4 -> 28.7: 196 KB a block
    (CHANNEL, 1, 2, 8, 512, 512, True),       # 22.7 -> 18.3
    (NVFP4, 2, 3, 8, 1280, 6144, False),
    (MXFP4, 4, 7, 256, 512, 2048, True),      # 38.6 -> 32.8
    (CHANNEL, 13, 1, 8, 640, 2048, True),     # 25.1 -> 24.1: one slot
    (BF16, 5, 1, 32, 512, 6016, True)])       # 41.7 -> 41.4
def test_a_layers_last_two_launches_are_one_where_a_cu_has_one_block(form, tokens, top_k, experts, depth, width, combined):
    down = _lib.Bank(form, _lib.LAYOUT_PREPARED, experts, depth, width, None, None, None)
    assert bool(_lib.library().dew_moe_combines_few(down, tokens, top_k, 0)) == combined
    assert not _lib.library().dew_moe_combines_few(down, 17, top_k, 0) and not _lib.library().dew_moe_combines_few(down, tokens, 8, 1)
    assert not _lib.library().dew_moe_combines_few(down, 0, top_k, 0) and not _lib.library().dew_moe_combines_few(None, tokens, top_k, 0)
