"""Where 256 x 256 tiles are taken (`fills_rounds`, csrc/wide.h), read off the one launch whose rule can be asked without a GPU: an e4m3 kernel
gradient, whose line a bf16 one shares."""

import pytest

from dew_amd import ops


# (groups, depth, width, taken): tiles over half of one round of 256, of two, and each side of both
@pytest.mark.parametrize("groups,depth,width,taken", [
    (4, 1024, 2048, False), (1, 2560, 3584, False), (9, 1024, 1024, True), (6, 1024, 1792, True), (8, 1024, 2048, True),      # 128, 140, 144, 168, 256
    (13, 1024, 1280, False), (33, 512, 1024, False), (1, 4352, 4096, False), (1, 4608, 4096, True), (9, 1024, 2048, True),    # 260, 264, 272, 288, 288
    (17, 1024, 2048, True), (256, 256, 256, True), (257, 512, 1024, False)])                                                  # 544, 256; more groups than it holds
def test_gradients_take_wide_tiles_where_they_fill_over_half_of_their_rounds(groups, depth, width, taken):
    for tokens in (512, 128 * 1001, 1 << 20):
        assert ops.kernel_gradient_takes_banks(tokens, depth, width, groups) == taken
    assert not ops.kernel_gradient_takes_banks(384, depth, width, groups)
