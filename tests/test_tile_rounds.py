"""Where an e4m3 kernel gradient takes both operands as banks (dew_moe_kernel_gradient_takes_banks, csrc/gemm.hip), a rule that can be asked
without a GPU and the one that the recipes' gradients follow: quarters of 256 x 256 tiles, one a block at most, and whole tiles from over half of
a round of 256 on."""

import pytest
import torch

from dew_amd import ops, projections


# (groups, depth, width, taken): each side of 64 tiles, of 141 and of a round; a second round just begun leaves in quarters
@pytest.mark.parametrize("groups,depth,width,taken", [
    (1, 128, 128, True), (1, 2048, 2048, True), (64, 256, 128, True), (5, 768, 1024, True),                                   # 1, 64, 64, 60
    (1, 1280, 3328, False), (13, 256, 1280, False), (11, 512, 768, False),                                                    # 65, 65, 66
    (4, 1024, 2048, False), (1, 2560, 3584, False), (3, 256, 47 * 256, True), (9, 1024, 1024, True), (6, 1024, 1792, True),   # 128, 140, 141, 144, 168
    (8, 1024, 2048, True), (1, 257 * 128, 256, False), (1, 257 * 256, 256, True), (13, 1024, 1280, True), (33, 512, 1024, True),    # 256, 129, 257, 260, 264
    (1, 4352, 4096, True), (1, 4608, 4096, True), (9, 1024, 2048, True), (17, 1024, 2048, True),                              # 272, 288, 288, 544
    (256, 256, 256, True), (257, 512, 1024, False)])                                                                          # 256; more groups than it holds
def test_gradients_take_banks(groups, depth, width, taken):
    for tokens in (512, 128 * 1001, 1 << 20):
        assert ops.kernel_gradient_takes_banks(tokens, depth, width, groups) == taken
    assert not ops.kernel_gradient_takes_banks(384, depth, width, groups)


@pytest.mark.parametrize("depth,width", [(512, 8192), (1280, 3328), (4352, 4096)])     # 64 tiles, 65, 272
def test_a_recipes_gradient_asks_the_library(monkeypatch, depth, width):
    """One rule: what the library answers is what the package does."""
    calls = []
    monkeypatch.setattr(ops, "quantize_columns", lambda x, *, mx, as_bank: calls.append(as_bank) or (None, None))
    monkeypatch.setattr(ops, "kernel_gradient_mxfp8", lambda *_, **__: "rows")
    monkeypatch.setattr(ops, "kernel_gradient_mxfp8_banks", lambda *_, **__: "banks")
    taken = ops.kernel_gradient_takes_banks(1024, depth, width, 1)
    got = projections._contracted(torch.empty(1024, depth), None, width, torch.tensor([0, 1024]), True, torch.bfloat16)
    assert got == ("banks" if taken else "rows") and calls == [taken]
