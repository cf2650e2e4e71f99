"""Which plain matrices are laid out at the call (`gemm._relaid_first`): a rule on shapes, which needs no GPU."""

import pytest
import torch

from dew_amd import gemm


# (groups, rows a group, depth, width, K-major, laid out first where rows are gathered, where they lie). Rows as they lie have tiles that need
# no order for up to 256 groups; one group more, and they are laid out where gathered ones are.
@pytest.mark.parametrize("groups,rows,depth,width,kmajor,gathered,lying", [
    (8, 4096, 4096, 4096, True, True, False), (256, 3000, 4096, 512, True, True, False), (257, 3000, 4096, 512, True, True, True),
    (257, 4100, 2048, 512, True, True, True), (257, 8300, 2048, 256, False, True, True), (256, 8300, 2048, 256, False, True, False),
    (300, 2999, 4096, 512, True, False, False), (300, 3000, 2048, 512, True, False, False), (300, 8000, 2048, 256, False, False, False),
    (300, 3000, 4096, 96, True, False, False)])
def test_rows_as_they_lie_of_many_groups_are_laid_out_as_gathered_ones_are(groups, rows, depth, width, kmajor, gathered, lying):
    matrices = torch.empty((groups, width, depth) if kmajor else (groups, depth, width), dtype=torch.bfloat16, device="meta")
    matrices = matrices.transpose(1, 2) if kmajor else matrices
    assert gemm._relaid_first(matrices, groups * rows) == gathered
    assert gemm._relaid_first(matrices, groups * rows, as_they_lie=True) == lying
