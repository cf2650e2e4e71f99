"""The counting sort over many blocks against a stable argsort: a block short of and past its slots, more rounds than one a wavefront, more
buckets than sixteen wavefronts' counters fit the LDS, dropped slots, a shared expert's rows."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,top_k,experts,shared", ((4097, 1, 8, 0), (2560, 2, 8, 0), (1707, 3, 64, 0), (5121, 8, 128, 5121), (65537, 1, 5, 0), (16385, 8, 256, 0),
                                                         (5000, 1, 907, 0), (5000, 1, 908, 0), (9000, 2, 1000, 9000), (700, 60, 1024, 0)))
def test_sorted_slots(tokens, top_k, experts, shared):
    from dew_amd import _lib, ops

    generator = torch.Generator("cuda").manual_seed(tokens)
    ids = (torch.rand((tokens, top_k), generator=generator, device="cuda") ** 3 * experts).to(torch.int32)     # (some experts have most)
    ids[torch.rand((tokens, top_k), generator=generator, device="cuda") < 0.02] = experts                    # (dropped)
    ids[0, 0] = -1
    groups, slots = experts + bool(shared), tokens * top_k + shared
    sizes, offsets, order, rows = (torch.full((n,), -7, dtype=torch.int32, device="cuda") for n in (groups, groups + 1, slots, slots))
    library = _lib.library()
    needed = library.dew_moe_permute_workspace_bytes(slots, groups)
    workspace = torch.full((needed + 256,), 113, dtype=torch.uint8, device="cuda")
    for _ in range(2):
        if shared:
            code = library.dew_moe_permute_shared(ids.data_ptr(), tokens, top_k, experts, shared, sizes.data_ptr(), offsets.data_ptr(), order.data_ptr(),
                                                  rows.data_ptr(), workspace.data_ptr(), needed, ops._stream())
        else:
            code = library.dew_moe_permute(ids.data_ptr(), tokens, top_k, experts, sizes.data_ptr(), offsets.data_ptr(), order.data_ptr(), rows.data_ptr(),
                                           workspace.data_ptr(), needed, ops._stream())
        _lib.check(code, "dew_moe_permute")
    assert bool((workspace[needed:] == 113).all())
    bucket = torch.where((ids < 0) | (ids >= experts), groups, ids).flatten()
    bucket = torch.cat((bucket, torch.full((shared,), experts, dtype=torch.int32, device="cuda"))).long()
    want = torch.argsort(bucket, stable=True)
    source = torch.cat((torch.arange(tokens * top_k, device="cuda") // top_k, torch.arange(shared, device="cuda")))
    counts = torch.bincount(bucket, minlength=groups + 1)[:groups]
    assert torch.equal(order.long(), want) and torch.equal(rows.long(), source[want])
    assert torch.equal(sizes.long(), counts) and torch.equal(offsets.long(), torch.cat((counts.new_zeros(1), counts.cumsum(0))))
