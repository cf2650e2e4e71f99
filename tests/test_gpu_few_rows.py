"""A decode step's launches for the fewest rows: strips whose depth several wavefronts share, against the tiles that they stand in for (the
same order of sums: the same bits), and the sort of a few slots in the router's launch, against the separate calls."""

import pytest
import torch
from test_gpu_one_call import bank

pytestmark = pytest.mark.gpu


# depths of whole chunks of four 64-deep steps, a part of one, and fewer chunks than shares of a round; groups of one row, of none, of more
# pieces than a block's threads, of two tiles
@pytest.mark.parametrize("quant", ("fp8_block", "fp8_channel", "nvfp4"))
@pytest.mark.parametrize("depth", (1024, 1280, 2304, 4096))
@pytest.mark.parametrize("sizes", ([1], [0, 3, 0, 1], [12], [33], [1] * 70))
def test_shared_strips_return_the_tiled_launchs_bits(quant, depth, sizes):
    from dew_amd import ops

    generator = torch.Generator("cuda").manual_seed(depth)
    experts, rows, width = len(sizes), sum(sizes) + 2, 128     # (of 70 groups the paired strips are too many: another launch, the same bits)
    gate, up = (ops.prepare(bank(experts, depth, width, quant, generator)) for _ in range(2))
    x = torch.randn((40, depth), generator=generator, device="cuda").to(torch.bfloat16)
    gather = torch.randint(0, 40, (rows,), generator=generator, device="cuda", dtype=torch.int32)
    scatter = torch.randperm(rows, generator=generator, device="cuda").to(torch.int32)
    counts = torch.tensor(sizes, dtype=torch.int32, device="cuda")
    offsets = ops.group_offsets(counts)
    bias = torch.randn((experts, width), generator=generator, device="cuda")
    calls = {"paired": lambda: ops.gateup_swiglu(x, gate, up, offsets, gather=gather),
             "paired, clamped": lambda: ops.gateup_swiglu(x, gate, up, None, sizes=counts, gather=gather, activation="geglu", limit=1.0),
             "as they lie": lambda: ops.gateup_swiglu(x[:rows].contiguous(), gate, up, offsets) if rows <= 40 else ops.gateup_swiglu(x, gate, up, offsets, gather=gather),
             "plain": lambda: ops.grouped_gemm(x, gate, offsets, gather=gather, scatter=scatter),
             "biased": lambda: ops.grouped_gemm(x, gate, None, sizes=counts, gather=gather, scatter=scatter, bias=bias, round_bias=True)}
    for name, call in calls.items():
        got = call()
        with ops.tile_rows(32):
            want = call()
        assert torch.equal(got, want) and bool(got.any()), name
        assert torch.equal(call(), want), name


# one matrix on each side of the lines from which its strips are shared: 128 and 256 strips of 4096 and 6144 deep, and of rows that fill the LDS
@pytest.mark.parametrize("quant", ("fp8_block", "fp8_channel", "nvfp4"))
@pytest.mark.parametrize("depth,width,rows", ((4096, 1024, 4), (4096, 1280, 4), (4096, 2048, 4), (6144, 2048, 4), (6144, 2176, 4), (6144, 1024, 8), (6144, 2048, 8),
                                              (8192, 1024, 7), (8192, 1024, 8)))
def test_one_matrix_on_the_lines_of_shared_strips(quant, depth, width, rows):
    from dew_amd import ops

    generator = torch.Generator("cuda").manual_seed(width)
    matrices = ops.prepare(bank(rows, depth, width, quant, generator))
    x = torch.randn((rows, depth), generator=generator, device="cuda").to(torch.bfloat16)
    for sizes in ([1] * rows, [0, rows - 1] + [0] * (rows - 2)):     # (the last row is no group's)
        offsets = ops.group_offsets(torch.tensor(sizes, dtype=torch.int32, device="cuda"))
        got = ops.grouped_gemm(x, matrices, offsets)
        with ops.tile_rows(32):
            want = ops.grouped_gemm(x, matrices, offsets)
        assert torch.equal(got, want) and bool(got[0].any())


@pytest.mark.parametrize("tokens,experts,top_k,shared", ((1, 8, 8, None), (1, 128, 8, None), (2, 8, 8, None), (16, 5, 1, None), (5, 300, 3, None),
                                                         (4, 64, 3, 256), (8, 16, 1, 256), (1, 20, 17, None), (17, 8, 1, None)))     # the last two: 17 slots
def test_a_few_slots_sort_as_many_do(tokens, experts, top_k, shared):
    from dew_amd import moe

    depth, hidden = 512, 256
    layer = moe.SparseMLP(num_experts=experts, top_k=top_k, hidden_features=hidden, out_features=depth, shared=shared)
    generator = torch.Generator("cuda").manual_seed(tokens)
    shapes = {"gate_proj": (depth, hidden), "up_proj": (depth, hidden), "down_proj": (hidden, depth)}
    held = {"experts": {n: {"kernel": bank(experts, *s, "fp8_block", generator)} for n, s in shapes.items()}}
    if shared:
        held["shared_experts"] = {n: {"kernel": bank(1, *s, "fp8_block", generator)} for n, s in shapes.items()}
    variables = {"params": {"gate": {"kernel": torch.randn((depth, experts), generator=generator, device="cuda") * depth ** -0.5}}, "quantization": held}
    x = torch.randn((tokens, depth), generator=generator, device="cuda").to(torch.bfloat16)
    want = layer._bound(variables, ())(x)
    got = layer._applied(variables, x)
    assert got is not None and torch.equal(got, want) and bool(got.any())
