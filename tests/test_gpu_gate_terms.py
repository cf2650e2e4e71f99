"""The gate's logits from three bf16 terms of the fp32 kernel, at the edges of every launch that forms them so: against the product in
float64, with operands whose terms are not the value's (infinities, NaN, the largest magnitudes), and in a layer's shares."""

import pytest
import torch

pytestmark = pytest.mark.gpu

# tokens, depth, experts: the launch each shape takes stands behind it (tiles of 32 tokens x tiles of 32 experts, wavefronts a tile)
SHAPES = [(14400, 80, 128),    # 2 x 4, 4; the depth ends inside a step
          (14400, 320, 131),   # the last lane's experts overlap the lane's before it
          (10300, 144, 40),    # 2 x 2, 4
          (10300, 448, 20),    # 2 x 1, 4; steps left over behind the unrolled ones
          (4200, 1088, 9),     # 1 x 1, 4
          (2000, 208, 300),    # 2 x 1, 8
          (1900, 112, 63),     # 1 x 1, 8
          (2040, 80, 32),      # 1 x 1, 16 in steps of 32; a depth behind the last step
          (2040, 96, 32),      # whole steps
          (2100, 1072, 8),     # 1 x 1, 16 in steps of 64; three chunks behind the last step
          (2100, 1088, 8),     # whole steps
          # chains of sums that end before a wavefront's share does, once and more often, with a depth behind the last step and without
          (14400, 4432, 128), (14400, 8512, 100), (10300, 4480, 40), (10300, 8464, 20), (4200, 4432, 9), (2000, 4432, 300), (1900, 8512, 63)]


@pytest.mark.parametrize("tokens,depth,experts", SHAPES)
def test_three_terms_are_the_fp32_products(tokens, depth, experts):
    """2^-19 of the summed magnitudes, as for the other launches: products exact in fp32, a few roundings a sum of up to 7168."""
    from dew_amd import ops

    generator = torch.Generator("cuda").manual_seed(depth + experts)
    x = torch.randn((tokens, depth), generator=generator, device="cuda").to(torch.bfloat16)
    kernel = torch.randn((depth, experts), generator=generator, device="cuda") * depth ** -0.5
    bias = torch.randn(experts, generator=generator, device="cuda")
    got = ops.router_logits(x, kernel, bias)
    exact = x.double() @ kernel.double() + bias.double()
    magnitudes = x.double().abs() @ kernel.double().abs() + bias.double().abs()
    assert bool(((got.double() - exact).abs() <= 2.0 ** -19 * magnitudes).all())
    assert torch.equal(got, ops.router_logits(x, kernel, bias))

    x[3, depth - 1], x[tokens - 1, 0], x[7, 5] = float("inf"), float("nan"), -3.0e38
    x[3, 2] = x[7, 2] = 0.0                              # (no product that overflows in fp32 alone meets an infinity of the other sign)
    kernel[1, 0], kernel[depth - 1, experts - 1], kernel[2, 2], kernel[:, 4] = float("-inf"), float("nan"), 3.4028e38, 0.0
    kernel.view(torch.int32)[9, 5] = 0x7F800001          # a NaN whose upper half is an infinity's
    got = ops.router_logits(x, kernel)
    exact = x.double() @ kernel.double()
    assert torch.equal(got.isnan(), exact.isnan())
    infinite = exact.abs() > torch.finfo(torch.float32).max
    assert torch.equal(got[infinite].double(), exact[infinite].sign() * float("inf"))
    plain = ~(infinite | exact.isnan())
    magnitudes = x.double().nan_to_num(0, 0, 0).abs() @ kernel.double().nan_to_num(0, 0, 0).abs()
    assert bool(((got.double() - exact)[plain].abs() <= 2.0 ** -19 * magnitudes[plain]).all())


@pytest.mark.parametrize("tokens,depth", [(2040, 512), (2040, 1088), (2100, 1088)])
def test_a_layers_shares_are_the_launchs_sums(tokens, depth):
    from dew_amd import formats, moe

    generator = torch.Generator("cuda").manual_seed(tokens + depth)
    normal = lambda *shape: torch.randn(shape, generator=generator, device="cuda")
    experts, hidden = 32 if tokens <= 2048 else 8, 128
    layer = moe.SparseMLP(num_experts=experts, top_k=2, hidden_features=hidden, out_features=depth)
    shapes = {"gate_proj": (depth, hidden), "up_proj": (depth, hidden), "down_proj": (hidden, depth)}
    variables = {"params": {"gate": {"kernel": normal(depth, experts) * depth ** -0.5}},
                 "quantization": {"experts": {n: {"kernel": formats.Bf16((normal(experts, *s) * 0.05).to(torch.bfloat16))} for n, s in shapes.items()}}}
    x = normal(tokens, depth).to(torch.bfloat16)
    x[5, 7], x[tokens - 1, depth - 1] = float("inf"), float("nan")
    want, got = layer._bound(variables, ())(x), layer._applied(variables, x)
    assert got is not None and torch.equal(got.nan_to_num(nan=9.0), want.nan_to_num(nan=9.0)) and bool(got[8].any())


@pytest.mark.parametrize("tokens,depth,experts", [(8192, 4096, 128), (4096, 4096, 8), (2048, 4096, 256)])
def test_operands_that_are_no_finite_numbers_cost_what_one_instruction_does(tokens, depth, experts):
    """Such sums are formed again beside each other, not one behind another: for all of them the pass takes what the fp32 instruction takes
    for the product (1.5 to 4 times the terms), where a walk of the depth a lane took 20 to 150 times. And no other token's sums change."""
    from dew_amd import ops

    generator = torch.Generator("cuda").manual_seed(7)
    x = torch.randn((tokens, depth), generator=generator, device="cuda").to(torch.bfloat16)
    kernel = torch.randn((depth, experts), generator=generator, device="cuda") * depth ** -0.5
    unwritten = x.clone()
    unwritten[tokens // 2:] = float("nan")
    one = x.clone()
    one[tokens // 3, depth // 2] = float("inf")

    def fastest(x):
        ops.router_logits(x, kernel)
        times = []
        for _ in range(5):
            begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            begin.record()
            for _ in range(4):
                ops.router_logits(x, kernel)
            end.record()
            end.synchronize()
            times.append(begin.elapsed_time(end))
        return min(times)

    plain = fastest(x)
    assert fastest(unwritten) <= 6 * plain and fastest(one) <= 6 * plain
    want, got = ops.router_logits(x, kernel), ops.router_logits(unwritten, kernel)
    assert torch.equal(got[:tokens // 2], want[:tokens // 2]) and bool(got[tokens // 2:].isnan().all())
    got = ops.router_logits(one, kernel)
    got[tokens // 3] = want[tokens // 3]
    assert torch.equal(got, want)


@pytest.mark.parametrize("tokens,depth,experts", SHAPES)
@pytest.mark.parametrize("exponent", (-100, -112, -126, -140))
def test_a_gate_value_that_three_terms_do_not_hold(tokens, depth, experts, exponent):
    """Below 2^-110 a value's last bits lie under bf16's least (its smallest subnormal is 2^-133), and under 2^-133 all of them. One column of such
    values, beside others that keep their bits."""
    from dew_amd import ops

    generator = torch.Generator("cuda").manual_seed(depth + experts)
    x = torch.randn((tokens, depth), generator=generator, device="cuda").to(torch.bfloat16) * 2.0 ** 60
    kernel = torch.randn((depth, experts), generator=generator, device="cuda") * depth ** -0.5
    want = ops.router_logits(x, kernel)
    kernel[:, experts // 2] = (kernel[:, experts // 2].double() * 2.0 ** exponent).float()
    got = ops.router_logits(x, kernel)
    exact, magnitudes = x.double() @ kernel.double(), x.double().abs() @ kernel.double().abs()
    assert bool(((got.double() - exact).abs() <= 2.0 ** -19 * magnitudes).all())
    want[:, experts // 2] = got[:, experts // 2]
    assert torch.equal(got, want)


# (what the fp32 instruction's sums, rounded after each product, are off)
@pytest.mark.parametrize("tokens,depth,experts,bar", [(8192, 7168, 256, 3.0e-7), (4096, 7168, 256, 3.0e-7), (3000, 5120, 128, 2.7e-7), (2112, 7168, 160, 3.0e-7),
                                                      (5000, 7168, 32, 3.0e-7), (2048, 7168, 256, 9.6e-8), (4100, 7168, 40, 3.0e-7)])
def test_sums_of_one_sign_are_no_further_off_than_rounded_ones(tokens, depth, experts, bar):
    """The instruction cuts its sums off, always to the same side: in one chain over a wavefront's share 7.2e-7 at 1792 depths."""
    from dew_amd import ops

    generator = torch.Generator("cuda").manual_seed(depth + experts)
    x = torch.randn((tokens, depth), generator=generator, device="cuda").abs().to(torch.bfloat16)
    kernel = torch.randn((depth, experts), generator=generator, device="cuda").abs() * depth ** -0.5
    for sign in (1.0, -1.0):
        exact = x.double() @ (sign * kernel).double()
        assert float((ops.router_logits(x, sign * kernel).double() - exact).norm() / exact.norm()) <= bar


@pytest.mark.parametrize("tokens,depth,experts", SHAPES)
def test_every_term_of_a_product_is_in_the_sum(tokens, depth, experts):
    """One product a sum, so that the sum is exact: all 24 bits of the gate's value times the token's."""
    from dew_amd import ops

    generator = torch.Generator("cuda").manual_seed(depth + experts)
    x = torch.zeros((tokens, depth), dtype=torch.bfloat16, device="cuda")
    at = torch.randint(0, depth, (tokens, 1), generator=generator, device="cuda")
    x.scatter_(1, at, 2.0 ** torch.randint(-20, 20, (tokens, 1), generator=generator, device="cuda").to(torch.bfloat16))
    kernel = torch.randn((depth, experts), generator=generator, device="cuda")
    assert torch.equal(ops.router_logits(x, kernel), kernel[at[:, 0]] * x.gather(1, at).float())
