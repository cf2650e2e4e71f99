"""Every grouped product's wrapper refuses, on the host and before any pointer reaches a kernel, what a launch would
trust blindly: operands off the device, index tensors of another dtype, short gathers, offsets of the wrong length.
The CPU half needs no GPU (a host tensor is the first thing refused); the GPU half hands device tensors with one
defect each and still launches nothing."""

import pytest
import torch

from dew_amd import _lib, ops
from dew_amd.ops import KernelError


def fake_bank(fmt, experts=2, depth=256, width=256):
    return ops.PreparedBank(_lib.Bank(fmt, _lib.LAYOUT_PREPARED, experts, depth, width, None, None, None), (experts, depth, width), ())


def products(device):
    """(name, call) for each product wrapper with well-formed operands on `device`; `call(**changes)` swaps operands."""
    rows, depth, width, experts = 6, 256, 256, 2
    pitch = ops.block_scale_pitch(depth)
    make = lambda shape, dtype: torch.zeros(shape, dtype=dtype, device=device)
    base = dict(offsets=make((experts + 1,), torch.int32), gather=make((rows,), torch.int32), scatter=make((rows,), torch.int32))
    x = make((rows, depth), torch.bfloat16)
    split, scale, scales = make((rows, 2 * depth), torch.uint8), make((rows,), torch.uint8), make((rows, pitch), torch.uint8)
    codes, mx_scales = make((rows, depth), torch.uint8), make((rows, depth // 32), torch.uint8)
    mx4, fp8, mx8 = fake_bank(_lib.W_MXFP4), fake_bank(_lib.W_FP8_BLOCK), fake_bank(_lib.W_MXFP8)

    def bound(function, *operands, scattered=True):
        def call(**changes):
            arguments = {**base, **changes}
            offsets = arguments.pop("offsets")
            if not scattered:
                arguments.pop("scatter")
            return function(*operands, offsets, **arguments)
        return call

    return [
        ("grouped_gemm", bound(ops.grouped_gemm, x, mx4)),
        ("gateup_swiglu", bound(ops.gateup_swiglu, x, mx4, mx4, scattered=False)),
        ("gateup_interleaved", bound(ops.gateup_interleaved, x, mx4, scattered=False)),
        ("grouped_gemm_split", bound(ops.grouped_gemm_split, split, scale, mx4)),
        ("gateup_swiglu_split", bound(ops.gateup_swiglu_split, split, scale, mx4, mx4, scattered=False)),
        ("gateup_swiglu_split_out", bound(ops.gateup_swiglu_split_out, split, scale, mx4, mx4, scattered=False)),
        ("grouped_gemm_split_blocks", bound(ops.grouped_gemm_split_blocks, split, scales, mx4)),
        ("grouped_gemm_mxfp8_rows", bound(ops.grouped_gemm_mxfp8_rows, codes, mx_scales, mx8)),
        ("grouped_gemm_fp8_rows", bound(ops.grouped_gemm_fp8_rows, codes, scales, fp8)),
    ]


SCATTERED = ("grouped_gemm", "grouped_gemm_split", "grouped_gemm_split_blocks", "grouped_gemm_mxfp8_rows", "grouped_gemm_fp8_rows")


@pytest.mark.parametrize("name", [name for name, _ in products("cpu")])
def test_a_host_operand_is_refused_before_any_launch(name):
    call = dict(products("cpu"))[name]
    with pytest.raises(KernelError, match="must be on the GPU"):
        call()


@pytest.mark.gpu
@pytest.mark.parametrize("name", [name for name, _ in products("cpu")])
def test_defective_index_tensors_are_refused_on_the_device_side_too(name):
    call = dict(products("cuda"))[name]
    device = torch.device("cuda")
    with pytest.raises(KernelError, match="gather must be torch.int32"):
        call(gather=torch.zeros(6, dtype=torch.int64, device=device))
    with pytest.raises(KernelError, match="cover every row"):
        call(gather=torch.zeros(3, dtype=torch.int32, device=device), rows=6)
    with pytest.raises(KernelError, match="offsets has 5 entries"):
        call(offsets=torch.zeros(5, dtype=torch.int32, device=device))
    with pytest.raises(KernelError, match="offsets must be torch.int32"):
        call(offsets=torch.zeros(3, dtype=torch.int64, device=device))
    with pytest.raises(KernelError, match="gather must be on the GPU"):
        call(gather=torch.zeros(6, dtype=torch.int32))
    with pytest.raises(KernelError, match="gather must be contiguous"):
        call(gather=torch.zeros(12, dtype=torch.int32, device=device)[::2])
    with pytest.raises(KernelError, match="rows asked of"):
        call(gather=None, rows=7)
    if name in SCATTERED:   # (the paired and gated products write sorted rows: they take no scatter)
        with pytest.raises(KernelError, match="scatter must be torch.int32"):
            call(scatter=torch.zeros(6, dtype=torch.int64, device=device))


def test_the_float32_gate_and_a_latent_layers_projections_refuse_on_the_host():
    """`gate_rows_add_f32` takes device tensors only; a latent layer's dense projection refuses a kernel of another shape,
    and a float32 kernel where the layer states no compute dtype (the reference would then run the projection in float32)."""
    from dew_amd import moe

    x, rows = torch.zeros((4, 64), dtype=torch.bfloat16), torch.zeros((4, 32), dtype=torch.bfloat16)
    with pytest.raises(KernelError, match="must be on the GPU"):
        ops.gate_rows_add_f32(x, torch.zeros(64), rows, rows)
    layer = moe.SparseMLP(num_experts=4, top_k=2, hidden_features=64, out_features=64, latent_features=32)
    assert layer._bound({}, ()).experts.out_features == 32
    variables = {"params": {"routed_expert_down_proj": {"kernel": torch.zeros((64, 32))}}}
    with pytest.raises(ValueError, match="states no compute dtype"):
        layer._bound(variables, ())._dense(x, "routed_expert_down_proj", 64, 32)
    with pytest.raises(ValueError, match=r"the layer's is \(64, 16\)"):
        layer._bound(variables, ())._dense(x, "routed_expert_down_proj", 64, 16)
    with pytest.raises(KeyError, match="routed_expert_up_proj"):
        layer._bound(variables, ())._dense(x, "routed_expert_up_proj", 32, 64)


@pytest.mark.parametrize("words", [0, 1, 511, 513])
def test_nvfp4_magnitudes_of_another_length_are_refused(words):
    """The quantizer reads every partial magnitude that `nvfp4_largest` writes, and so no shorter tensor."""
    assert _lib.library().dew_moe_nvfp4_partials() == 512
    with pytest.raises(KernelError, match=f"largest has {words} words, not nvfp4_largest's 512"):
        ops.quantize_nvfp4(torch.zeros((128, 128), dtype=torch.bfloat16), torch.zeros(words, dtype=torch.int32), rows=True, tokens=False)


def test_what_a_steps_launch_refuses_bears_its_name():
    """Both entry points share their checks, each under its own name; magnitudes are an NVFP4 bank's alone. (Refused before any address is read.)"""
    lib, bank, at = _lib.library(), _lib.Bank(), 4096
    step = lambda w, form, largest, blocks, groups: lib.dew_moe_quantize_step_matrices(w, form, 0, 0, 1, 256, 256, largest, blocks, groups, 128, at, at, bank, None)
    assert step(None, _lib.W_NVFP4, None, None, 0) != 0
    assert lib.dew_moe_last_error().decode().startswith("dew_moe_quantize_step_matrices: w, the prepared buffer")
    assert step(at, _lib.W_NVFP4, None, at, 0) != 0
    assert lib.dew_moe_last_error().decode() == "dew_moe_quantize_step_matrices: offsets must not be null, 0 groups in units of 128"
    for form in (_lib.W_FP8_BLOCK, _lib.W_MXFP8):
        assert step(at, form, at, None, 0) == lib.dew_moe_quantize_matrices(None, form, 0, 0, 1, 256, 256, at, bank, None) != 0
        assert lib.dew_moe_last_error().decode().startswith("dew_moe_quantize_matrices: w, the prepared buffer")
        assert step(at, form, at, None, 0) != 0
        assert lib.dew_moe_last_error().decode() == f"dew_moe_quantize_step_matrices: a bank of format {form} has no tensor scale to form from magnitudes"


@pytest.mark.parametrize("count", [0, 4])
def test_one_launch_forms_the_magnitudes_of_one_to_three_operands(count):
    with pytest.raises(KernelError, match=f"{count} operands: one launch forms the magnitudes of 1 to 3"):
        ops.nvfp4_largest_of(*[torch.zeros((128, 128), dtype=torch.bfloat16)] * count)


@pytest.mark.gpu
def test_an_operand_whose_magnitudes_are_formed_lies_as_it_is_shaped():
    """`nvfp4_largest` is a row quantizer's first read: contiguous, as `quantize_nvfp4` takes it. (`nvfp4_largest_of` takes matrices either way round.)"""
    x = torch.ones((2, 128, 256), dtype=torch.bfloat16, device="cuda")
    for turned in (x.transpose(1, 2), x.transpose(0, 1), x[0].transpose(0, 1)):
        with pytest.raises(KernelError, match="x must be contiguous"):
            ops.nvfp4_largest(turned)
    assert torch.equal(ops.nvfp4_largest_of(x.transpose(1, 2))[0], ops.nvfp4_largest(x))


@pytest.mark.parametrize("shape", [(128,), (2, 128, 128), ()])
def test_an_nvfp4_operand_that_is_no_matrix_is_refused(shape):
    with pytest.raises(KernelError, match=r"not \[rows, depth\]"):
        ops.quantize_nvfp4(torch.zeros(shape, dtype=torch.bfloat16), torch.zeros(512, dtype=torch.int32), rows=True, tokens=False)


def test_tensor_scales_go_to_banks_that_carry_them_one_an_expert():
    nvfp4 = fake_bank(_lib.W_NVFP4, experts=3)
    for count in (0, 1, 2, 4):
        with pytest.raises(KernelError, match=f"{count} tensor scales for the bank's 3 experts"):
            nvfp4.under(torch.zeros(count))
    with pytest.raises(KernelError, match="must be on the GPU"):
        nvfp4.under(torch.zeros(3))
    x, largest = torch.zeros((128, 128), dtype=torch.bfloat16), torch.zeros(512, dtype=torch.int32)
    for fmt in (_lib.W_FP8_BLOCK, _lib.W_FP8_CHANNEL, _lib.W_MXFP8, _lib.W_BF16):
        bank = fake_bank(fmt, experts=3)
        with pytest.raises(KernelError, match="only an NVFP4 bank carries tensor scales"):
            bank.under(torch.zeros(3))
        with pytest.raises(KernelError, match="only an NVFP4 bank carries tensor scales"):
            ops.quantize_nvfp4(x, largest, rows=True, tokens=False, bank=bank)


@pytest.mark.gpu
def test_tensor_scales_of_another_dtype_or_spacing_are_refused_on_the_device_too():
    nvfp4 = fake_bank(_lib.W_NVFP4, experts=3)
    with pytest.raises(KernelError, match="scales must be torch.float32"):
        nvfp4.under(torch.zeros(3, dtype=torch.float64, device="cuda"))
    with pytest.raises(KernelError, match="scales must be contiguous"):
        nvfp4.under(torch.zeros(6, device="cuda")[::2])
    with pytest.raises(KernelError, match="largest must be torch.int32"):
        ops.quantize_nvfp4(torch.zeros((128, 128), dtype=torch.bfloat16, device="cuda"), torch.zeros(512, device="cuda"), rows=True, tokens=False)
