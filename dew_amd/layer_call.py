"""A sparse layer's forward pass as one foreign call (`dew_moe_layer_forward`): what `SparseMLP` and `GptOssMLP` run where
their options are the ones that call covers. `forward` returns None wherever it does not apply, and the layer then makes the
separate calls, which also raise whatever is wrong with the arguments."""

import ctypes

import torch

from . import _lib, formats, gemm, ops, selection

_TERMS = {"e4m3": 0, "e2m3": 1, "e2m3x2": 2}
_ROUTE = selection.Route(gemm.GROUPED_MATMUL, "hip", "hip")


def described(router: _lib.Router, gating: int, limit: float, shared: bool) -> _lib.Layer:
    """The fixed part of a layer's calls."""
    return _lib.Layer(router, gating, limit, int(shared))


def computes(layer, of: type, names: tuple) -> bool:
    """Whether `layer` computes with `of`'s own methods and properties `names`, the ones that the call stands for: a subclass that
    overrides one of them is run through it."""
    return all(getattr(type(layer), name) is getattr(of, name) for name in names)


def _parameter(tensor, shape: tuple) -> bool:
    return (torch.is_tensor(tensor) and tensor.is_cuda and tensor.dtype == torch.float32 and tensor.is_contiguous()
            and tuple(tensor.shape) == shape)


def _held(bank):
    """The prepared form of a bank whose extents the one call takes as `gemm`'s selector would, else None: formats that
    multiply in 64-deep steps and 32-column atoms are checked by the call, the others are whole 128s."""
    if isinstance(bank, (formats.NvFp4, formats.Fp8Blocks, formats.Fp8Channels)) or (isinstance(bank, formats.Bf16) and bank.transposed):
        _, depth, width = bank.shape
        if depth % 128 or width % 128:
            return None
    elif not isinstance(bank, (formats.Mxfp4Blocks, formats.Bf16, ops.PreparedBank)):
        return None
    return gemm.prepared(bank)


def forward(layer: _lib.Layer, x: torch.Tensor, gate_kernel, gate_bias, selection_bias, banks, biases=(None, None)):
    """The layer's output for `x [..., D]`, or None. `banks`: gate, up and down (an interleaved layer's gate_up, None, down)."""
    if not (torch.is_tensor(x) and x.is_cuda and x.dtype == torch.bfloat16 and x.is_contiguous()) or x.numel() == 0:
        return None
    depth, experts = x.shape[-1], layer.router.experts
    if not _parameter(gate_kernel, (depth, experts)):
        return None
    for bias in (gate_bias, selection_bias):
        if bias is not None and not _parameter(bias, (experts,)):
            return None
    if selection._CHOICES.get():    # a caller names its kernels: the selector answers
        return None
    gate, up, down = (None if bank is None else bank if isinstance(bank, ops.PreparedBank) else _held(bank) for bank in banks)
    if gate is None or down is None or (up is None) != (banks[1] is None) or gate.shape[1] != depth or down.shape[2] != depth:
        return None
    if up is not None and (up.shape != gate.shape or up.descriptor.format != gate.descriptor.format):
        return None
    for bias, bank in zip(biases, (gate, down), strict=True):
        if bias is not None and not _parameter(bias, (bank.shape[0], bank.shape[2])):
            return None
    tokens = x.numel() // depth
    terms = _TERMS[gemm.SPLIT_SECOND_TERM] if gemm.SPLIT_ROWS else -1
    f16_from = ops.F16_ROWS_FROM if ops.F16_ROWS else -1
    library, address = _lib.library(), ctypes.addressof
    fixed = address(layer)
    first, second, third = address(gate.descriptor), None if up is None else address(up.descriptor), address(down.descriptor)
    needed = library.dew_moe_layer_workspace_bytes(fixed, first, second, third, tokens, terms, f16_from)
    if needed == 0:
        return None
    workspace = torch.empty(needed, dtype=torch.uint8, device=x.device)
    out = torch.empty_like(x)
    code = library.dew_moe_layer_forward(fixed, x.data_ptr(), gate_kernel.data_ptr(), ops._ptr(gate_bias), ops._ptr(selection_bias), first, second,
                                         third, ops._ptr(biases[0]), ops._ptr(biases[1]), tokens, terms, f16_from, out.data_ptr(),
                                         workspace.data_ptr(), needed, ops._stream())
    if code == _lib.EINVAL:
        return None
    _lib.check(code, "dew_moe_layer_forward")
    if _ROUTE not in selection._ROUTES:
        selection._ROUTES.append(_ROUTE)
    return out
