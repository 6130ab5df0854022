"""Several dense projections of one input: quantize the activations once, multiply many times.

``mmq`` quantizes its input to q8_1 blocks on every call.  When the same activations feed
several packed weights (q/k/v, a shared expert's gate/up), that work and its HBM traffic can be
paid once: ``quantize_q8_1`` returns the library's q8_1 workspace as an opaque uint8 tensor and
``mmq_prepared`` runs only the matmul half on it.  A workspace that is quantized before its format is
known holds int8 operands (exact fp16 ones when ``set_forward_operand("half")`` forces them), so the
results are bit-identical to ``mmq`` wherever ``mmq`` multiplies the same kind: formats other than IQ2_S
in calls below the size at which ``mmq`` switches to its scaled operands (``forward_operand_for``), and every
format where ``mmq`` runs on the decode kernels (``forward_kernel_for``), which both then do: up to 32 rows, up to
128 on the matrices that they are the faster for.  Otherwise they are the same q8_1 algebra with another summation order or operand rounding (IQ2_S: exact
fp16 in ``mmq``, int8 here, whose kernel is about a third slower for that format; large calls: scaled
operands in ``mmq``, up to 8e-4 of the largest output apart).  A caller that knows what the workspace
will be multiplied with names the kind itself (``operand=`` of both functions, the same value in both);
``mmq_multi`` does, from the formats and the summed width of its projections, so q/k/v of a long
sequence run on the scaled kernels like one large ``mmq``.

The reference has no such operator; it lists this reuse as its next optimisation
(docs/mmq_fwd_optimization.md:299-307).  ``mmq_multi`` is the convenience wrapper with autograd
(gradient with respect to the input only, as for ``mmq``: the sum of the projections'
``mmq_grad_input``, that of two neighbours of one shape and format taken in fp32); its forward is one call into the
library, which quantizes and multiplies.
"""

from __future__ import annotations

import ctypes
from typing import Sequence

import torch

from . import _native, _validate

torch.library.define("torch_ggml_ops::quantize_q8_1", '(Tensor input, str operand="") -> Tensor')
torch.library.define(
    "torch_ggml_ops::mmq_prepared",
    "(Tensor workspace, Tensor packed_weight, int rows, int in_features, int quant_type, int out_features, "
    'str operand="") -> Tensor',
)


def _stream(tensor: torch.Tensor) -> int:
    return _native.stream_of(tensor.device)


def _workspace_kind(operand: str) -> int:
    """Operand kind of a workspace: the named one, or what the process-wide setting gives an unknown format."""
    if operand == "":
        return _native.lib.tgo_forward_operand_for(0, 0, 0, 1)
    if operand not in ("int8", "half", "scaled"):
        raise ValueError(f'operand must be "int8", "half", "scaled" or "" (by the setting); got {operand!r}')
    return _native.OPERANDS[operand]


def _activation_shape(input: torch.Tensor) -> tuple[int, int]:
    _validate.activation(input, "input")
    in_features = int(input.shape[-1])
    return input.numel() // in_features, in_features


@torch.library.impl("torch_ggml_ops::quantize_q8_1", "CUDA")
def _quantize_device(input: torch.Tensor, operand: str = "") -> torch.Tensor:
    rows, in_features = _activation_shape(input)
    kind = _workspace_kind(operand)
    with _native.on_device(input.device):
        workspace = input.new_empty((_native.lib.tgo_q8_workspace_bytes(rows, in_features),), dtype=torch.uint8)
        _native.check(
            _native.lib.tgo_quantize_q8_1_as(
                input.data_ptr(), workspace.data_ptr(), rows, in_features, kind, _stream(input)
            )
        )
    return workspace


@torch.library.register_fake("torch_ggml_ops::quantize_q8_1")
def _quantize_fake(input, operand=""):
    # (tgo_q8_workspace_bytes: two bytes per value, two fp32 per 32 values, 20 bytes per 256 values, 4 per row, 1 KiB)
    in_features = input.shape[-1]
    rows = input.numel() // in_features
    padded = (rows + 31) // 32 * 32
    size = 2 * padded * in_features + 8 * padded * (in_features // 32) + 20 * padded * (in_features // 256) + 4 * padded + 1024
    return input.new_empty((size,), dtype=torch.uint8)


@torch.library.impl("torch_ggml_ops::mmq_prepared", "CUDA")
def _mmq_prepared_device(
    workspace: torch.Tensor, packed_weight: torch.Tensor, rows: int, in_features: int, quant_type: int,
    out_features: int, operand: str = "",
) -> torch.Tensor:
    _validate.prepared(workspace, packed_weight, rows, in_features, quant_type, out_features)
    kind = _workspace_kind(operand)
    expected = _native.lib.tgo_q8_workspace_bytes(rows, in_features)
    if workspace.numel() != expected:
        raise RuntimeError(
            f"workspace holds {workspace.numel()} bytes; quantize_q8_1 of [{rows}, {in_features}] writes {expected}"
        )
    with _native.on_device(workspace.device):
        output = workspace.new_empty((rows, out_features), dtype=torch.bfloat16)
        # (weights are unpacked once per call only together with their activations)
        scratch_bytes = _native.ranges_scratch_bytes(rows, in_features, out_features, quant_type)
        _scratch, scratch = _native.scratch_of(workspace, scratch_bytes)
        _native.check(
            _native.lib.tgo_mmq_forward_prepared_scratch(
                workspace.data_ptr(), packed_weight.data_ptr(), output.data_ptr(), scratch,
                rows, in_features, out_features, int(quant_type), kind, _stream(workspace),
            )
        )
    return output


@torch.library.register_fake("torch_ggml_ops::mmq_prepared")
def _mmq_prepared_fake(workspace, packed_weight, rows, in_features, quant_type, out_features, operand=""):
    return workspace.new_empty((rows, out_features), dtype=torch.bfloat16)


torch.library.define(
    "torch_ggml_ops::mmq_multi_forward",
    "(Tensor input, Tensor[] packed_weights, int[] quant_types, int[] out_features, str operand) -> Tensor[]",
)
torch.library.define(
    "torch_ggml_ops::mmq_pair_grad_input",
    "(Tensor first_grad_output, Tensor second_grad_output, Tensor first_packed_weight, Tensor second_packed_weight, "
    "int quant_type, int in_features) -> Tensor",
)


def _check_projections(packed_weights, quant_types, out_features) -> None:
    if not (len(packed_weights) == len(quant_types) == len(out_features)) or not packed_weights:
        raise ValueError("packed_weights, quant_types and out_features must be non-empty and of equal length")


@torch.library.impl("torch_ggml_ops::mmq_multi_forward", "CUDA")
def _multi_device(input, packed_weights, quant_types, out_features, operand):
    rows, in_features = _activation_shape(input)
    kind = _workspace_kind(operand)
    _check_projections(packed_weights, quant_types, out_features)
    with _native.on_device(input.device):
        workspace = input.new_empty((_native.lib.tgo_q8_workspace_bytes(rows, in_features),), dtype=torch.uint8)
        for weight, quant_type, features in zip(packed_weights, quant_types, out_features):
            _validate.prepared(workspace, weight, rows, in_features, quant_type, features)
        outputs = [input.new_empty((*input.shape[:-1], features)) for features in out_features]
        count = len(outputs)
        pointers = ctypes.c_void_p * count
        widths, types = (ctypes.c_int64 * count)(*out_features), (ctypes.c_int * count)(*quant_types)
        projections = (
            input.data_ptr(), count, pointers(*(w.data_ptr() for w in packed_weights)),
            pointers(*(o.data_ptr() for o in outputs)), widths, types, workspace.data_ptr(),
        )
        # one product over the columns of all projections, where that pays: the same bits
        unpacked_bytes = (
            _native.lib.tgo_multi_forward_scratch_bytes(count, widths, types, rows, in_features) if operand == "scaled" else 0
        )
        if unpacked_bytes > 0:
            _scratch, scratch = _native.scratch_of(input, unpacked_bytes)
            _native.check(
                _native.lib.tgo_mmq_multi_forward_unpacked(*projections, scratch, rows, in_features, _stream(input))
            )
            return outputs
        scratch_bytes = max(
            _native.ranges_scratch_bytes(rows, in_features, features, quant_type)
            for quant_type, features in zip(quant_types, out_features)
        )
        _scratch, scratch = _native.scratch_of(input, scratch_bytes)
        _native.check(
            _native.lib.tgo_mmq_multi_forward(*projections, scratch, rows, in_features, kind, _stream(input))
        )
    return outputs


@torch.library.register_fake("torch_ggml_ops::mmq_multi_forward")
def _multi_fake(input, packed_weights, quant_types, out_features, operand):
    return [input.new_empty((*input.shape[:-1], features)) for features in out_features]


@torch.library.impl("torch_ggml_ops::mmq_pair_grad_input", "CUDA")
def _pair_grad_input_device(first_grad, second_grad, first_weight, second_weight, quant_type, in_features):
    rows, in_features, out_features = _validate.dense(first_grad, first_weight, quant_type, in_features, backward=True)
    if _validate.dense(second_grad, second_weight, quant_type, in_features, backward=True) != (rows, in_features, out_features):
        raise RuntimeError("the two projections of a pair must have the same shape")
    if second_grad.device != first_grad.device:
        raise RuntimeError("all tensors of a pair must be on the same device")
    with _native.on_device(first_grad.device):
        grad_input = first_grad.new_empty((*first_grad.shape[:-1], in_features))
        workspace = first_grad.new_empty(
            (_native.lib.tgo_pair_grad_workspace_bytes(rows, out_features, in_features, quant_type),), dtype=torch.uint8
        )
        _native.check(
            _native.lib.tgo_mmq_pair_grad_input(
                first_grad.data_ptr(), second_grad.data_ptr(), first_weight.data_ptr(), second_weight.data_ptr(),
                grad_input.data_ptr(), workspace.data_ptr(), rows, out_features, in_features, int(quant_type), _stream(first_grad),
            )
        )
    return grad_input


@torch.library.register_fake("torch_ggml_ops::mmq_pair_grad_input")
def _pair_grad_input_fake(first_grad, second_grad, first_weight, second_weight, quant_type, in_features):
    return first_grad.new_empty((*first_grad.shape[:-1], in_features))


def _pair_grad_input_backward(ctx, grad_grad_input):
    raise RuntimeError("torch_ggml_ops::mmq_pair_grad_input does not support higher-order gradients")


torch.library.register_autograd("torch_ggml_ops::mmq_pair_grad_input", _pair_grad_input_backward)


torch.library.define(
    "torch_ggml_ops::mmq_multi_grad_input",
    "(Tensor[] grad_outputs, Tensor[] packed_weights, int[] quant_types, int in_features) -> Tensor",
)


def _multi_grad_workspace_bytes(rows: int, out_features: Sequence[int], in_features: int) -> int:
    """Workspace of ``mmq_multi_grad_input``; 0 where the projections' gradients are better taken one by one."""
    count = len(out_features)
    return _native.lib.tgo_multi_grad_workspace_bytes(count, (ctypes.c_int64 * count)(*out_features), rows, in_features)


@torch.library.impl("torch_ggml_ops::mmq_multi_grad_input", "CUDA")
def _multi_grad_input_device(grad_outputs, packed_weights, quant_types, in_features):
    if not (len(grad_outputs) == len(packed_weights) == len(quant_types)) or not grad_outputs:
        raise ValueError("grad_outputs, packed_weights and quant_types must be non-empty and of equal length")
    first = grad_outputs[0]
    shapes = [
        _validate.dense(grad, weight, quant_type, in_features, backward=True)
        for grad, weight, quant_type in zip(grad_outputs, packed_weights, quant_types)
    ]
    rows, in_features, _ = shapes[0]
    if any(shape[0] != rows for shape in shapes):
        raise RuntimeError("all gradients must have the same rows")
    if any(grad.device != first.device for grad in grad_outputs):
        raise RuntimeError("all gradients must be on the same device")
    out_features = [shape[2] for shape in shapes]
    count = len(grad_outputs)
    pointers = ctypes.c_void_p * count
    with _native.on_device(first.device):
        grad_input = first.new_empty((*first.shape[:-1], in_features))
        workspace = first.new_empty((_multi_grad_workspace_bytes(rows, out_features, in_features),), dtype=torch.uint8)
        _native.check(
            _native.lib.tgo_mmq_multi_grad_input(
                count, pointers(*(g.data_ptr() for g in grad_outputs)), pointers(*(w.data_ptr() for w in packed_weights)),
                (ctypes.c_int64 * count)(*out_features), (ctypes.c_int * count)(*quant_types), grad_input.data_ptr(),
                workspace.data_ptr(), rows, in_features, _stream(first),
            )
        )
    return grad_input


@torch.library.register_fake("torch_ggml_ops::mmq_multi_grad_input")
def _multi_grad_input_fake(grad_outputs, packed_weights, quant_types, in_features):
    return grad_outputs[0].new_empty((*grad_outputs[0].shape[:-1], in_features))


def _multi_grad_input_backward(ctx, grad_grad_input):
    raise RuntimeError("torch_ggml_ops::mmq_multi_grad_input does not support higher-order gradients")


torch.library.register_autograd("torch_ggml_ops::mmq_multi_grad_input", _multi_grad_input_backward)


class _MultiProjection(torch.autograd.Function):
    @staticmethod
    def forward(ctx, input, quant_types, out_features, *packed_weights):
        rows, in_features = _activation_shape(input)
        quant_types, out_features = [int(q) for q in quant_types], [int(n) for n in out_features]
        operand = multi_operand(quant_types, rows, out_features)
        outputs = torch.ops.torch_ggml_ops.mmq_multi_forward.default(input, packed_weights, quant_types, out_features, operand)
        ctx.quant_types, ctx.out_features = quant_types, out_features
        ctx.in_features = in_features
        ctx.save_for_backward(*packed_weights)
        return tuple(outputs)

    @staticmethod
    def backward(ctx, *grad_outputs):
        grad_input = None
        if ctx.needs_input_grad[0]:
            weights = ctx.saved_tensors
            present = [i for i, grad in enumerate(grad_outputs) if grad is not None]
            if len(present) > 1:
                rows = grad_outputs[present[0]].numel() // ctx.out_features[present[0]]
                if _multi_grad_workspace_bytes(rows, [ctx.out_features[i] for i in present], ctx.in_features) > 0:
                    # one product over the weight rows of all projections
                    grad_input = torch.ops.torch_ggml_ops.mmq_multi_grad_input.default(
                        [grad_outputs[i].contiguous() for i in present], [weights[i] for i in present],
                        [ctx.quant_types[i] for i in present], ctx.in_features,
                    )
                    return (grad_input, None, None) + (None,) * len(weights)
            i = 0
            while i < len(weights):
                grad, weight, quant_type = grad_outputs[i], weights[i], ctx.quant_types[i]
                i += 1
                if grad is None:
                    continue
                # two neighbours of one shape and format (key and value): one kernel, summed in fp32
                if (
                    i < len(weights) and grad_outputs[i] is not None and ctx.quant_types[i] == quant_type
                    and ctx.out_features[i] == ctx.out_features[i - 1]
                ):
                    term = torch.ops.torch_ggml_ops.mmq_pair_grad_input.default(
                        grad.contiguous(), grad_outputs[i].contiguous(), weight, weights[i], quant_type, ctx.in_features
                    )
                    i += 1
                else:
                    term = torch.ops.torch_ggml_ops.mmq_grad_input.default(grad.contiguous(), weight, quant_type, ctx.in_features)
                grad_input = term if grad_input is None else grad_input + term
        return (grad_input, None, None) + (None,) * len(ctx.saved_tensors)


def multi_operand(quant_types: Sequence[int], rows: int, out_features: Sequence[int]) -> str:
    """The operand kind for one workspace that feeds all these projections of ``rows`` activations.

    What ``mmq`` would take for one weight as wide as all of them together; int8, which every format's kernels
    read, when the formats disagree.
    """
    total = sum(int(features) for features in out_features)
    kinds = {_native.forward_operand_for(int(quant_type), int(rows), total) for quant_type in quant_types}
    return kinds.pop() if len(kinds) == 1 else "int8"


def quantize_q8_1(input: torch.Tensor, operand: str = "") -> torch.Tensor:
    """q8_1 workspace of ``input`` (bf16, last dimension a multiple of 256) for ``mmq_prepared``.

    ``operand``: "int8", "half" or "scaled" operands, or "" for what the process-wide setting gives a
    workspace of unknown use (int8 unless "half" is forced).
    """
    return torch.ops.torch_ggml_ops.quantize_q8_1.default(input, operand)


def mmq_prepared(
    workspace: torch.Tensor, packed_weight: torch.Tensor, rows: int, in_features: int, quant_type: int,
    out_features: int, operand: str = "",
) -> torch.Tensor:
    """``[rows, out_features]`` product of the activations behind ``workspace`` with one packed weight.

    ``operand`` must be what ``quantize_q8_1`` was given for this workspace; the output is NaN when it is not.
    """
    return torch.ops.torch_ggml_ops.mmq_prepared.default(
        workspace, packed_weight, int(rows), int(in_features), int(quant_type), int(out_features), operand
    )


def mmq_multi(
    input: torch.Tensor,
    packed_weights: Sequence[torch.Tensor],
    quant_types: Sequence[int],
    out_features: Sequence[int],
) -> tuple[torch.Tensor, ...]:
    """``tuple(mmq(input, w, q, n) for ...)`` with the activations quantized once."""
    _check_projections(packed_weights, quant_types, out_features)
    return _MultiProjection.apply(input, tuple(quant_types), tuple(out_features), *packed_weights)


__all__ = ["mmq_multi", "mmq_prepared", "multi_operand", "quantize_q8_1"]
